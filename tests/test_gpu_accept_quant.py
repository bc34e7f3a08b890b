"""GPU: fused greedy acceptance (bit-exact against the oracle and numpy.argmax) and the device quantizers (bit-exact
against the oracle's ggml-semantics quantizers, which tests/test_oracle.py pins against numpy)."""
import numpy as np
import pytest

import backburner_amd as bb
import oracle as orc

pytestmark = pytest.mark.gpu
VOCAB = 151936


@pytest.fixture(scope="module")
def ws():
    w = bb.Workspace()
    yield w
    w.close()


def gpu_accept(ws, logits, draft):
    n_rows, vocab = logits.shape
    dl = bb.DeviceBuffer.from_array(np.ascontiguousarray(logits, np.float32))
    dd = bb.DeviceBuffer.from_array(np.ascontiguousarray(draft, np.int32) if len(draft) else np.zeros(1, np.int32))
    do = bb.DeviceBuffer((2 + n_rows) * 4)
    ws.accept(dl.ptr, n_rows, vocab, dd.ptr, do.ptr)
    bb.device_sync()
    out = do.download(np.int32)
    return int(out[0]), int(out[1]), out[2:]


def planted(rng, k_true, n_rows=17, vocab=VOCAB, ties=True):
    logits = rng.standard_normal((n_rows, vocab)).astype(np.float32)
    draft = rng.integers(0, vocab, n_rows - 1).astype(np.int32)
    for i in range(min(k_true, n_rows - 1)):
        logits[i, draft[i]] = logits[i].max() + 0.5
        if ties:   # an exact tie above the draft token: the lower index must win
            j = int(rng.integers(0, vocab))
            logits[i, j] = logits[i, draft[i]]
            if j < draft[i]:
                draft[i] = j
    if k_true < n_rows - 1 and np.argmax(logits[k_true]) == draft[k_true]:
        logits[k_true, draft[k_true]] = logits[k_true].min() - 1.0
    return logits, draft


@pytest.mark.parametrize("k_true", list(range(17)))
def test_accept_planted_full_vocab(ws, k_true):
    rng = np.random.default_rng(500 + k_true)
    logits, draft = planted(rng, k_true)
    k, b, am = gpu_accept(ws, logits, draft)
    ko, bo, amo = orc.accept(logits, draft)
    assert np.array_equal(am, amo) and np.array_equal(am, np.argmax(logits, axis=1))
    assert (k, b) == (ko, bo) == (k_true, int(np.argmax(logits[k_true])))


def test_accept_edge_values(ws):
    vocab = 4099                                           # not a multiple of 4: the scalar path
    logits = np.full((5, vocab), -1.0, np.float32)
    logits[0, [5, 700, 3]] = 2.0                           # tie -> 3
    logits[1, 400] = 0.0; logits[1, 20] = -0.0             # -0 == +0 -> 20
    logits[2, 50] = np.nan; logits[2, 40] = np.inf         # first NaN -> 50
    logits[3, :] = -np.inf; logits[3, 4098] = -np.inf      # all equal -> 0
    logits[4, 4098] = 1e30                                 # last element
    draft = np.array([3, 20, 50, 1], np.int32)
    k, b, am = gpu_accept(ws, logits, draft)
    ko, bo, amo = orc.accept(logits, draft)
    assert list(am) == list(amo) == [3, 20, 50, 0, 4098] and (k, b) == (ko, bo) == (3, 0)
    for n_rows in (1, 2, 64):                              # n_rows limits
        rng = np.random.default_rng(n_rows)
        lg, dr = planted(rng, n_rows // 2, n_rows=n_rows, vocab=1000, ties=False)
        assert gpu_accept(ws, lg, dr)[:2] == orc.accept(lg, dr)[:2]


@pytest.mark.parametrize("vocab", [1, 3, 4, 255, 1024, 16383, 16384, 16385, 16388, 50001, 50004])
def test_accept_segment_edges(ws, vocab):
    """Both load widths, 6 to 36 rows of every segment size (the largest, 16,384, from 50,001 values on): the largest value,
    ties, -0 == +0, NaN of either sign and rows of -inf at the first, middle and last places of a row, against numpy.argmax."""
    rng = np.random.default_rng(vocab)
    at = sorted({0, 1 % vocab, vocab // 2, max(0, vocab - 2), vocab - 1, min(16383, vocab - 1), min(16384, vocab - 1)})
    rows = [np.full(vocab, -np.inf, np.float32)]
    for p in at:
        a = rng.standard_normal(vocab).astype(np.float32); a[p] = 100.0; rows.append(a)
        a = np.full(vocab, -1.0, np.float32); a[p] = -0.0; a[at[-1]] = 0.0; rows.append(a)
        a = rng.standard_normal(vocab).astype(np.float32); a[p:] = np.where(rng.random(vocab - p) < 0.5, np.nan, a[p:]); a[p] = -np.nan
        rows.append(a)
        a = np.full(vocab, -np.inf, np.float32); a[p] = -3e38; rows.append(a)
        a = np.full(vocab, np.inf, np.float32); a[:p] = 1.0; rows.append(a)
    logits = np.stack(rows)
    print(f"accept edges vocab={vocab} rows={len(rows)}", flush=True)
    am = gpu_accept(ws, logits, np.zeros(len(rows) - 1, np.int32))[2]
    assert np.array_equal(am, np.argmax(logits, axis=1))


def segment(n_rows, vocab):
    """The host's segment size: the smallest that keeps to 140 workgroups, else the largest."""
    for seg in (4096, 8192):
        if n_rows * -(-vocab // seg) <= 140:
            return seg
    return 16384


@pytest.mark.parametrize("seg,n,vocab", [(s, n, m * s + d) for s, n, m in ((4096, 5, 3), (8192, 20, 4), (16384, 33, 3))
                                         for d in (-4, -1, 0, 1, 4)])
def test_accept_around_each_segment(ws, seg, n, vocab):
    """Each segment size in both load widths, rows that end just before, at and just past a segment: every row's largest value, a
    tie behind it or its first NaN at the last place of one segment and the first of the next."""
    assert segment(n, vocab) == seg
    rng = np.random.default_rng(vocab)
    logits = rng.standard_normal((n, vocab)).astype(np.float32)
    at = [p for p in (0, 3, 4, seg - 1, seg, seg + 1, 2 * seg - 1, 2 * seg, vocab - 2, vocab - 1)]
    for i in range(n):
        p, kind = at[i % len(at)], i % 3
        logits[i, p] = np.nan if kind == 2 else 50.0
        if kind == 1:
            logits[i, at[(i + 3) % len(at)]] = 50.0
        if kind == 2:
            logits[i, at[(i + 5) % len(at)]] = -np.nan
    print(f"accept seg={seg} rows={n} vocab={vocab}", flush=True)
    am = gpu_accept(ws, logits, np.zeros(n - 1, np.int32))[2]
    assert np.array_equal(am, np.argmax(logits, axis=1))


@pytest.mark.parametrize("vocab", [12 * 16384 + 5, 12 * 16384 + 4, 262144])
def test_accept_several_segments_per_workgroup(ws, vocab):
    """64 rows of 13 or 16 segments: 832 or 1,024 workgroups of one segment become 256 of four (the last one shorter), in both
    load widths; ties and NaN in different segments of one workgroup and across workgroups."""
    n = 64
    rng = np.random.default_rng(77)
    logits = rng.standard_normal((n, vocab)).astype(np.float32)
    at = rng.integers(0, vocab, n); at[:4] = [0, vocab - 1, 4 * 16384 - 1, 4 * 16384]
    logits[np.arange(n), at] = 50.0
    logits[5, at[5]:] = np.nan
    for i, (p, q) in enumerate([(16383, 16384), (100, 3 * 16384 + 7), (2 * 16384, 4 * 16384), (16384 + 5, vocab - 1)]):
        logits[8 + 2 * i, [p, q]] = 60.0                               # a tie: the lower index
        logits[9 + 2 * i, q] = np.nan; logits[9 + 2 * i, p] = -np.nan   # the first NaN
    am = gpu_accept(ws, logits, np.zeros(n - 1, np.int32))[2]
    assert np.array_equal(am, np.argmax(logits, axis=1))


def test_accept_repeated_calls_reset_counter(ws):
    rng = np.random.default_rng(9)
    for it in range(5):
        logits, draft = planted(rng, it * 3, vocab=20000)
        assert gpu_accept(ws, logits, draft)[:2] == orc.accept(logits, draft)[:2]


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0])
def test_device_quantizer_bitexact(fmt):
    rng = np.random.default_rng(3 + fmt)
    nb = 20000
    x = rng.standard_normal(nb * 32).astype(np.float32) * np.repeat(10.0 ** rng.uniform(-6, 4, nb), 32).astype(np.float32)
    x[:32] = 0.0
    x[32:64] = np.arange(32, dtype=np.float32) - 16.0
    x[64:96] = 0.5
    x[96:128] = -3.0
    x[128:160] = np.tile([2.0, -2.0], 16)                  # equal magnitudes, opposite signs: the first (+) sets q4_0's d
    x[160:192] = np.tile([-2.0, 2.0], 16)                  # ... the first (-)
    x[192:224] = -0.0                                      # an all -0 block: max stays +0, q4_0's d is -0
    x[224:256] = rng.uniform(-1, 1, 32)
    x[224 + 30], x[224 + 31] = -5.0, 5.0                   # the largest magnitude twice, at the block's end
    x[256:288] = rng.uniform(-1, 1, 32)
    x[256 + 17] = 7.0                                      # in the second half (the other 16 lanes' reduction)
    dx = bb.DeviceBuffer.from_array(x)
    hb = 34 if fmt == bb.FMT_Q8_0 else 18
    dy = bb.DeviceBuffer(nb * hb)
    bb.quantize_device(fmt, dx.ptr, dy.ptr, x.size)
    bb.device_sync()
    assert np.array_equal(dy.download(np.uint8), orc.quantize(fmt, x))


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
def test_synth_pages_match_oracle_generator(fmt):
    """libpa_synth's device generator writes the oracle's rows (same stream, same quantizer)."""
    nkv, hd, nk = 8, 128, 777
    hb = bb.head_bytes(fmt, hd)
    rs = nkv * hb
    ch = orc.outlier_channels(42, nkv, hd, 4)
    dch = bb.DeviceBuffer.from_array(ch)
    buf = bb.DeviceBuffer(nk * rs)
    assert bb.synth().pa_synth_fill_rows(buf.ptr, fmt, nkv, hd, rs, 100, nk, 42, 1.0, 4, dch.ptr, 8.0, None) == 0
    bb.device_sync()
    got = buf.download(np.uint8)
    ref = orc.fill_rows(42, fmt, nkv, hd, nk, j0=100, n_outliers=4, outlier_mul=8.0)
    mism = int((got != ref).sum())
    print("synth byte mismatches:", mism, "of", ref.size)
    assert mism == 0
