"""HIP-graph capture of the device engine path: a captured pa_hip_attn / pa_hip_attn_reply call, replayed several times
with eager work and synchronisations between the replays, must give the eager result bit for bit on every replay
(the kernels are deterministic; the call enqueues no memset, so nothing in the graph depends on a memset node).

The workspace is sized by one eager call before the capture (a capture may not allocate)."""
import numpy as np
import pytest

import backburner_amd as bb
import oracle as orc

pytestmark = pytest.mark.gpu

# decode (split-K + the wide merge), verify (MMA kernel + merge), prefill-like (MMA kernel, few slots), hd 256
CASES = [
    (bb.FMT_Q8_0, 8, 8, 128, 8192, bb.QMODE_GGML),
    (bb.FMT_Q4_0, 8, 128, 128, 3000, bb.QMODE_GGML),
    (bb.FMT_Q8_0, 2, 1024, 128, 2048, bb.QMODE_GGML),
    (bb.FMT_Q8_0, 2, 48, 256, 1500, bb.QMODE_F16),
]


@pytest.mark.parametrize("fmt,nkv,rows,hd,nk,qmode", CASES)
@pytest.mark.parametrize("reply", [False, True])
def test_graph_replays_match_eager(fmt, nkv, rows, hd, nk, qmode, reply):
    print(f"graph fmt={fmt} nkv={nkv} rows={rows} hd={hd} nk={nk} reply={reply}", flush=True)
    syn = bb.synth()
    hb = orc.head_bytes(fmt, hd); rs = nkv * hb
    K = orc.fill_rows(80 + rows, fmt, nkv, hd, nk, rs=rs); V = orc.fill_rows(81 + rows, fmt, nkv, hd, nk, rs=rs)
    Q = orc.normal(82 + rows, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    Q2 = orc.normal(83 + rows, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    shape = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs)
    pages = bb.pages_from_rows(K, V, rs, 4096)
    n = nkv * rows
    ws = bb.Workspace()
    stream = syn.pa_synth_stream_new()
    dq = bb.DeviceBuffer.from_array(Q); dq2 = bb.DeviceBuffer.from_array(Q2)
    out_bytes = n * hd * (2 if reply else 4) + n * (4 if reply else 8)
    dout = bb.DeviceBuffer(out_bytes); dout2 = bb.DeviceBuffer(out_bytes)

    def call(q, out, st):
        if reply:
            ws.attn_reply(shape, pages, q.ptr, out.ptr, out.ptr + n * hd * 2, st)
        else:
            ws.attn(shape, pages, q.ptr, out.ptr, out.ptr + n * hd * 4, out.ptr + n * hd * 4 + n * 4, st)

    gx = None
    try:
        call(dq, dout, stream)                                       # eager: sizes the workspace, gives the answer
        assert syn.pa_synth_stream_sync(stream) == 0
        want = dout.download(np.uint8)
        call(dq2, dout2, stream)                                     # another problem's answer, to tell them apart
        assert syn.pa_synth_stream_sync(stream) == 0
        other = dout2.download(np.uint8)
        assert not np.array_equal(want, other)
        assert syn.pa_synth_capture_begin(stream) == 0
        call(dq, dout, stream)
        gx = syn.pa_synth_capture_end(stream)
        assert gx, "capture failed"
        for rep in range(4):
            dout.upload(np.full(out_bytes, 0x7f, np.uint8))          # poison: every replay must write everything
            assert syn.pa_synth_graph_launch(gx, stream) == 0
            assert syn.pa_synth_stream_sync(stream) == 0
            got = dout.download(np.uint8)
            assert np.array_equal(got, want), f"replay {rep} differs from the eager call"
            call(dq2, dout2, stream)                                 # eager work on the same workspace between replays
            assert syn.pa_synth_stream_sync(stream) == 0
            assert np.array_equal(dout2.download(np.uint8), other)
    finally:
        if gx:
            syn.pa_synth_graph_free(gx)
        ws.close()
        pages.close()


def test_graph_replays_accept():
    """pa_hip_accept captured in a graph (its completion counter is reset by the kernel itself, no memset): every replay
    over poisoned output equals the eager call, and the counter stays usable for the eager calls in between."""
    print("graph accept", flush=True)
    syn = bb.synth()
    rng = np.random.default_rng(44)
    logits = rng.standard_normal((17, 151936)).astype(np.float32)
    draft = rng.integers(0, 151936, 16).astype(np.int32)
    for i in range(6):
        logits[i, draft[i]] = logits[i].max() + 1.0
    dl, dd, do = bb.DeviceBuffer.from_array(logits), bb.DeviceBuffer.from_array(draft), bb.DeviceBuffer(19 * 4)
    ws = bb.Workspace()
    stream = syn.pa_synth_stream_new()
    gx = None
    try:
        ws.accept(dl.ptr, 17, 151936, dd.ptr, do.ptr, stream)
        assert syn.pa_synth_stream_sync(stream) == 0
        want = do.download(np.int32)
        k, bonus, am = orc.accept(logits, draft)
        assert want[0] == k == 6 and want[1] == bonus and np.array_equal(want[2:], am)
        assert syn.pa_synth_capture_begin(stream) == 0
        ws.accept(dl.ptr, 17, 151936, dd.ptr, do.ptr, stream)
        gx = syn.pa_synth_capture_end(stream)
        assert gx, "capture failed"
        for rep in range(4):
            do.upload(np.full(19, -7, np.int32))
            assert syn.pa_synth_graph_launch(gx, stream) == 0
            assert syn.pa_synth_stream_sync(stream) == 0
            assert np.array_equal(do.download(np.int32), want), f"replay {rep}"
            ws.accept(dl.ptr, 17, 151936, dd.ptr, do.ptr, stream)
            assert syn.pa_synth_stream_sync(stream) == 0
            assert np.array_equal(do.download(np.int32), want)
    finally:
        if gx:
            syn.pa_synth_graph_free(gx)
        ws.close()


def captured_replays(syn, ws, call, dout, stream, compare):
    """call(ws) captured on `stream` (no eager call of it before) and replayed over poisoned output, compare(bytes) each."""
    n = dout.nbytes
    assert syn.pa_synth_capture_begin(stream) == 0
    refused, gx = None, None
    try:
        call(ws)
    except bb.PaHipError as e:
        refused = str(e)
    gx = syn.pa_synth_capture_end(stream)
    try:
        assert refused is None, refused
        assert gx, "capture failed"
        for _ in range(3):
            dout.upload(np.full(n, 0x7f, np.uint8))
            assert syn.pa_synth_graph_launch(gx, stream) == 0
            assert syn.pa_synth_stream_sync(stream) == 0
            compare(dout.download(np.uint8))
    finally:
        if gx:
            syn.pa_synth_graph_free(gx)


@pytest.mark.parametrize("rows", [33, 48])
def test_accept_captured_after_a_larger_eager_call(rows):
    """One eager call of the largest shape sizes the workspace for every smaller one: 64 rows of 262,144 values take several
    segments per workgroup (256 partials), 33 and 48 rows one each (528 and 768)."""
    print(f"graph accept {rows} rows after 64", flush=True)
    syn = bb.synth()
    rng = np.random.default_rng(45)
    logits = rng.standard_normal((64, 262144), dtype=np.float32)
    draft = rng.integers(0, 262144, 63).astype(np.int32)
    for i in range(6):
        logits[i, draft[i]] = 50.0
    dl, dd = bb.DeviceBuffer.from_array(logits), bb.DeviceBuffer.from_array(draft)
    big, do = bb.DeviceBuffer(66 * 4), bb.DeviceBuffer((2 + rows) * 4)
    k, bonus, am = orc.accept(logits[:rows], draft[:rows - 1])
    want = np.concatenate([[k, bonus], am]).astype(np.int32)
    ws = bb.Workspace()
    stream = syn.pa_synth_stream_new()
    try:
        ws.accept(dl.ptr, 64, 262144, dd.ptr, big.ptr, stream)
        assert syn.pa_synth_stream_sync(stream) == 0
        captured_replays(syn, ws, lambda w: w.accept(dl.ptr, rows, 262144, dd.ptr, do.ptr, stream), do, stream,
                         lambda got: np.testing.assert_array_equal(got.view(np.int32), want))
    finally:
        ws.close()


def attn_problem(fmt, nkv, rows, hd, nk, qmode, seed):
    """shape, pages and Q of one call, and a run(ws, out, stream) of it."""
    hb = orc.head_bytes(fmt, hd); rs = nkv * hb
    rng = np.random.default_rng(seed)
    K = orc.fill_rows(seed, fmt, nkv, hd, nk, rs=rs); V = orc.fill_rows(seed + 1, fmt, nkv, hd, nk, rs=rs)
    n = nkv * rows
    dq = bb.DeviceBuffer.from_array(rng.standard_normal((n, hd), dtype=np.float32))
    shape, pages = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs), bb.pages_from_rows(K, V, rs, 4096)

    def run(ws, out, st):
        ws.attn(shape, pages, dq.ptr, out.ptr, out.ptr + n * hd * 4, out.ptr + n * hd * 4 + n * 4, st)

    def split(got):
        f = got.view(np.float32)
        return f[:n * hd].reshape(n, hd), f[n * hd:n * hd + n], f[n * hd + n:]

    return run, split, n * hd * 4 + n * 8, pages


def check_captured_after(first, then):
    """`then` captured on a workspace that has seen the eager call `first` (None: a fresh one): accepted, and every replay
    equal to the eager result on another workspace up to the fp16 rounding of P against another chunk's reference max."""
    print(f"capture {then} after {first}", flush=True)
    syn = bb.synth()
    ws, ws2 = bb.Workspace(), bb.Workspace()
    stream = syn.pa_synth_stream_new()
    held = []
    try:
        if first:
            run, _, nbytes, pages = attn_problem(*first, seed=600)
            held.append(pages)
            run(ws, bb.DeviceBuffer(nbytes), stream)
            assert syn.pa_synth_stream_sync(stream) == 0
        run, split, nbytes, pages = attn_problem(*then, seed=700)
        held.append(pages)
        dout, dref = bb.DeviceBuffer(nbytes), bb.DeviceBuffer(nbytes)
        run(ws2, dref, stream)
        assert syn.pa_synth_stream_sync(stream) == 0
        ref = split(dref.download(np.uint8))

        def compare(got):
            eo, em, el = orc.rel_err(*split(got), *ref)
            assert eo < 1e-3 and em < 1e-6 and el < 1e-3, (eo, em, el)

        captured_replays(syn, ws, lambda w: run(w, dout, stream), dout, stream, compare)
    finally:
        ws.close()
        ws2.close()
        for p in held:
            p.close()


@pytest.mark.parametrize("first,then", [
    # 10 chunks of 768 padded rows per head, then 50 of 128 that a whole round would make 64
    ((bb.FMT_Q8_0, 8, 520, 128, 6400, bb.QMODE_GGML), (bb.FMT_Q8_0, 8, 48, 128, 6400, bb.QMODE_GGML)),
    # one chunk, written directly, needs no slots (a longer context would)
    (None, (bb.FMT_Q8_0, 8, 4096, 256, 64, bb.QMODE_F16)),
])
def test_captured_call_needs_no_headroom(first, then):
    """The room that a workspace takes ahead for longer contexts is no reason to refuse a captured call whose own slots fit."""
    check_captured_after(first, then)


@pytest.mark.parametrize("first,then", [
    # 128 chunks of 64 rows per head, then 32 of 256 in 64-row blocks where 256-row blocks would take 64
    ((bb.FMT_Q8_0, 4, 48, 256, 16384, bb.QMODE_F16), (bb.FMT_F16, 4, 240, 256, 33333, bb.QMODE_F16)),
    ((bb.FMT_Q8_0, 4, 48, 256, 16384, bb.QMODE_F16), (bb.FMT_Q8_0, 4, 600, 256, 20000, bb.QMODE_GGML)),
    # one chunk of 64-row blocks, two of 256-row blocks
    (None, (bb.FMT_Q4_0, 2, 16384, 256, 12288, bb.QMODE_F16)),
])
def test_captured_head256_call_in_the_slots_of_64_row_blocks(first, then):
    """Head dim 256 over long contexts: the 256-row blocks take more chunks than the 64-row blocks that short contexts run; a
    captured call whose workspace holds the latter's count takes that."""
    check_captured_after(first, then)
