"""GPU parity of the device engine path (pa_hip_attn, through the C ABI) against the CPU oracle on the same bytes.

Tolerance: 2e-3 relative on O (per row, after rebasing to the oracle's max), on m
(relative to max(1, |m|)) and on l, against the ggml-faithful restatement (orc_attn_ggml) in PA_QMODE_GGML, and against
the fp64 closed form with the reference engines' rounding (f16(q*scale)) in PA_QMODE_F16."""
import numpy as np
import pytest

import backburner_amd as bb
import oracle as orc

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.fixture(scope="module")
def ws():
    w = bb.Workspace()
    yield w
    w.close()


def case(fmt, nkv, rows, hd, nk, seed, rs_pad=0, k_amp=1.0, outliers=0):
    hb = orc.head_bytes(fmt, hd)
    rs = nkv * hb + rs_pad
    K = orc.fill_rows(seed, fmt, nkv, hd, nk, rs=rs, amp=k_amp, n_outliers=outliers, outlier_mul=8.0)
    V = orc.fill_rows(seed + 1, fmt, nkv, hd, nk, rs=rs)
    Q = orc.normal(seed + 2, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    return K, V, Q, rs


def run_and_check(ws, fmt, nkv, rows, hd, nk, seed, qmode=bb.QMODE_GGML, page_keys=bb.PAGE, rs_pad=0, k_amp=1.0, outliers=0,
                  tol=TOL):
    print(f"case fmt={fmt} nkv={nkv} rows={rows} hd={hd} nk={nk} qmode={qmode} pages={page_keys}", flush=True)
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, seed, rs_pad, k_amp, outliers)
    shape = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs)
    O, m, l = bb.attn_host(shape, K, V, Q, page_keys=page_keys, ws=ws)
    if qmode == bb.QMODE_GGML:
        ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_GGML, rs=rs), Q, K, V, nk)
    else:
        ref = orc.attn_exact(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_F16, rs=rs), Q, K, V, nk)
    eo, em, el = orc.rel_err(O, m, l, *ref)
    assert eo < tol and em < tol and el < tol, (eo, em, el)
    return eo, em, el


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
@pytest.mark.parametrize("rows", [8, 48, 128, 300])
@pytest.mark.parametrize("hd", [128, 256])
def test_parity_ggml(ws, fmt, rows, hd):
    run_and_check(ws, fmt, 2, rows, hd, 1000, seed=100 + rows + hd + fmt, page_keys=512)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
@pytest.mark.parametrize("rows", [9, 32, 33, 64, 100, 160, 224])
def test_mma_row_blocks(ws, fmt, rows):
    """One row block narrower than the workgroup's waves: 4 waves up to 128 rows (9-64 rows leave one to three waves
    that only stage; 100 rows leave none), 8 waves above (160 and 224 rows leave three and one)."""
    run_and_check(ws, fmt, 2, rows, 128, 1500, seed=300 + rows + fmt, page_keys=512)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0])
@pytest.mark.parametrize("nkv,rows", [(1, 8), (3, 8), (3, 128)])
def test_odd_kv_heads(ws, fmt, nkv, rows):
    """An odd KV-head count has no head pairs for the decode kernel: decode goes to the matrix-core kernel (one live
    wave per row block) and verify keeps its full row blocks; both over ragged pages."""
    run_and_check(ws, fmt, nkv, rows, 128, 2100, seed=500 + 10 * nkv + rows + fmt, page_keys=1000)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
@pytest.mark.parametrize("rows", [8, 48])
def test_parity_reference_rounding(ws, fmt, rows):
    run_and_check(ws, fmt, 4, rows, 256, 700, seed=7 + rows + fmt, qmode=bb.QMODE_F16, page_keys=256)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
@pytest.mark.parametrize("rows", [6, 16, 18, 48, 64, 96, 150])
def test_mma256_row_blocks(ws, fmt, rows):
    """Head dim 256 with fp16 queries (the reference engines' f16(q*scale)) on the matrix-core kernel: 16 rows per wave,
    64-row blocks. 6 to 48 rows leave one to three waves that only stage, 64 rows none; 96 and 150 rows take several
    row blocks, the last one partly past the rows."""
    run_and_check(ws, fmt, 2, rows, 256, 1500, seed=700 + rows + fmt, qmode=bb.QMODE_F16, page_keys=512)


@pytest.mark.parametrize("fmt,rows,qmode", [(f, r, bb.QMODE_F16) for f in (bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16) for r in (65, 224, 225, 257)]
                         + [(f, r, bb.QMODE_GGML) for f in (bb.FMT_Q8_0, bb.FMT_Q4_0) for r in (513, 577)])
def test_head256_wide_rows(ws, fmt, rows, qmode):
    """Head dim 256 above 64 rows over one head and 387 tiles, about where the host weighs 64-row blocks against 256-row ones:
    the first rows past a 64-row block, the last count with idle waves, the first without, a further row block of one row or
    wave; over pages that end inside a tile, hold less than one or nothing, in the default chunks, in one chunk per row block
    (every page change inside the workgroup) and in chunks of one or two tiles."""
    page_keys = [500, 7, 0, 64, 11740]
    nk, nkv = sum(page_keys), 1
    print(f"case fmt={fmt} rows={rows} qmode={qmode} nk={nk}", flush=True)
    K, V, Q, rs = case(fmt, nkv, rows, 256, nk, 1700 + rows + fmt)
    shape = bb.make_shape(nkv, rows, 256, fmt, qmode, rs=rs)
    oshape = orc.make_shape(nkv, rows, 256, fmt, orc.QMODE_F16 if qmode == bb.QMODE_F16 else orc.QMODE_GGML, rs=rs)
    ref = (orc.attn_exact if qmode == bb.QMODE_F16 else orc.attn_ggml)(oshape, Q, K, V, nk)
    for workgroups in (0, 1, 800):
        ws.set_split(mma_workgroups=workgroups)
        try:
            O, m, l = bb.attn_host(shape, K, V, Q, page_keys=page_keys, ws=ws)
        finally:
            ws.set_split()
        eo, em, el = orc.rel_err(O, m, l, *ref)
        assert eo < TOL and em < TOL and el < TOL, (workgroups, eo, em, el)


def run_and_check_rows(ws, fmt, nkv, rows, hd, page_keys, pick, seed, qmode, rs_pad=0, outliers=0, workgroups=(0,)):
    """A call of many rows over a long context, checked at the rows `pick` of every head (the oracle runs those only): each
    row's result depends on its own query."""
    nk = sum(page_keys)
    print(f"case fmt={fmt} nkv={nkv} rows={rows} hd={hd} nk={nk} qmode={qmode} pages={len(page_keys)}", flush=True)
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, seed, rs_pad, 1.0, outliers)
    shape = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs)
    at = np.concatenate([h * rows + np.asarray(pick) for h in range(nkv)])
    oshape = orc.make_shape(nkv, len(pick), hd, fmt, orc.QMODE_F16 if qmode == bb.QMODE_F16 else orc.QMODE_GGML, rs=rs)
    ref = (orc.attn_exact if qmode == bb.QMODE_F16 else orc.attn_ggml)(oshape, np.ascontiguousarray(Q[at]), K, V, nk)
    pages = bb.pages_from_rows(K, V, rs, page_keys)
    n = nkv * rows
    dq, do, dml = bb.DeviceBuffer.from_array(Q), bb.DeviceBuffer(n * hd * 4), bb.DeviceBuffer(n * 8)
    try:
        for w in workgroups:
            ws.set_split(mma_workgroups=w)
            do.upload(np.full(n * hd * 4, 0x7f, np.uint8))
            ws.attn(shape, pages, dq.ptr, do.ptr, dml.ptr, dml.ptr + n * 4)
            bb.device_sync()
            O, ml = do.download(np.float32).reshape(n, hd), dml.download(np.float32)
            eo, em, el = orc.rel_err(O[at], ml[:n][at], ml[n:][at], *ref)
            assert eo < TOL and em < TOL and el < TOL, (w, eo, em, el)
    finally:
        ws.set_split()
        pages.close()


# head dim 256 where 256-row blocks (mma_kernel) are clearly the faster ones, so that the host's estimate takes them: 65-128
# rows over 4 heads from 16,000 keys, 200 rows from 32,000, more rows and heads over 16,000-33,000; in exact block dots above 512
WIDE = [(bb.FMT_Q8_0, bb.QMODE_F16, 4, 65, 16100), (bb.FMT_Q4_0, bb.QMODE_F16, 3, 96, 24100), (bb.FMT_F16, bb.QMODE_F16, 4, 97, 24100),
        (bb.FMT_F16, bb.QMODE_GGML, 4, 72, 24100), (bb.FMT_Q8_0, bb.QMODE_F16, 4, 200, 33100), (bb.FMT_Q4_0, bb.QMODE_F16, 4, 224, 33100),
        (bb.FMT_F16, bb.QMODE_GGML, 4, 257, 33100), (bb.FMT_Q4_0, bb.QMODE_F16, 4, 225, 33100), (bb.FMT_Q8_0, bb.QMODE_F16, 3, 513, 24100),
        (bb.FMT_F16, bb.QMODE_F16, 2, 1100, 24100), (bb.FMT_Q8_0, bb.QMODE_GGML, 2, 769, 33100), (bb.FMT_Q4_0, bb.QMODE_GGML, 3, 545, 33100)]


@pytest.mark.parametrize("fmt,qmode,nkv,rows,nk", WIDE)
def test_head256_long_contexts(ws, fmt, qmode, nkv, rows, nk):
    """256-row blocks at head dim 256: several KV heads (their place in the pages, Q, the slots and the result), padded rows,
    outlier keys in the exact block dots, f16 K in ggml's rounding (the scale multiplies the score), idle waves or none, a
    last row block of one row or wave, pages that end inside a tile or hold nothing; in the default chunks and in one per row
    block."""
    exact = qmode == bb.QMODE_GGML and fmt != bb.FMT_F16
    pages = [4096, 500, 7, 0, 64, 4096, 1000]
    pages += [nk - sum(pages)]
    edge = {0, 1, 31, 32, 63, 64, rows // 2, rows - 2, rows - 1} | {r for r in (255, 256, 511, 512) if r < rows}
    run_and_check_rows(ws, fmt, nkv, rows, 256, pages, sorted(edge), 2600 + rows + fmt, qmode, rs_pad=48, outliers=4 if exact else 0,
                       workgroups=(0, 1))


@pytest.mark.parametrize("fmt,qmode,rows", [(bb.FMT_Q8_0, bb.QMODE_F16, 72), (bb.FMT_Q4_0, bb.QMODE_GGML, 1100)])
def test_head256_over_two_launches(ws, fmt, qmode, rows):
    """256-row blocks over 150 pages: two launches into one slot array."""
    r = np.random.default_rng(rows)
    pages = [int(x) for x in r.integers(200, 330, size=150)]
    run_and_check_rows(ws, fmt, 4, rows, 256, pages, [0, 33, 64, rows - 1], 2800 + rows, qmode)


@pytest.mark.parametrize("nkv,rows,hd,nk", [(8, 128, 128, 1000), (8, 1000, 128, 2049), (4, 48, 256, 4096), (4, 300, 256, 70), (8, 64, 128, 33)])
def test_short_context_split(ws, nkv, rows, hd, nk):
    """Short contexts take fewer chunks than the workgroups that fit (down to one, written directly): the default split
    against the same call in one chunk and in as many as it has tiles."""
    K, V, Q, rs = case(bb.FMT_Q8_0, nkv, rows, hd, nk, 2300 + rows)
    shape = bb.make_shape(nkv, rows, hd, bb.FMT_Q8_0, rs=rs)
    print(f"case nkv={nkv} rows={rows} hd={hd} nk={nk}", flush=True)
    outs = []
    for workgroups in (0, 1, 100000):
        ws.set_split(mma_workgroups=workgroups)
        try:
            outs.append(bb.attn_host(shape, K, V, Q, ws=ws))
        finally:
            ws.set_split()
    for O, m, l in outs[1:]:                                  # the fp16 rounding of P against another reference max
        eo, em, el = orc.rel_err(O, m, l, *outs[0])
        assert eo < 1e-3 and em < 1e-6 and el < 1e-3, (eo, em, el)


@pytest.mark.parametrize("fmt,qmode,nkv,rows,hd,nk", [
    (bb.FMT_F16, bb.QMODE_GGML, 8, 120, 128, 983), (bb.FMT_F16, bb.QMODE_F16, 8, 64, 128, 702), (bb.FMT_F16, bb.QMODE_GGML, 8, 784, 128, 256),
    (bb.FMT_Q4_0, bb.QMODE_GGML, 8, 40, 128, 1807), (bb.FMT_Q8_0, bb.QMODE_F16, 8, 232, 128, 256), (bb.FMT_Q8_0, bb.QMODE_GGML, 4, 426, 256, 256),
    (bb.FMT_F16, bb.QMODE_F16, 4, 48, 256, 3141), (bb.FMT_F16, bb.QMODE_F16, 4, 1236, 256, 256)])
def test_short_context_error(ws, fmt, qmode, nkv, rows, hd, nk):
    """A short context in fewer chunks than it has tiles is as exact as with one tile per chunk: every tile's probabilities are
    taken against its own maximum, so that the largest of each tile is 1 in fp16 either way. The chunks then differ by fp32
    merging only, 1e-7 of errors of 1e-4: 1 % of them is far above that (with one reference per chunk: 1.1 to 1.6 times)."""
    print(f"case fmt={fmt} qmode={qmode} nkv={nkv} rows={rows} hd={hd} nk={nk}", flush=True)
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, 2400 + rows, outliers=4)
    shape = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs)
    ref = orc.attn_exact(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_F16 if qmode == bb.QMODE_F16 else orc.QMODE_GGML, rs=rs), Q, K, V, nk)
    err = []
    for workgroups in (0, 100000):                            # the default, one tile per chunk
        ws.set_split(mma_workgroups=workgroups)
        try:
            O, m, l = bb.attn_host(shape, K, V, Q, ws=ws)
        finally:
            ws.set_split()
        D = O.astype(np.float64) * np.exp(m.astype(np.float64) - ref[1])[:, None] - ref[0]
        err.append(np.linalg.norm(D) / np.linalg.norm(ref[0]))
    print(f"error of O: default {err[0]:.3e}, one tile per chunk {err[1]:.3e}", flush=True)
    assert err[0] < 1.01 * err[1], err


@pytest.mark.parametrize("amps", [(30, 0.01, 0.01, 0.01, 0.01, 0.01, 0.01, 0.01, 0.01, 0.01), (0.01, 0.1, 1, 3, 10, 30, 40, 50, 60, 70),
                                  (50, 1, 50, 0.1, 20, 0.01, 60, 1, 0.01, 40), (60, 50, 40, 30, 25, 20, 15, 10, 5, 1)])
@pytest.mark.parametrize("fmt,qmode,nkv,rows,hd", [(bb.FMT_F16, bb.QMODE_F16, 8, 1500, 128), (bb.FMT_Q8_0, bb.QMODE_GGML, 8, 1500, 128),
                                                   (bb.FMT_Q4_0, bb.QMODE_GGML, 8, 64, 128), (bb.FMT_Q8_0, bb.QMODE_F16, 4, 1536, 256),
                                                   (bb.FMT_Q4_0, bb.QMODE_GGML, 4, 1536, 256)])
def test_tile_maxima_far_apart(ws, fmt, qmode, nkv, rows, hd, amps):
    """Keys whose size changes by the tile, so that a row's tile maxima rise, fall and alternate by hundreds of powers of two
    within one chunk: a tile's reference follows its maximum no further down than 2^20 below the row's largest, and nothing
    overflows or is lost."""
    nk = 32 * len(amps) - 5
    X = np.random.default_rng(rows + hd + len(amps)).standard_normal((nk, nkv, hd), dtype=np.float32)
    X *= np.repeat(np.array(amps, np.float32), 32)[:nk, None, None]
    hb = orc.head_bytes(fmt, hd); rs = nkv * hb
    K = orc.rows_from_f32(fmt, X, rs, hb)
    V = orc.fill_rows(3, fmt, nkv, hd, nk, rs=rs)
    Q = orc.normal(5, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    print(f"case fmt={fmt} qmode={qmode} nkv={nkv} rows={rows} hd={hd} amps={amps}", flush=True)
    O, m, l = bb.attn_host(bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs), K, V, Q, ws=ws)
    f16q = qmode == bb.QMODE_F16
    ref = orc.attn_exact(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_F16 if f16q else orc.QMODE_GGML, rs=rs), Q, K, V, nk)
    assert np.isfinite(O).all() and np.isfinite(m).all() and np.isfinite(l).all()
    # Scores of hundreds magnify what a score is rounded by: quantized K in fp16 operands by 2^-11 of it, and the exact block dots
    # at head dim 128, whose row scale is a pair of fp16 values, by up to |dot| dk 2^-25 per block, here 2^17 * 2 * 2^-25 = 0.8 %.
    # Those two are compared with the same call in one tile per chunk, the others with the oracle.
    eo, em, el = orc.rel_err(O, m, l, *ref)
    print(f"max rel err O {eo:.2e} m {em:.2e} l {el:.2e}", flush=True)
    if fmt == bb.FMT_F16 or (hd == 256 and not f16q):
        assert eo < TOL and em < TOL and el < TOL, (eo, em, el)
    else:
        ws.set_split(mma_workgroups=100000)                   # the same scores, one tile per chunk
        try:
            one = bb.attn_host(bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs), K, V, Q, ws=ws)
        finally:
            ws.set_split()
        eo, em, el = orc.rel_err(O, m, l, *one)
        assert eo < 1e-3 and em < 1e-6 and el < 1e-3, (eo, em, el)


@pytest.mark.parametrize("qmode", [bb.QMODE_GGML, bb.QMODE_F16])
@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0, bb.FMT_F16])
@pytest.mark.parametrize("rows", [9, 33, 64])
def test_two_streams(ws, fmt, rows, qmode):
    """Up to 64 rows over long chunks (two tile streams per workgroup, folded through LDS): chunks of 36 tiles (the last
    one shorter) and one chunk of all 73, an odd count whose last step has one tile, over pages that end inside a step, hold
    less than a tile or nothing."""
    for workgroups in (4, 1):
        ws.set_split(mma_workgroups=workgroups)
        try:
            run_and_check(ws, fmt, 2, rows, 128, 2281, seed=1900 + rows + fmt, qmode=qmode, page_keys=[1000, 7, 0, 64, 1210])
        finally:
            ws.set_split()


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_F16])
def test_mma256_split_invariance(ws, fmt):
    """The head-dim-256 kernel at the reference's 48 rows x 4 KV heads over chunks of 1, 2, 3, 5 and 40 tiles and one
    chunk holding all 157 tiles (written directly): each split within the bar of the fp64 form, splits agreeing to the
    fp16 rounding of P."""
    nkv, rows, hd, nk = 4, 48, 256, 5000
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, 811 + fmt)
    shape = bb.make_shape(nkv, rows, hd, fmt, bb.QMODE_F16, rs=rs)
    ref = orc.attn_exact(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_F16, rs=rs), Q, K, V, nk)
    outs = []
    for want in (200, 100, 60, 35, 4, 1):
        print("mma256 split: workgroups", want * nkv, flush=True)
        ws.set_split(mma_workgroups=want * nkv)
        try:
            outs.append(bb.attn_host(shape, K, V, Q, page_keys=1500, ws=ws))
        finally:
            ws.set_split()
        eo, em, el = orc.rel_err(*outs[-1], *ref)
        assert eo < TOL and em < TOL and el < TOL, (want, eo, em, el)
    for O, m, l in outs[1:]:
        eo, em, el = orc.rel_err(O, m, l, *outs[0])
        assert eo < 1e-3 and em < 1e-6 and el < 1e-3, (eo, em, el)


def test_outlier_channels_and_padding(ws):
    """K with 4 x8 outlier channels per head (the long-context decode configuration) and rows padded past nkv*hb."""
    run_and_check(ws, bb.FMT_Q8_0, 8, 8, 128, 2048, seed=31, rs_pad=16, outliers=4)


@pytest.mark.parametrize("pages", [[3, 0, 64, 1, 130], [1], [4096, 4096, 17], [10] * 140, [1024, 1024, 1024, 5000], [64] * 140,
                                   [96, 96, 96], [512, 1024, 512]])
def test_ragged_pages(ws, pages):
    """Uneven page sizes, empty pages, single keys and more pages than one launch holds (140 > 128); equal power-of-two
    pages (found by shift in the decode kernel) with a shorter or a longer last page, in one launch and over two, and
    equal pages that are not a power of two of tiles or a longer page in the middle (found by the page-table walk)."""
    run_and_check(ws, bb.FMT_Q8_0, 2, 8, 128, sum(pages), seed=5 + len(pages), page_keys=pages)


@pytest.mark.parametrize("rows", [8, 128, 512])
def test_empty(ws, rows):
    shape = bb.make_shape(2, rows, 128, bb.FMT_Q8_0)
    Q = orc.normal(1, 0, 2 * rows * 128).reshape(2 * rows, 128)
    O, m, l = bb.attn_host(shape, np.zeros(0, np.uint8), np.zeros(0, np.uint8), Q, page_keys=[], ws=ws)
    assert np.all(O == 0) and np.all(np.isneginf(m)) and np.all(l == 0)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0])
def test_split_invariance(ws, fmt):
    """Splitting the keys over tile groups (split-K slots folded by the merge kernel, or one group writing the result
    itself) changes the result only by where P is rounded to fp16 (relative to a different running max): l and m agree
    to fp32 reordering, O within the P rounding (~2^-11 per weight); every split is also within the parity bar of the
    oracle."""
    K, V, Q, rs = case(fmt, 2, 8, 128, 5000, 77)            # pages of 1500 keys: 157 tiles
    shape = bb.make_shape(2, 8, 128, fmt, rs=rs)
    ref = orc.attn_ggml(orc.make_shape(2, 8, 128, fmt, orc.QMODE_GGML, rs=rs), Q, K, V, 5000)
    outs = []
    for groups in (1, 3, 17, 40, 64, 157):
        print("split: decode groups", groups, flush=True)
        ws.set_split(decode_groups=groups)
        try:
            outs.append(bb.attn_host(shape, K, V, Q, page_keys=1500, ws=ws))
        finally:
            ws.set_split()
        eo, em, el = orc.rel_err(*outs[-1], *ref)
        assert eo < TOL and em < TOL and el < TOL, (groups, eo, em, el)
    for O, m, l in outs[1:]:
        eo, em, el = orc.rel_err(O, m, l, *outs[0])
        assert eo < 1e-3 and em < 1e-6 and el < 1e-5, (eo, em, el)


@pytest.mark.parametrize("fmt", [bb.FMT_Q8_0, bb.FMT_Q4_0])
@pytest.mark.parametrize("rows", [128, 512])
def test_mma_split_invariance(ws, fmt, rows):
    """The verify / prefill kernel over chunks of 1, 2, 3, 5 and 40 tiles (the two-tile register prefetch with its
    empty-range loads past a chunk's end, uneven last chunks) and one chunk holding every tile (the result written
    directly): each split is within the parity bar of the oracle, and splits agree with each other to the fp16
    rounding of P, which the split moves (P is rounded relative to a different running max), in O and in l (the sum
    of the same fp16 P that the PV product uses, 2^-11 per term at most), and on m to fp32 rounding."""
    nkv, hd, nk = 2, 128, 5000                                # pages of 1500 keys: 157 tiles
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, 91 + rows)
    shape = bb.make_shape(nkv, rows, hd, fmt, rs=rs)
    ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_GGML, rs=rs), Q, K, V, nk)
    units = nkv * (2 if rows == 512 else 1)                   # KV heads x row blocks (256 rows per block at 512 rows)
    outs = []
    for want in (200, 100, 60, 35, 4, 1):                     # chunks of 1, 2, 3, 5, 40 and 157 tiles
        print("mma split: workgroups", want * units, flush=True)
        ws.set_split(mma_workgroups=want * units)
        try:
            outs.append(bb.attn_host(shape, K, V, Q, page_keys=1500, ws=ws))
        finally:
            ws.set_split()
        eo, em, el = orc.rel_err(*outs[-1], *ref)
        assert eo < TOL and em < TOL and el < TOL, (want, eo, em, el)
    for O, m, l in outs[1:]:
        eo, em, el = orc.rel_err(O, m, l, *outs[0])
        assert eo < 1e-3 and em < 1e-6 and el < 2.0 ** -11, (eo, em, el)


@pytest.mark.parametrize("fmt,rows,hd,qmode", [(bb.FMT_Q8_0, 8, 128, bb.QMODE_GGML), (bb.FMT_Q4_0, 128, 128, bb.QMODE_GGML),
                                               (bb.FMT_Q8_0, 48, 256, bb.QMODE_F16), (bb.FMT_Q8_0, 48, 256, bb.QMODE_GGML)])
@pytest.mark.parametrize("chunk", [64, 1000, 4096])
def test_chunk_keys(ws, fmt, rows, hd, qmode, chunk):
    """config_req.gpu_chunk (keys per workgroup, pa_hip_ws_set_chunk_keys) on the decode, verify and head-dim-256 kernels
    (fp16 queries, and ggml's rounding with exact block dots): every chunking within the parity bar of the oracle."""
    nkv, nk = 2, 5000
    print(f"chunk keys {chunk}: fmt={fmt} rows={rows} hd={hd} qmode={qmode}", flush=True)
    K, V, Q, rs = case(fmt, nkv, rows, hd, nk, 1200 + chunk + rows)
    shape = bb.make_shape(nkv, rows, hd, fmt, qmode, rs=rs)
    if qmode == bb.QMODE_GGML:
        ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_GGML, rs=rs), Q, K, V, nk)
    else:
        ref = orc.attn_exact(orc.make_shape(nkv, rows, hd, fmt, orc.QMODE_F16, rs=rs), Q, K, V, nk)
    ws.set_chunk_keys(chunk)
    try:
        out = bb.attn_host(shape, K, V, Q, page_keys=1500, ws=ws)
    finally:
        ws.set_chunk_keys(0)
    eo, em, el = orc.rel_err(*out, *ref)
    assert eo < TOL and em < TOL and el < TOL, (eo, em, el)


def test_bad_arguments(ws):
    with pytest.raises(bb.PaHipError, match="hd must be"):
        bb.attn_host(bb.make_shape(1, 8, 64, bb.FMT_Q8_0), np.zeros(68, np.uint8), np.zeros(68, np.uint8),
                     np.zeros((8, 64), np.float32), page_keys=[1], ws=ws)
    s = bb.make_shape(2, 8, 128, bb.FMT_Q8_0)
    s.rs = 100
    with pytest.raises(bb.PaHipError, match="too small"):
        bb.attn_host(s, np.zeros(100, np.uint8), np.zeros(100, np.uint8), np.zeros((16, 128), np.float32), page_keys=[1], ws=ws)


def test_decode_128k_full_size(ws):
    """The long-context decode layer at full size (131,072 q8_0 keys, 8 KV heads, GQA 8, outlier channels): GPU-made
    pages downloaded and checked against the oracle on the same bytes."""
    nkv, rows, hd, nk = 8, 8, 128, 131072
    hb = bb.head_bytes(bb.FMT_Q8_0, hd)
    rs = nkv * hb
    syn = bb.synth()
    kbuf, vbuf = bb.DeviceBuffer(nk * rs), bb.DeviceBuffer(nk * rs)
    ch = orc.outlier_channels(1001, nkv, hd, 4)
    dch = bb.DeviceBuffer.from_array(ch)
    assert syn.pa_synth_fill_rows(kbuf.ptr, 1, nkv, hd, rs, 0, nk, 1001, 1.0, 4, dch.ptr, 8.0, None) == 0
    assert syn.pa_synth_fill_rows(vbuf.ptr, 1, nkv, hd, rs, 0, nk, 1002, 1.0, 0, None, 1.0, None) == 0
    bb.device_sync()
    Q = orc.normal(1003, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    pages = bb.Pages([kbuf.ptr + i * 4096 * rs for i in range(32)], [vbuf.ptr + i * 4096 * rs for i in range(32)], [4096] * 32, [])
    dq = bb.DeviceBuffer.from_array(Q)
    do, dml = bb.DeviceBuffer(nkv * rows * hd * 4), bb.DeviceBuffer(nkv * rows * 8)
    shape = bb.make_shape(nkv, rows, hd, bb.FMT_Q8_0)
    ws.attn(shape, pages, dq.ptr, do.ptr, dml.ptr, dml.ptr + nkv * rows * 4)
    bb.device_sync()
    O = do.download(np.float32).reshape(-1, hd)
    ml = dml.download(np.float32)
    K = kbuf.download(np.uint8)
    V = vbuf.download(np.uint8)
    ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, orc.Q8_0), Q, K, V, nk)
    eo, em, el = orc.rel_err(O, ml[:nkv * rows], ml[nkv * rows:], *ref)
    print("decode 128k parity", eo, em, el)
    assert eo < TOL and em < TOL and el < TOL, (eo, em, el)


@pytest.mark.parametrize("rows", [8, 128])
def test_page_above_2p20_keys(ws, rows):
    """One page of 2^20 + 100 keys, walked in place by the decode path (8 rows) and the matrix-core path (128 rows):
    each tile's buffer range covers its own 32 rows, so a page of any length needs no split. Both against the oracle
    on the same bytes."""
    nkv, hd, nk = 2, 128, (1 << 20) + 100
    print(f"page above 2^20 keys rows={rows}", flush=True)
    rs = nkv * bb.head_bytes(bb.FMT_Q8_0, hd)
    syn = bb.synth()
    kbuf, vbuf = bb.DeviceBuffer(nk * rs), bb.DeviceBuffer(nk * rs)
    assert syn.pa_synth_fill_rows(kbuf.ptr, 1, nkv, hd, rs, 0, nk, 2001, 1.0, 0, None, 1.0, None) == 0
    assert syn.pa_synth_fill_rows(vbuf.ptr, 1, nkv, hd, rs, 0, nk, 2002, 1.0, 0, None, 1.0, None) == 0
    bb.device_sync()
    Q = orc.normal(2003 + rows, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    pages = bb.Pages([kbuf.ptr], [vbuf.ptr], [nk], [])
    dq = bb.DeviceBuffer.from_array(Q)
    do, dml = bb.DeviceBuffer(nkv * rows * hd * 4), bb.DeviceBuffer(nkv * rows * 8)
    ws.attn(bb.make_shape(nkv, rows, hd, bb.FMT_Q8_0), pages, dq.ptr, do.ptr, dml.ptr, dml.ptr + nkv * rows * 4)
    bb.device_sync()
    O = do.download(np.float32).reshape(-1, hd)
    ml = dml.download(np.float32)
    ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, orc.Q8_0), Q, kbuf.download(np.uint8), vbuf.download(np.uint8), nk)
    eo, em, el = orc.rel_err(O, ml[:nkv * rows], ml[nkv * rows:], *ref)
    print("page above 2^20 parity", eo, em, el)
    assert eo < TOL and em < TOL and el < TOL, (eo, em, el)


@pytest.mark.parametrize("fmt,rows,nk,nkv", [(bb.FMT_Q8_0, 128, 98304, 8), (bb.FMT_Q4_0, 8, 143360, 8),
                                             (bb.FMT_Q4_0, 128, 143360, 8), (bb.FMT_Q8_0, 4096, 4096, 8),
                                             (bb.FMT_Q8_0, 4096, 65536, 1)])
def test_full_size_verify_and_q4(ws, fmt, rows, nk, nkv):
    """The other full-size workloads: 16-token verify over 98,304 q8_0 keys, and 1-token decode / 16-token verify over
    143,360 q4_0 keys (8 KV heads, GQA 8, pages of 4096); the prefill chunk's 4096 rows per KV head over one page of 8
    heads, and over the full 65,536 keys for one head. GPU-made pages checked against the oracle on the same bytes."""
    hd = 128
    print(f"full size fmt={fmt} rows={rows} nk={nk}", flush=True)
    rs = nkv * bb.head_bytes(fmt, hd)
    syn = bb.synth()
    kbuf, vbuf = bb.DeviceBuffer(nk * rs), bb.DeviceBuffer(nk * rs)
    assert syn.pa_synth_fill_rows(kbuf.ptr, fmt, nkv, hd, rs, 0, nk, 3001 + fmt, 1.0, 0, None, 1.0, None) == 0
    assert syn.pa_synth_fill_rows(vbuf.ptr, fmt, nkv, hd, rs, 0, nk, 3002 + fmt, 1.0, 0, None, 1.0, None) == 0
    bb.device_sync()
    Q = orc.normal(3003 + rows, 0, nkv * rows * hd).reshape(nkv * rows, hd)
    npg = nk // 4096
    pages = bb.Pages([kbuf.ptr + i * 4096 * rs for i in range(npg)], [vbuf.ptr + i * 4096 * rs for i in range(npg)],
                     [4096] * npg, [])
    dq = bb.DeviceBuffer.from_array(Q)
    do, dml = bb.DeviceBuffer(nkv * rows * hd * 4), bb.DeviceBuffer(nkv * rows * 8)
    ws.attn(bb.make_shape(nkv, rows, hd, fmt), pages, dq.ptr, do.ptr, dml.ptr, dml.ptr + nkv * rows * 4)
    bb.device_sync()
    O = do.download(np.float32).reshape(-1, hd)
    ml = dml.download(np.float32)
    ref = orc.attn_ggml(orc.make_shape(nkv, rows, hd, fmt), Q, kbuf.download(np.uint8), vbuf.download(np.uint8), nk)
    eo, em, el = orc.rel_err(O, ml[:nkv * rows], ml[nkv * rows:], *ref)
    print("full size parity", fmt, rows, nk, eo, em, el)
    assert eo < TOL and em < TOL and el < TOL, (eo, em, el)
