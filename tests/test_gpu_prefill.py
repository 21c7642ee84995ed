"""Large-M prompt prefill (vx_model_forward of a long prompt: chunks of up to
2048 rows through vxh_rmsnorm_rows_panel, vxh_gemm_rows, vxh_rope_kv_rows,
vxh_attention_rows and vxh_swiglu_rows_panel) against the oracle, which runs the prompt one token per
forward like the reference (src/speculative.c:100-107, src/model.c:391-628).

Checked at the fp32 bar (1e-4 + 1e-3 |ref|): the last token's logits, every
cached K/V row of every layer, and the logits of a verify step run on the
prefilled cache.  The same prompt through the batched decode forward
(prefill_min_rows = 0) agrees with the large-M path at the same bar.
"""
import ctypes as C
import itertools

import numpy as np
import pytest

import _native as N
import test_gpu_gemm   # the vxh_qmat mirror
from _gguf import llama_gguf, GGML_Q4_0, GGML_Q8_0
from _native import close, max_violation
from _oracle_model import OracleModel

pytestmark = pytest.mark.gpu
O = N.oracle()


@pytest.fixture(scope="module")
def P():
    if not N.product_available():
        pytest.fail("product library not built")
    L = N.product()
    assert L.vxh_init() == 0, L.vxh_last_error()
    return L


def load(P, path, n_ctx, prefill_min_rows=None, thr=0.0):
    """The FFN gate-skip is off (threshold 0) on both sides by default: with
    ~4e5 gate decisions per prompt one may sit within rounding of 0.01 and
    move a row by ~1e-3.  test_prefill_at_gate_threshold runs the reference's
    0.01 and certifies any such decision."""
    mp = C.POINTER(N.VxModelDev)()
    assert P.vx_model_create(path.encode(), C.byref(mp)) == 0, N.product_error()
    mp.contents.config.n_ctx = n_ctx
    opt = N.VxModelOptions()
    P.vx_model_get_options(mp, C.byref(opt))
    opt.ffn_gate_threshold = thr
    if prefill_min_rows is not None:
        opt.prefill_min_rows = prefill_min_rows
    assert P.vx_model_set_options(mp, C.byref(opt)) == 0
    return mp


CASES = [
    # layers, d, heads, kv, ff, vocab, matrix type, prompt length
    (2, 256, 4, 2, 512, 512, GGML_Q4_0, 512),
    (2, 256, 8, 2, 640, 300, GGML_Q4_0, 600),
    (1, 192, 3, 3, 384, 256, GGML_Q8_0, 300),
    (1, 256, 2, 1, 256, 64, GGML_Q4_0, 300),      # head_dim 128: two chunks per attention wavefront
]


@pytest.mark.parametrize("case", CASES)
def test_prefill_matches_oracle(P, tmp_path, case):
    L, d, h, kv, ff, V, mt, n = case
    print(f"prefill {n} tokens: {L}L d{d} {h}/{kv} heads ff{ff} V{V} {'Q4_0' if mt == GGML_Q4_0 else 'Q8_0'}",
          flush=True)
    rng = np.random.default_rng(sum(case))
    path = str(tmp_path / "m.gguf")
    raw = llama_gguf(path, rng, L, d, h, kv, ff, V, std=0.05, norm_random=True, emb_type=mt, out_type=mt,
                     matrix_type=mt)
    n_ctx = 1024
    prompt = rng.integers(0, V, n).astype(np.int32)
    mp = load(P, path, n_ctx)
    mb = load(P, path, n_ctx, prefill_min_rows=0)
    try:
        got = np.zeros(V, np.float32)
        assert P.vx_model_forward(mp, prompt, n, got) == 0, N.product_error()
        assert mp.contents.cache_len == n
        base = np.zeros(V, np.float32)
        assert P.vx_model_forward(mb, prompt, n, base) == 0, N.product_error()
        hd, kvd = d // h, kv * (d // h)
        kv_gpu = []
        for l in range(L):
            k = np.zeros((n, kvd), np.float32)
            v = np.zeros((n, kvd), np.float32)
            assert P.vx_model_read_kv(mp, l, n, k, v) == 0, N.product_error()
            kv_gpu.append((k, v))
        toks = rng.integers(0, V, 5).astype(np.int32)
        ver = np.zeros((5, V), np.float32)
        assert P.vx_model_verify(mp, toks, 5, ver) == 0, N.product_error()
    finally:
        P.vx_model_destroy(mp)
        P.vx_model_destroy(mb)
    om = OracleModel(raw, L, d, h, kv, ff, V, n_ctx=n_ctx, gate_thr=0.0)
    ref = np.zeros(V, np.float32)
    assert O.or_forward(om.ptr, prompt, n, ref) == 0
    print(f"last-token logits: max |diff| {np.abs(got.astype(np.float64) - ref).max():.2e} "
          f"(batched path {np.abs(base.astype(np.float64) - ref).max():.2e})")
    assert close(got, ref), max_violation(got, ref)
    assert close(got, base), max_violation(got, base)
    kc = om.k_cache.reshape(L, n_ctx, kvd)
    vc = om.v_cache.reshape(L, n_ctx, kvd)
    for l, (k, v) in enumerate(kv_gpu):
        assert close(k, kc[l, :n]), ("K", l, max_violation(k, kc[l, :n]))
        assert close(v, vc[l, :n]), ("V", l, max_violation(v, vc[l, :n]))
    vref = np.zeros((5, V), np.float32)
    assert O.or_forward_all(om.ptr, toks, 5, vref) == 0
    print(f"verify after prefill: max |diff| {np.abs(ver.astype(np.float64) - vref).max():.2e}")
    assert close(ver, vref), max_violation(ver, vref)


@pytest.mark.parametrize("d,h,kv", [(256, 4, 2), (256, 2, 1), (192, 2, 1)])
def test_prefill_buffers_grow(P, tmp_path, d, h, kv):
    """Prompts of 60, 1300 and 2100 rows in turn on one model (the prefill
    buffers grow; 2100 is more than one chunk; at head_dim 96 the chunks stay
    at 512 rows): logits and cached rows as the batched decode forward gives
    them (fp32 bar)."""
    print(f"prefill growth d{d} {h}/{kv}", flush=True)
    rng = np.random.default_rng(d + h)
    path = str(tmp_path / "m.gguf")
    V, n_ctx, kvd = 64, 2200, kv * (d // h)
    llama_gguf(path, rng, 1, d, h, kv, 256, V, std=0.05, norm_random=True, emb_type=GGML_Q4_0, out_type=GGML_Q4_0,
               matrix_type=GGML_Q4_0)
    mp, mb = load(P, path, n_ctx), load(P, path, n_ctx, prefill_min_rows=0)
    try:
        for n in (60, 1300, 2100):
            prompt = rng.integers(0, V, n).astype(np.int32)
            out = []
            for m in (mp, mb):
                P.vx_model_kv_truncate(m, 0)
                lg, k, v = np.zeros(V, np.float32), np.zeros((n, kvd), np.float32), np.zeros((n, kvd), np.float32)
                assert P.vx_model_forward(m, prompt, n, lg) == 0, N.product_error()
                assert m.contents.cache_len == n
                assert P.vx_model_read_kv(m, 0, n, k, v) == 0, N.product_error()
                out.append((lg, k, v))
            for got, ref in zip(*out):
                assert close(got, ref), (n, max_violation(got, ref))
    finally:
        P.vx_model_destroy(mp)
        P.vx_model_destroy(mb)


def _rows_gemm(P, typ, W, X, R=None, scale=1.0, in_place=False):
    """vxh_rows_panel + vxh_gemm_rows on host arrays: Y = R + scale X W^T
    (in_place: Y is R's buffer)."""
    vp = C.c_void_p
    L = N.bind_vxh(P)
    L.vxh_qmat_alloc.argtypes = [vp, C.c_int, C.c_int, C.c_int]
    L.vxh_qmat_set_rows.argtypes = [vp, vp, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int, vp]
    L.vxh_qmat_free.argtypes = [vp]
    L.vxh_rows_panel_bytes.restype = C.c_size_t
    L.vxh_rows_panel_bytes.argtypes = [C.c_int, C.c_int]
    L.vxh_rows_panel.argtypes = [vp, C.c_int, C.c_int, C.c_int, vp, vp]
    L.vxh_gemm_rows.argtypes = [vp, vp, C.c_int, vp, C.c_int, C.c_int, vp, C.c_int, C.c_float, vp]
    M, cols = X.shape
    rows = W.shape[0]
    q = test_gpu_gemm._QMat()
    assert L.vxh_qmat_alloc(C.byref(q), typ, rows, cols) == 0, L.vxh_last_error()
    assert L.vxh_qmat_set_rows(C.byref(q), N._ptr(W), 0, rows, rows, 0, 0, None) == 0, L.vxh_last_error()
    dx = N.DevBuf(L, X)
    px = N.DevBuf(L, nbytes=L.vxh_rows_panel_bytes(M, cols))
    dy = N.DevBuf(L, nbytes=4 * M * rows)
    dr = N.DevBuf(L, R) if R is not None else None
    if in_place:
        dy.free()
        dy = dr
    try:
        assert L.vxh_rows_panel(dx.ptr, cols, M, cols, px.ptr, None) == 0, L.vxh_last_error()
        assert L.vxh_gemm_rows(C.byref(q), px.ptr, M, dy.ptr, rows, rows, dr.ptr if dr else None, rows, scale,
                               None) == 0, L.vxh_last_error()
        assert L.vxh_stream_sync(None) == 0
        return dy.get(np.float32, M * rows).reshape(M, rows)
    finally:
        for b in (dx, px, dy, dr):
            if b is not None:
                b.free()
        L.vxh_qmat_free(C.byref(q))


def _oracle_rows(typ, W, X):
    """The oracle's GEMV, one call per row, on 8 threads (ctypes releases
    the GIL), and the fp64 value of the same products."""
    from concurrent.futures import ThreadPoolExecutor
    M, cols = X.shape
    rows = W.shape[0]
    ref = np.zeros((M, rows), np.float32)
    if typ == GGML_Q4_0:
        def one(m):
            O.or_gemv_q4_0(N._ptr(W), np.ascontiguousarray(X[m]), ref[m], rows, cols)
        exact_w = N.q4_values(W)
    else:
        A = np.zeros(rows * cols, np.float32)
        O.or_dequantize_row_q8_0(N._ptr(W), A, rows * cols, 1.0)
        A = A.reshape(rows, cols)

        def one(m):
            O.or_gemv_f32(ref[m], A, np.ascontiguousarray(X[m]), rows, cols)
        exact_w = N.q8_values(W)
    with ThreadPoolExecutor(8) as ex:
        list(ex.map(one, range(M)))
    return ref, X.astype(np.float64) @ exact_w.T



@pytest.mark.parametrize("typ,rows,cols", [(GGML_Q4_0, 11008, 4096), (GGML_Q4_0, 4096, 11008),
                                           (GGML_Q8_0, 11008, 4096), (GGML_Q8_0, 4096, 11008)])
def test_rows_gemm_full_chunk(P, typ, rows, cols):
    """One 512-row prefill chunk through the 7B FFN shapes (gate/up 11008x4096
    and down 4096x11008) against the oracle GEMV of every row."""
    name = "Q4_0" if typ == GGML_Q4_0 else "Q8_0"
    print(f"rows gemm {name} {rows}x{cols} M=512", flush=True)
    rng = np.random.default_rng(rows + cols + typ)
    W = N.rand_q4_0(rng, rows, cols) if typ == GGML_Q4_0 else N.rand_q8_0(rng, rows, cols)
    X = rng.normal(0, 1, (512, cols)).astype(np.float32)
    Y = _rows_gemm(P, typ, W, X)
    ref, exact = _oracle_rows(typ, W, X)
    ok, nfb = N.parity(Y, ref, exact)
    print(f"max |d| {np.abs(Y.astype(np.float64) - ref).max():.2e}; elements on the exact-value fallback: {nfb}; "
          f"max error vs fp64: gpu {np.abs(Y - exact).max():.2e}, oracle {np.abs(ref - exact).max():.2e}")
    assert ok, max_violation(Y, ref)


@pytest.mark.parametrize("typ", [GGML_Q4_0, GGML_Q8_0])
@pytest.mark.parametrize("mag", [1e5, 1e-6, "mixed"])
def test_rows_gemm_row_scales(P, typ, mag):
    """Hidden rows far from unit size: fp16 hi/lo of 1e5 overflows and of
    1e-6 keeps a few bits, so the rows panel scales every row by a power of
    two and the GEMM epilogue scales it back.  Each output row is compared
    relative to its own size (the fp32 bar applied to Y / s, ref / s), and a
    residual R and a 0.5 scale are carried through on the way."""
    rows, cols, M = 1024, 4096, 70
    print(f"rows gemm row scales {mag} {'Q4_0' if typ == GGML_Q4_0 else 'Q8_0'}", flush=True)
    rng = np.random.default_rng(7 + typ)
    W = N.rand_q4_0(rng, rows, cols) if typ == GGML_Q4_0 else N.rand_q8_0(rng, rows, cols)
    if mag == "mixed":
        s = np.where(np.arange(M) % 2 == 0, 1e5, 1e-6)
    else:
        s = np.full(M, mag)
    X = (rng.normal(0, 1, (M, cols)) * s[:, None]).astype(np.float32)
    R = (rng.normal(0, 1, (M, rows)) * s[:, None]).astype(np.float32)
    Y = _rows_gemm(P, typ, W, X, R, 0.5)
    ref, exact = _oracle_rows(typ, W, X)
    ref = (R.astype(np.float64) + 0.5 * ref.astype(np.float64))
    exact = R.astype(np.float64) + 0.5 * exact
    assert np.all(np.isfinite(Y))
    g, o, e = (Y / s[:, None], ref / s[:, None], exact / s[:, None])
    ok, nfb = N.parity(g, o, e)
    print(f"max |d|/s {np.abs(g - o).max():.2e}; elements on the exact-value fallback: {nfb}")
    assert ok, max_violation(g, o)


@pytest.mark.parametrize("M,K", [(1, 32), (7, 1056), (64, 4096), (65, 96), (5, 4128), (7, 8192), (7, 8224), (513, 8224),
                                 (100, 11264), (9, 11296), (7, 12288), (7, 12320), (17, 18944), (33, 22560), (5, 24608),
                                 (1024, 96), (1030, 4096), (1025, 4128), (1024, 11296)])
@pytest.mark.parametrize("kind", ["rmsnorm", "rmsnorm_w", "swiglu"])
def test_rows_panel_kinds(P, kind, M, K):
    """The fused panels against the panel of the same rows from vxh_rmsnorm /
    vxh_swiglu_rows (rows in registers and longer ones, ragged row groups, odd
    block counts).  The swiglu rows are the same floats, so the panels are the
    same bytes; the norm's sum of squares may be added in another order,
    which moves 1/rms by a few of its roundings (2^-20 allowed), and the two
    fp16 parts keep 2^-21 of the row's largest."""
    print(f"rows panel {kind} M={M} K={K}", flush=True)
    vp = C.c_void_p
    L = N.bind_vxh(P)
    f, i = C.c_float, C.c_int
    L.vxh_rows_panel_bytes.restype, L.vxh_rows_panel_bytes.argtypes = C.c_size_t, [i, i]
    L.vxh_rows_panel.argtypes = [vp, i, i, i, vp, vp]
    L.vxh_rmsnorm.argtypes = [vp, i, i, i, vp, vp, i, vp]
    L.vxh_swiglu_rows.argtypes = [vp, i, i, i, f, vp, i, vp]
    L.vxh_rmsnorm_rows_panel.argtypes = [vp, i, i, i, vp, vp, vp]
    L.vxh_swiglu_rows_panel.argtypes = [vp, i, i, i, f, vp, vp]
    rng = np.random.default_rng(M + K)
    ld = 2 * K if kind == "swiglu" else K + 4
    x = (rng.normal(0, 1, (M, ld)) * np.exp(rng.normal(0, 3, (M, 1)))).astype(np.float32)
    w = rng.normal(1, 0.2, K).astype(np.float32)
    dx, dw, dh = N.DevBuf(L, x), N.DevBuf(L, w), N.DevBuf(L, nbytes=4 * M * K)
    nb = L.vxh_rows_panel_bytes(M, K)
    pa, pb = (N.DevBuf(L, np.zeros(nb, np.uint8)) for _ in range(2))
    wp = dw.ptr if kind == "rmsnorm_w" else None
    if kind == "swiglu":
        assert L.vxh_swiglu_rows(dx.ptr, ld, M, K, 0.01, dh.ptr, K, None) == 0
        assert L.vxh_swiglu_rows_panel(dx.ptr, ld, M, K, 0.01, pb.ptr, None) == 0
    else:
        assert L.vxh_rmsnorm(dx.ptr, ld, M, K, wp, dh.ptr, K, None) == 0
        assert L.vxh_rmsnorm_rows_panel(dx.ptr, ld, M, K, wp, pb.ptr, None) == 0
    assert L.vxh_rows_panel(dh.ptr, K, M, K, pa.ptr, None) == 0
    assert L.vxh_stream_sync(None) == 0
    a, b = pa.get(np.uint8, nb), pb.get(np.uint8, nb)
    rows, n_pairs = (M + 63) // 64 * 64, (K + 63) // 64

    def decode(p):
        """[row][column] of a panel, row scales applied."""
        s = p[:rows * n_pairs * 256].view(np.float16).astype(np.float64)
        s = s.reshape(rows // 64, n_pairs, 2, 2, 2, 2, 2, 32, 8)   # rg, pair, mt, blk, s, hi/lo, half, row, element
        v = s.sum(axis=5).transpose(0, 2, 6, 1, 3, 5, 4, 7)        # rg, mt, row, pair, blk, half, s, element
        v = v.reshape(rows, n_pairs * 64)
        rs = p[rows * n_pairs * 256:][:4 * M].view(np.float32).astype(np.float64)
        return v[:M] * rs[:, None], v[M:]

    (va, ta), (vb, tb) = decode(a), decode(b)
    h = dh.get(np.float32, M * K).reshape(M, K).astype(np.float64)
    assert not ta.any() and not tb.any() and not vb[:, K:].any()
    assert np.all(np.abs(va[:, :K] - h) <= 2.0 ** -22 * np.abs(h).max(axis=1, keepdims=True))
    if kind == "swiglu":
        assert np.array_equal(a, b)
    else:
        assert np.all(np.abs(vb[:, :K] - h) <= 2.0 ** -20 * np.abs(h) + 2.0 ** -21 * np.abs(h).max(axis=1, keepdims=True))
    for buf in (dx, dw, dh, pa, pb):
        buf.free()


SPLITS = ["64x256", "64x128 K/4", "64x64 K/8", "64x32 K/8"]


def _rows_split(M, rows, cols):
    """The split the dispatch takes, by its rule (rounds of workgroups times
    the weight of one, of which a fixed part does not shrink with K)."""
    f = np.float32
    groups = lambda tiles: (M + 63) // 64 * (((rows + 31) // 32 + tiles - 1) // tiles)
    k = f(min((cols + 63) // 64 / 64, 1.0))
    weight = lambda w, fixed: f(w) if k == 1 else f(fixed) + (f(w) - f(fixed)) * k
    n0 = groups(8)
    last = f(0) if n0 % 512 == 0 else weight(2.0, 0.29) if n0 % 512 <= 256 else weight(4.05, 0.2)
    t = [weight(4.05, 0.2) * f(n0 // 512) + last]
    t += [weight(w, c) * f((groups(n) + 255) // 256) for w, c, n in ((1.1, 0.15, 4), (0.65, 0.1, 2), (0.38, 0.07, 1))]
    return SPLITS[int(np.argmin(t))]


@pytest.mark.parametrize("typ", [GGML_Q4_0, GGML_Q8_0])
@pytest.mark.parametrize("M,rows,cols,split", [
    (1, 1, 32, "64x32 K/8"), (17, 300, 128, "64x32 K/8"), (32, 96, 544, "64x32 K/8"), (33, 33, 1120, "64x32 K/8"),
    (65, 4096, 96, "64x32 K/8"), (96, 2080, 544, "64x32 K/8"), (300, 8160, 4128, "64x32 K/8"),
    (250, 4064, 288, "64x64 K/8"), (256, 4096, 64, "64x64 K/8"), (230, 4001, 4128, "64x64 K/8"),
    (130, 9000, 544, "64x128 K/4"), (200, 6001, 288, "64x128 K/4"), (500, 4064, 288, "64x128 K/4"),
    (512, 4096, 96, "64x128 K/4"), (90, 11233, 1120, "64x128 K/4"), (500, 2049, 1056, "64x128 K/4"),
    (161, 11233, 160, "64x256"), (1025, 8224, 32, "64x256"), (2048, 4097, 96, "64x256"), (129, 21984, 64, "64x256"),
    (600, 11233, 160, "64x256"), (540, 22001, 32, "64x256"), (512, 22016, 96, "64x256"),
    (2048, 4096, 1056, "64x256"), (2048, 4096, 4128, "64x256")])
def test_rows_gemm_splits(P, typ, M, rows, cols, split):
    """Every split of the prompt GEMM (64 x 32 and 64 x 64 with K over 8
    wavefronts, 64 x 128 with K over 4, 64 x 256 with K whole) at ragged rows
    (last row groups of 1, 24 and up to 64 rows), columns and K (one block, odd
    block counts, fewer pairs than K slices), the residual from a buffer of
    its own and in place.  Bound per output: two fp16 parts keep each
    activation to 2^-22 of its row's largest, and the fp32 sums round once per
    16 products and twice per block (the last term: at most 2^-24 of the sum
    of magnitudes each)."""
    assert _rows_split(M, rows, cols) == split
    print(f"rows gemm split {'Q4_0' if typ == GGML_Q4_0 else 'Q8_0'} {M}x{rows}x{cols}", flush=True)
    rng = np.random.default_rng(M + rows + cols + typ)
    W = N.rand_q4_0(rng, rows, cols) if typ == GGML_Q4_0 else N.rand_q8_0(rng, rows, cols)
    X = rng.normal(0, 1, (M, cols)).astype(np.float32)
    R = rng.normal(0, 1, (M, rows)).astype(np.float32)
    Y = _rows_gemm(P, typ, W, X, R)
    assert np.array_equal(Y, _rows_gemm(P, typ, W, X, R, in_place=True))
    w = N.q4_values(W) if typ == GGML_Q4_0 else N.q8_values(W)
    w = np.asarray(w, np.float64).reshape(rows, cols)
    prod, mag = X.astype(np.float64) @ w.T, np.abs(X).astype(np.float64) @ np.abs(w).T
    top = np.abs(X).max(axis=1).astype(np.float64)[:, None] * np.abs(w).sum(axis=1)[None, :]
    bound = 2.0 ** -22 * top + (cols / 8 + 8) * 2.0 ** -24 * mag + 2.0 ** -23 * (np.abs(R) + np.abs(prod))
    assert np.all(np.abs(Y - (R + prod)) <= bound)


def _oracle_prefill(om, prompt, L, n_ctx, kvd, flips, near=None, idx=None):
    """The oracle's prompt forward from an empty cache with the given gate
    decisions inverted: (last-token logits, K rows [L][n][kvd], V rows)."""
    n = len(prompt)
    om.cache_len = 0
    om.m.flip = len(flips)
    for f, (j, l, col) in enumerate(flips):
        om.m.flip_tok[f], om.m.flip_layer[f], om.m.flip_col[f] = j, l, col
    if near is not None:
        om.m.gate_near, om.m.gate_near_idx = near.ctypes.data, idx.ctypes.data
    ref = np.zeros(om.n_vocab, np.float32)
    try:
        assert O.or_forward(om.ptr, prompt, n, ref) == 0
    finally:
        om.m.gate_near, om.m.gate_near_idx = None, None
        om.m.flip = 0
    kc = om.k_cache.reshape(L, n_ctx, kvd)[:, :n].copy()
    vc = om.v_cache.reshape(L, n_ctx, kvd)[:, :n].copy()
    return ref, kc, vc


def test_prefill_at_gate_threshold(P, tmp_path):
    """The large-M prefill at the reference's FFN gate-skip threshold 0.01
    (src/model.c:582-585).  The skip is a step at |silu(g)| = 0.01, so a gate
    within the two sides' rounding distance of it may fall either way.  Prompt
    tokens are explained in order: the first token whose cached K/V rows (or,
    for the last token, logits) differ must match once one or two of its own
    gate decisions at layers below the first differing one -- each within the
    fp32 rounding window 2 sqrt(d) 2^-24 of the threshold -- are inverted in
    the oracle; then the next differing token, up to 3 inversions in all.
    With no inversion needed this is the plain fp32 bar."""
    L, d, h, kv, ff, V, mt, n = 2, 256, 4, 2, 512, 512, GGML_Q4_0, 512
    print(f"prefill {n} tokens at gate threshold 0.01: {L}L d{d} ff{ff}", flush=True)
    rng = np.random.default_rng(4242)
    path = str(tmp_path / "m.gguf")
    raw = llama_gguf(path, rng, L, d, h, kv, ff, V, std=0.05, norm_random=True, emb_type=mt, out_type=mt,
                     matrix_type=mt)
    n_ctx, kvd = 1024, kv * (d // h)
    prompt = rng.integers(0, V, n).astype(np.int32)
    mp = load(P, path, n_ctx, thr=0.01)
    try:
        got = np.zeros(V, np.float32)
        assert P.vx_model_forward(mp, prompt, n, got) == 0, N.product_error()
        kg = np.zeros((L, n, kvd), np.float32)
        vg = np.zeros((L, n, kvd), np.float32)
        for l in range(L):
            assert P.vx_model_read_kv(mp, l, n, kg[l], vg[l]) == 0, N.product_error()
    finally:
        P.vx_model_destroy(mp)
    om = OracleModel(raw, L, d, h, kv, ff, V, n_ctx=n_ctx, gate_thr=0.01)
    tol = 2.0 * np.sqrt(d) * 2.0 ** -24
    near = np.zeros((n, L), np.float32)
    idx = np.zeros((n, L), np.int32)

    def first_bad(ref, kc, vc):
        for j in range(n):
            for l in range(L):
                if not (close(kg[l, j], kc[l, j]) and close(vg[l, j], vc[l, j])):
                    return j, l
        return (None, None) if close(got, ref) else (n - 1, L)

    flips, where = [], []
    ref, kc, vc = _oracle_prefill(om, prompt, L, n_ctx, kvd, flips, near, idx)
    print(f"closest gate to the threshold: {near.min():.2e} (window {tol:.2e})")
    while True:
        j0, lb = first_bad(ref, kc, vc)
        if j0 is None:
            break
        assert len(flips) < 3, ("more gate decisions needed than 3", where, j0, lb)
        # a decision at layer l changes this token's K/V from layer l + 1 on
        cands = [(l, int(idx[j0, l]), float(near[j0, l])) for l in range(min(lb, L)) if near[j0, l] <= tol]
        assert cands, ("token", j0, "differs at layer", lb, "with no gate within the rounding window",
                       float(near[j0, :lb].min()) if lb else None, tol)
        found = None
        for combo in [[c] for c in cands] + [list(p) for p in itertools.combinations(cands, 2)]:
            if len(flips) + len(combo) > 3:
                continue
            trial = flips + [(j0, l, col) for l, col, _ in combo]
            r, k2, v2 = _oracle_prefill(om, prompt, L, n_ctx, kvd, trial, near, idx)
            j1, _ = first_bad(r, k2, v2)
            if j1 is None or j1 > j0:
                found = (trial, combo, r, k2, v2)
                break
        assert found, ("no inverted gate decision of token", j0, "explains the GPU result", cands)
        flips, (ref, kc, vc) = found[0], found[2:]
        where += [(j0, l, col, dist) for l, col, dist in found[1]]
    for j, l, col, dist in where:
        print(f"certified gate at the threshold: token {j}, layer {l}, column {col} (distance {dist:.2e})")
    print(f"last-token logits: max |diff| {np.abs(got.astype(np.float64) - ref).max():.2e} "
          f"after {len(where)} inverted decision(s)")
    assert close(got, ref), max_violation(got, ref)
    for l in range(L):
        assert close(kg[l], kc[l]) and close(vg[l], vc[l]), l


def test_prefill_after_cache_allocated_again(P, tmp_path):
    """The large-M prefill's attention workspace is sized for the cache's
    n_ctx and the attention cap.  A cache dropped (fp16-KV mode on, then off)
    and allocated again for a larger n_ctx, and a cap changed between
    prefills, must each rebuild it: a prompt past the old n_ctx and one under
    a 64-position cap both match the oracle."""
    L, d, h, kv, ff, V = 2, 256, 4, 2, 512, 300
    print("prefill after the cache is allocated again (n_ctx 256 -> 1024) and after a cap change", flush=True)
    rng = np.random.default_rng(77)
    path = str(tmp_path / "m.gguf")
    raw = llama_gguf(path, rng, L, d, h, kv, ff, V, std=0.05, norm_random=True)
    mp = load(P, path, 256)
    try:
        first = rng.integers(0, V, 200).astype(np.int32)
        lg = np.zeros(V, np.float32)
        assert P.vx_model_forward(mp, first, len(first), lg) == 0, N.product_error()
        opt = N.VxModelOptions()
        P.vx_model_get_options(mp, C.byref(opt))
        opt.kv_half = 1
        assert P.vx_model_set_options(mp, C.byref(opt)) == 0, N.product_error()
        assert mp.contents.cache_len == 0
        mp.contents.config.n_ctx = 1024
        opt.kv_half = 0
        assert P.vx_model_set_options(mp, C.byref(opt)) == 0, N.product_error()
        prompt = rng.integers(0, V, 900).astype(np.int32)
        got = np.zeros(V, np.float32)
        assert P.vx_model_forward(mp, prompt, len(prompt), got) == 0, N.product_error()
        opt.attn_cap = 64
        assert P.vx_model_set_options(mp, C.byref(opt)) == 0, N.product_error()
        P.vx_model_kv_truncate(mp, 0)
        got_cap = np.zeros(V, np.float32)
        assert P.vx_model_forward(mp, prompt[:600], 600, got_cap) == 0, N.product_error()
    finally:
        P.vx_model_destroy(mp)
    om = OracleModel(raw, L, d, h, kv, ff, V, n_ctx=1024, gate_thr=0.0)
    ref = np.zeros(V, np.float32)
    assert O.or_forward(om.ptr, prompt, len(prompt), ref) == 0
    assert close(got, ref), max_violation(got, ref)
    om = OracleModel(raw, L, d, h, kv, ff, V, n_ctx=1024, gate_thr=0.0, attn_cap=64)
    assert O.or_forward(om.ptr, prompt[:600], 600, ref) == 0
    assert close(got_cap, ref), max_violation(got_cap, ref)
