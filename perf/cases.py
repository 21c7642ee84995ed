"""The work a user of the engine has it do, as measurable cases.

Three kinds of case call the host API on whole models or decoder blocks
(one-token decode, a verify step, a prompt); the others call the device C ABI
the engine is built from, one layer or block at a time: the skinny GEMM, the
FFN block of a verify step, the prompt GEMM, the attention of a verify step
and of a prompt chunk, the sampling decision.  Sizes are those of the
repository's benchmark configurations (a 7B-shape target, a 22-layer draft,
a 28-layer GQA model with a 152064-entry vocabulary) and odd ones around
them.  Weights, caches and inputs are made on the GPU from the seed.
"""
import ctypes as C
import os

import numpy as np
import torch

vp = C.c_void_p
HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "veltrix-engine_amd", "lib", "libveltrix_amd.so")
DEV = "cuda"


# --------------------------------------------------------------------------
# the library
# --------------------------------------------------------------------------
class Qmat(C.Structure):
    _fields_ = [("type", C.c_int), ("n_rows", C.c_int), ("n_cols", C.c_int), ("n_pairs", C.c_int),
                ("qs", vp), ("d", vp), ("cached", C.c_int), ("tq", vp), ("td", vp)]


class Panel(C.Structure):
    _fields_ = [("data", vp), ("corr", vp), ("rscale", vp), ("xs", vp), ("M", C.c_int), ("K", C.c_int),
                ("avx2", C.c_int), ("rs_ld", C.c_int)]


class Epilogue(C.Structure):
    _fields_ = [("kind", C.c_int), ("y", vp), ("ldy", C.c_int), ("r", vp), ("ldr", C.c_int), ("thr", C.c_float),
                ("scale", C.c_float), ("n_out", C.c_int)]


class Workspace(C.Structure):
    _fields_ = [("acc", vp), ("acc_elems", C.c_size_t), ("part", vp), ("part_floats", C.c_size_t)]


class Pro(C.Structure):
    _fields_ = [("kind", C.c_int), ("x", vp), ("ldx", C.c_int), ("src", vp), ("ld_src", C.c_int), ("w", vp),
                ("x_out", vp), ("ld_xout", C.c_int), ("ss", vp), ("ss_in", vp), ("ss_K", C.c_int),
                ("thr", C.c_float), ("clear", vp), ("n_clear", C.c_size_t), ("part", vp), ("n_chunks", C.c_int),
                ("n_heads", C.c_int), ("n_kv_heads", C.c_int), ("head_dim", C.c_int)]


class VocabWs(C.Structure):
    _fields_ = [("part", vp), ("cnt", vp), ("stats", vp), ("max_rows", C.c_int)]


class ModelConfig(C.Structure):
    _fields_ = ([(n, C.c_int) for n in ("n_layers", "n_heads", "n_kv_heads", "n_embd", "n_head_dim", "n_ff",
                                        "n_vocab", "n_ctx")] +
                [("rope_theta", C.c_float), ("rope_freq_base", C.c_float)] +
                [(n, C.c_int) for n in ("n_threads", "arch", "mlp_type", "norm_type", "rope_partial_dims")] +
                [(n, C.c_bool) for n in ("has_q_bias", "has_k_bias", "has_v_bias", "has_post_attn_norm",
                                         "has_post_ffn_norm", "has_ffn_bias")])


class Model(C.Structure):
    _fields_ = ([("config", ModelConfig), ("tensors", vp), ("n_tensors", C.c_int)] +
                [("p%d" % i, vp) for i in range(25)] + [("k_cache", vp), ("v_cache", vp), ("cache_len", C.c_int)])


class ModelOptions(C.Structure):
    _fields_ = [("q4_kernel", C.c_int), ("attn_cap", C.c_int), ("ffn_gate_threshold", C.c_float),
                ("fused", C.c_int), ("pro_max_rows", C.c_int), ("kv_half", C.c_int), ("prefill_min_rows", C.c_int)]


class SynthSpec(C.Structure):
    _fields_ = [("seed", C.c_uint64), ("std", C.c_float), ("matrix_type", C.c_int), ("embd_type", C.c_int),
                ("output_type", C.c_int)]


_lib = None


def lib():
    global _lib
    if _lib is None:
        torch.zeros(1, device=DEV)
        L = C.CDLL(LIB)
        i, f, z = C.c_int, C.c_float, C.c_size_t
        args = {
            "vxh_qmat_alloc": [vp, i, i, i], "vxh_qmat_free": [vp],
            "vxh_qmat_set_rows": [vp, vp, i, i, i, i, i, vp],
            "vxh_panel_alloc": [vp, i, i], "vxh_panel_free": [vp],
            "vxh_workspace_alloc": [vp, z, z], "vxh_workspace_free": [vp],
            "vxh_prep_panel": [vp, vp, i, i, i, i, vp, i, vp],
            "vxh_gemm": [vp, vp, i, vp, vp, i, vp],
            "vxh_gemm_acc": [vp, vp, i, vp, i, i, f, vp, i, f, i, vp],
            "vxh_gemm_pro": [vp, i, vp, vp, i, i, f, vp, vp, vp],
            "vxh_swiglu_panel_norm": [vp, i, i, i, f, vp, i, vp, z, vp, vp],
            "vxh_acc_store": [vp, i, i, i, vp, i, vp, i, vp],
            "vxh_rows_panel": [vp, i, i, i, vp, vp],
            "vxh_gemm_rows": [vp, vp, i, vp, i, i, vp, i, f, vp],
            "vxh_fill_f32": [vp, f, z, vp], "vxh_copy": [vp, vp, z, vp],
            "vxh_attention": [vp, i, i, i, i, i, i, i, vp, vp, vp, i, vp, vp],
            "vxh_attention_qkv_keep": [vp, i, vp, i] + [vp] * 5 + [i] * 8 + [vp, vp, vp, i, vp, vp],
            "vxh_attention_qkv_f16": [vp, i, vp, i] + [vp] * 5 + [i] * 8 + [vp, vp, vp, i, vp, vp],
            "vxh_vocab_ws_alloc": [vp, i], "vxh_vocab_ws_free": [vp],
            "vxh_sample_keep_mc": [vp, i, f, f, vp, vp, vp, vp, vp, vp],
            "vxh_row_stats_mc": [vp, i, i, i, f, vp, vp, vp],
            "vxh_accept_mc": [vp, i, i, vp, vp, i, i, vp, vp, i, f, vp, vp, vp, vp],
            "vx_model_create_synthetic": [vp, vp, vp], "vx_model_get_options": [vp, vp],
            "vx_model_set_options": [vp, vp], "vx_model_forward": [vp, vp, i, vp],
            "vx_model_verify": [vp, vp, i, vp], "vx_model_kv_truncate": [vp, i], "vx_model_destroy": [vp],
            "vx_model_read_tensor": [vp, C.c_char_p, vp, z],
        }
        for name, a in args.items():
            getattr(L, name).argtypes = a
        for name in ("vxh_rows_panel_bytes", "vxh_gemm_workspace_elems", "vxh_attention_workspace_floats"):
            getattr(L, name).restype = z
        for name in ("vx_model_get_options", "vx_model_kv_truncate", "vx_model_destroy", "vxh_vocab_ws_free"):
            getattr(L, name).restype = None
        L.vxh_last_error.restype = C.c_char_p
        L.vx_last_error.restype = C.c_char_p
        if L.vxh_init() != 0:
            raise RuntimeError(L.vxh_last_error().decode())
        _lib = L
    return _lib


def ok(rc):
    if rc != 0:
        raise RuntimeError("%d: %s / %s" % (rc, _lib.vxh_last_error().decode(), _lib.vx_last_error().decode()))


def ptr(t):
    return vp(t.data_ptr()) if t is not None else None


class Owned:
    """A struct the library fills, given back when the state goes."""

    def __init__(self, struct, free):
        self.s, self.free = struct, free
        self.ref = C.byref(struct)

    def __del__(self):
        self.free(self.ref)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def blocks(g, kind, rows, cols):
    """Weights N(0, 0.02^2) as GGUF blocks: (fp16 scales, whole numbers, the
    block bytes as a uint8 tensor)."""
    nb = cols // 32
    d = (0.0075 if kind == "q4_0" else 0.00055) * (1 + 0.2 * torch.rand(rows, nb, generator=g, device=DEV))
    d = d.to(torch.float16)
    z = torch.randn(rows, nb, 32, generator=g, device=DEV) * 0.02 / d[..., None].float()
    if kind == "q4_0":
        q = torch.clamp(torch.round(z), -8, 7).to(torch.int16)
        s = (q + 8).to(torch.uint8)
        body = s[..., 0::2] | (s[..., 1::2] << 4)
    else:
        q = torch.clamp(torch.round(z), -127, 127).to(torch.int16)
        body = q.to(torch.int8).view(torch.uint8)
    raw = torch.cat([d.view(torch.uint8).reshape(rows, nb, 2), body], dim=2).contiguous()
    return d, q, raw


def dense64(d, q):
    return (q.double() * d.double()[..., None]).reshape(d.shape[0], -1)


TYPES = {"q4_0": 2, "q8_0": 8}
BLOCK_BYTES = {"q4_0": 18, "q8_0": 34}


def matrix(kind, rows, cols, parts):
    """A device matrix of the raw block tensors `parts`: [(raw, group, stride, offset)]."""
    L = lib()
    m = Owned(Qmat(), L.vxh_qmat_free)
    ok(L.vxh_qmat_alloc(m.ref, TYPES[kind], rows, cols))
    for raw, group, stride, off in parts:
        ok(L.vxh_qmat_set_rows(m.ref, ptr(raw), 1, raw.shape[0], group or raw.shape[0], stride, off, None))
    torch.cuda.synchronize()
    return m


def wbytes(kind, rows, cols):
    return rows * (cols // 32) * BLOCK_BYTES[kind]


def rope_tables(n_pos, hd, theta):
    """cos and sin of float32 angles pos / theta^(2i/hd), as the reference forms them."""
    powf = C.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = C.c_float, [C.c_float, C.c_float]
    f = np.array([np.float32(1.0) / np.float32(powf(theta, np.float32(2 * i) / np.float32(hd)))
                  for i in range(hd // 2)], np.float32)
    ang = np.arange(n_pos, dtype=np.float32)[:, None] * f[None, :]
    return ang


def rotate64(x, ang):
    """RoPE on adjacent pairs of x[rows][heads][hd] at angles ang[rows][hd/2] (fp64)."""
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], dim=-1).reshape(x.shape)


def attend64(q, k, v, n_past, cap):
    """Causal attention of q[M][H][hd] over k, v[ctx][KV][hd] in fp64, one kv head at a time."""
    M, H, hd = q.shape
    KV = k.shape[1]
    G = H // KV
    out = torch.empty_like(q)
    n = torch.arange(M, device=DEV) + n_past + 1
    if cap:
        n = torch.clamp(n, max=cap)
    mask = torch.arange(k.shape[0], device=DEV)[None, :] >= n[:, None]
    for g in range(KV):
        qs = q[:, g * G:(g + 1) * G].transpose(0, 1).reshape(G * M, hd)
        s = (qs @ k[:, g].T.contiguous()) / hd ** 0.5
        s = s.view(G, M, -1).masked_fill(mask, float("-inf"))
        p = torch.exp(s - s.amax(dim=2, keepdim=True))
        p = p / (p.sum(dim=2, keepdim=True) + 1e-10)
        out[:, g * G:(g + 1) * G] = (p.view(G * M, -1) @ v[:, g].contiguous()).view(G, M, hd).transpose(0, 1)
    return out


# --------------------------------------------------------------------------
# whole models and decoder blocks: decode (one token), verify (k + 1 tokens,
# every row's logits), prompt (n tokens, the last row's logits)
# --------------------------------------------------------------------------
class ModelHandle:
    """A model; it goes when its state and every view of its cache have gone."""

    def __init__(self, cfg, spec):
        L = lib()
        self.m, self.destroy = vp(), L.vx_model_destroy
        ok(L.vx_model_create_synthetic(C.byref(cfg), C.byref(spec), C.byref(self.m)))

    def __del__(self):
        if self.m:
            self.destroy(self.m)


class DeviceArray:
    """The model's cache, whose device address the model struct holds, as an
    array (the tensors made of it keep it, and so the model)."""

    def __init__(self, handle, address, shape, half):
        self.handle = handle
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f2" if half else "<f4", "data": (address, False),
                                         "version": 2}


class ModelState:
    def __init__(self, case, seed):
        L = lib()
        c = case
        past, rows = c["past"], c["rows"]
        cfg = ModelConfig(n_layers=c["layers"], n_heads=c["heads"], n_kv_heads=c["kv_heads"], n_embd=c["d"],
                          n_ff=c["ff"], n_vocab=c["vocab"], n_ctx=past + rows + 16, rope_theta=10000.0)
        spec = SynthSpec(seed=seed, std=0.02, matrix_type=TYPES[c["weights"]], embd_type=TYPES[c["weights"]],
                         output_type=TYPES[c["output"]])
        handle = ModelHandle(cfg, spec)
        self.handle, self.m = handle, handle.m
        opt = ModelOptions()
        L.vx_model_get_options(self.m, C.byref(opt))
        opt.ffn_gate_threshold = 0.0        # the skip of small gates is a step: no rounding bound holds across it
        opt.kv_half = 1 if c["kv16"] else 0
        ok(L.vx_model_set_options(self.m, C.byref(opt)))
        rng = np.random.default_rng(seed)
        self.tokens = rng.integers(0, c["vocab"], rows).astype(np.int32)
        self.logits = np.zeros((rows if c["op"] == "verify" else 1, c["vocab"]), np.float32)
        self.past = past
        self.call = L.vx_model_verify if c["op"] == "verify" else L.vx_model_forward
        self.truncate = L.vx_model_kv_truncate
        self.args = (self.m, vp(self.tokens.ctypes.data), rows, vp(self.logits.ctypes.data))
        # the first forward allocates the cache; then the past rows of a
        # conversation in progress are put into it
        ok(L.vx_model_forward(self.m, vp(self.tokens.ctypes.data), 1, vp(self.logits.ctypes.data)))
        mod = C.cast(self.m, C.POINTER(Model)).contents
        mod.cache_len = past
        kvd = c["kv_heads"] * (c["d"] // c["heads"])
        caches = [torch.as_tensor(DeviceArray(handle, base, (c["layers"], cfg.n_ctx, kvd), c["kv16"]), device=DEV)
                  for base in (mod.k_cache, mod.v_cache)]
        if past:
            for l in range(c["layers"]):
                for cache, t in zip(caches, past_rows(seed, l, past, kvd, bool(c["kv16"]))):
                    cache[l, :past] = t
            torch.cuda.synchronize()
        # the cache rows a pass writes
        self.k_new, self.v_new = (cache[:, past:past + rows] for cache in caches)


def past_rows(seed, layer, past, kvd, half):
    g = gen(seed * 1000 + layer)
    k, v = normal(g, past, kvd), normal(g, past, kvd)
    return (k.half(), v.half()) if half else (k, v)


def run_model(s):
    s.truncate(s.m, s.past)
    ok(s.call(*s.args))
    return [s.logits.copy(), s.k_new, s.v_new]


def exact_model(case, seed):
    c = case
    s = ModelState(case, seed)
    L = lib()
    hd, kvd = c["d"] // c["heads"], c["kv_heads"] * (c["d"] // c["heads"])

    def read(name, rows, cols, kind):
        nb = cols // 32
        raw = np.empty((rows, nb, BLOCK_BYTES[kind]), np.uint8)
        ok(L.vx_model_read_tensor(s.m, name.encode(), vp(raw.ctypes.data), raw.nbytes))
        t = torch.from_numpy(raw).to(DEV)
        d = t[..., :2].contiguous().view(torch.float16)[..., 0]
        b = t[..., 2:]
        if kind == "q4_0":
            q = torch.stack([b & 15, b >> 4], dim=-1).reshape(rows, nb, 32).to(torch.int16) - 8
        else:
            q = b.contiguous().view(torch.int8)
        return dense64(d, q)

    def norm(x):
        return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-5)

    W = c["weights"]
    ids = torch.from_numpy(s.tokens).long().to(DEV)
    x = read("token_embd.weight", c["vocab"], c["d"], W)[ids]
    M, past = c["rows"], c["past"]
    ang = torch.from_numpy(rope_tables(past + M, hd, 10000.0)[past:]).to(DEV).double()
    ks, vs = [], []
    for l in range(c["layers"]):
        p = "blk.%d." % l
        h = norm(x)
        q = (h @ read(p + "attn_q.weight", c["d"], c["d"], W).T).view(M, c["heads"], hd)
        k = (h @ read(p + "attn_k.weight", kvd, c["d"], W).T).view(M, c["kv_heads"], hd)
        v = (h @ read(p + "attn_v.weight", kvd, c["d"], W).T).view(M, c["kv_heads"], hd)
        q, k = rotate64(q, ang), rotate64(k, ang)
        if c["kv16"]:
            k, v = k.half().double(), v.half().double()
        ks.append(k.reshape(M, kvd))
        vs.append(v.reshape(M, kvd))
        if past:
            pk, pv = past_rows(seed, l, past, kvd, bool(c["kv16"]))
            k = torch.cat([pk.double().view(past, -1, hd), k])
            v = torch.cat([pv.double().view(past, -1, hd), v])
        a = attend64(q, k, v, past, 4096).reshape(M, c["d"])
        x = x + a @ read(p + "attn_output.weight", c["d"], c["d"], W).T
        h = norm(x)
        gate = h @ read(p + "ffn_gate.weight", c["ff"], c["d"], W).T
        up = h @ read(p + "ffn_up.weight", c["ff"], c["d"], W).T
        x = x + (gate / (1 + torch.exp(-gate)) * up) @ read(p + "ffn_down.weight", c["d"], c["ff"], W).T
    if c["op"] != "verify":
        x = x[-1:]
    logits = norm(x) @ read("output.weight", c["vocab"], c["d"], c["output"]).T
    return [logits.cpu().numpy(), torch.stack(ks), torch.stack(vs)]


def work_model(c):
    hd = c["d"] // c["heads"]
    kvd, M, past = c["kv_heads"] * hd, c["rows"], c["past"]
    n = c["d"] * (2 * c["d"] + 2 * kvd + 3 * c["ff"])
    ctx = min(past + M, 4096)
    pairs = sum(min(past + m + 1, 4096) for m in range(M))
    outs = M if c["op"] == "verify" else 1
    kv = 2 * kvd * (2 if c["kv16"] else 4)
    b = c["layers"] * (wbytes(c["weights"], n // c["d"], c["d"]) + kv * (ctx + M))
    b += wbytes(c["output"], c["vocab"], c["d"]) + M * wbytes(c["weights"], 1, c["d"]) + 4 * outs * c["vocab"]
    f = c["layers"] * (2 * M * n + 4 * pairs * c["d"]) + 2 * outs * c["vocab"] * c["d"]
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------------------
# gemm: M rows through one quantised matrix (panel, GEMM, store or residual)
# --------------------------------------------------------------------------
class GemmState:
    pass


def gemm_inputs(case, seed):
    g = gen(seed)
    w = blocks(g, case["weights"], case["n"], case["k"])
    x = normal(g, case["rows"], case["k"])
    r = normal(g, case["rows"], case["n"]) if case["resid"] else None
    return w, x, r


def prepare_gemm(case, seed):
    L = lib()
    (d, q, raw), x, r = gemm_inputs(case, seed)
    s = GemmState()
    M, N, K = case["rows"], case["n"], case["k"]
    s.x, s.r, s.y = x, r, torch.zeros(M, N, device=DEV)
    s.w = matrix(case["weights"], N, K, [(raw, 0, 0, 0)])
    s.panel = Owned(Panel(), L.vxh_panel_free)
    ok(L.vxh_panel_alloc(s.panel.ref, M, K))
    s.ws = Owned(Workspace(), L.vxh_workspace_free)
    ok(L.vxh_workspace_alloc(s.ws.ref, L.vxh_gemm_workspace_elems(s.w.s.n_rows, M), 4))
    s.ep = Epilogue(kind=1 if case["resid"] else 0, y=ptr(s.y), ldy=N, r=ptr(r), ldr=N, scale=1.0, n_out=N)
    s.prep = (s.panel.ref, ptr(x), K, M, K, 0, None, 0, None)
    s.gemm = (s.w.ref, s.panel.ref, M, C.byref(s.ep), s.ws.ref, 0, None)
    return s


def run_gemm(s):
    ok(_lib.vxh_prep_panel(*s.prep))
    ok(_lib.vxh_gemm(*s.gemm))
    return s.y


def exact_gemm(case, seed):
    (d, q, _), x, r = gemm_inputs(case, seed)
    y = x.double() @ dense64(d, q).T
    return y + r.double() if r is not None else y


def work_gemm(c):
    M, N, K = c["rows"], c["n"], c["k"]
    return {"bytes": wbytes(c["weights"], N, K) + 4 * M * (K + N * (2 if c["resid"] else 1)),
            "flops": 2 * M * N * K}


# --------------------------------------------------------------------------
# ffn: the FFN block of a verify batch (pending residual, RMSNorm, gate/up,
# SwiGLU, down, residual)
# --------------------------------------------------------------------------
def ffn_inputs(case, seed):
    g = gen(seed)
    M, d, F = case["rows"], case["d"], case["ff"]
    wg, wu, wd = (blocks(g, case["weights"], n, k) for n, k in ((F, d), (F, d), (d, F)))
    x, pend = normal(g, M, d), normal(g, M, d).double()
    w = 1 + 0.1 * normal(g, d)
    return wg, wu, wd, x, pend, w


def prepare_ffn(case, seed):
    L = lib()
    wg, wu, wd, x, pend, w = ffn_inputs(case, seed)
    s = GemmState()
    M, d, F = case["rows"], case["d"], case["ff"]
    gu = (F + 15) // 16 * 32
    s.wgu = matrix(case["weights"], gu, d, [(wg[2], 16, 32, 0), (wu[2], 16, 32, 16)])
    s.wd = matrix(case["weights"], d, F, [(wd[2], 0, 0, 0)])
    s.x, s.pend, s.w = x, pend, w
    s.t = torch.zeros(M, d, device=DEV)
    s.y = torch.zeros(M, d, device=DEV)
    s.acc_gu = torch.zeros(M, gu, device=DEV, dtype=torch.float64)
    s.acc_x = torch.zeros(M, d, device=DEV, dtype=torch.float64)
    s.ss = torch.zeros(16, device=DEV, dtype=torch.float64)
    s.panel = Owned(Panel(), L.vxh_panel_free)
    ok(L.vxh_panel_alloc(s.panel.ref, M, F))
    s.pro = Pro(kind=2, x=ptr(x), ldx=d, src=ptr(pend), ld_src=d, w=ptr(w), x_out=ptr(s.t), ld_xout=d, ss=ptr(s.ss))
    s.a0 = (ptr(s.ss), 0.0, 32, None)
    s.a1 = (s.wgu.ref, M, C.byref(s.pro), ptr(s.acc_gu), gu, gu, 1.0, None, None, None)
    s.a2 = (ptr(s.acc_gu), gu, M, F, 0.0, ptr(s.ss), d, None, 0, s.panel.ref, None)
    s.a3 = (s.wd.ref, s.panel.ref, M, ptr(s.acc_x), d, d, 1.0, None, 0, 0.0, 0, None)
    s.a4 = (ptr(s.acc_x), d, M, d, ptr(s.y), d, ptr(s.t), d, None)
    return s


def run_ffn(s):
    ok(_lib.vxh_fill_f32(*s.a0))
    ok(_lib.vxh_gemm_pro(*s.a1))
    ok(_lib.vxh_swiglu_panel_norm(*s.a2))
    ok(_lib.vxh_gemm_acc(*s.a3))
    ok(_lib.vxh_acc_store(*s.a4))
    return [s.t, s.y]


def exact_ffn(case, seed):
    wg, wu, wd, x, pend, w = ffn_inputs(case, seed)
    t = x.double() + pend
    h = w.double() * t / torch.sqrt((t * t).mean(dim=1, keepdim=True) + 1e-5)
    g, u = h @ dense64(*wg[:2]).T, h @ dense64(*wu[:2]).T
    return [t, t + (g / (1 + torch.exp(-g)) * u) @ dense64(*wd[:2]).T]


def work_ffn(c):
    M, d, F = c["rows"], c["d"], c["ff"]
    return {"bytes": wbytes(c["weights"], 3 * F, d) + M * d * (4 + 8 + 4 + 4) + 4 * d, "flops": 6 * M * d * F}


# --------------------------------------------------------------------------
# rows: a prompt chunk through one quantised matrix (large M)
# --------------------------------------------------------------------------
def prepare_rows(case, seed):
    L = lib()
    (d, q, raw), x, r = gemm_inputs(case, seed)
    s = GemmState()
    M, N, K = case["rows"], case["n"], case["k"]
    s.x, s.r, s.y = x, r, torch.zeros(M, N, device=DEV)
    s.w = matrix(case["weights"], N, K, [(raw, 0, 0, 0)])
    s.px = torch.zeros(L.vxh_rows_panel_bytes(M, K), device=DEV, dtype=torch.uint8)
    s.a0 = (ptr(x), K, M, K, ptr(s.px), None)
    s.a1 = (s.w.ref, ptr(s.px), M, ptr(s.y), N, N, ptr(r), N, 1.0, None)
    return s


def run_rows(s):
    ok(_lib.vxh_rows_panel(*s.a0))
    ok(_lib.vxh_gemm_rows(*s.a1))
    return s.y


# --------------------------------------------------------------------------
# attn: the attention of a decode or verify batch from its q|k|v sums (RoPE
# and the new cache rows included)
# --------------------------------------------------------------------------
def attn_inputs(case, seed):
    g = gen(seed)
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    qkv = normal(g, M, (H + 2 * KV) * hd).double()
    kc, vc = normal(g, past + M, KV * hd), normal(g, past + M, KV * hd)
    if case["kv16"]:
        kc, vc = kc.half(), vc.half()
    ang = rope_tables(past + M + 1, hd, 10000.0)
    return qkv, kc, vc, torch.from_numpy(ang).to(DEV)


def prepare_attn(case, seed):
    L = lib()
    s = GemmState()
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    s.src, s.kc, s.vc, ang = attn_inputs(case, seed)
    s.cos, s.sin = torch.cos(ang.double()).float(), torch.sin(ang.double()).float()
    s.qkv = s.src.clone()
    s.out = torch.zeros(M, H * hd, device=DEV)
    n_ctx, cap = past + M, case["cap"]
    s.ws = Owned(Workspace(), L.vxh_workspace_free)
    ok(L.vxh_workspace_alloc(s.ws.ref, 32, L.vxh_attention_workspace_floats(M, n_ctx, cap, H, KV, hd)))
    s.kv16 = case["kv16"]
    s.past, s.n_new = past, M
    s.args = (ptr(s.qkv), (H + 2 * KV) * hd, None, 0, None, None, None, ptr(s.cos), ptr(s.sin), past + M + 1, M,
              past, n_ctx, H, KV, hd, cap, ptr(s.kc), ptr(s.vc), ptr(s.out), H * hd, s.ws.ref, None)
    return s


def run_attn(s):
    if s.kv16:
        s.qkv.copy_(s.src)              # the fp16 entry point consumes its sums
        ok(_lib.vxh_attention_qkv_f16(*s.args))
    else:
        ok(_lib.vxh_attention_qkv_keep(*s.args))
    return [s.out, s.kc[s.past:], s.vc[s.past:]]


def exact_attn(case, seed):
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    qkv, kc, vc, ang = attn_inputs(case, seed)
    # the tables a caller hands over are float32
    c, s = torch.cos(ang.double()).float().double()[past:past + M], torch.sin(ang.double()).float().double()[past:past + M]
    x = qkv.view(M, H + 2 * KV, hd)
    a, b = x[..., 0::2], x[..., 1::2]
    rot = torch.stack([a * c[:, None] - b * s[:, None], a * s[:, None] + b * c[:, None]], dim=-1).reshape(x.shape)
    q, k, v = rot[:, :H], rot[:, H:H + KV], x[:, H + KV:]
    if case["kv16"]:
        k, v = k.half().double(), v.half().double()
    kk = torch.cat([kc[:past].double().view(past, KV, hd), k])
    vv = torch.cat([vc[:past].double().view(past, KV, hd), v])
    return [attend64(q.contiguous(), kk, vv, past, case["cap"]).reshape(M, -1), k.reshape(M, -1), v.reshape(M, -1)]


def work_attn(c):
    M, H, KV, hd, past = c["rows"], c["heads"], c["kv_heads"], c["hd"], c["past"]
    cap = c["cap"] or 1 << 30
    e = 2 if c["kv16"] else 4
    return {"bytes": 2 * e * KV * hd * (min(past + M, cap) + M) + M * hd * (8 * (H + 2 * KV) + 4 * H),
            "flops": 4 * H * hd * sum(min(past + m + 1, cap) for m in range(M))}


# --------------------------------------------------------------------------
# prompt attention: M rotated q rows over a cache that holds their keys
# --------------------------------------------------------------------------
def pattn_inputs(case, seed):
    g = gen(seed)
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    return normal(g, M, H * hd), normal(g, past + M, KV * hd), normal(g, past + M, KV * hd)


def prepare_pattn(case, seed):
    L = lib()
    s = GemmState()
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    s.q, s.kc, s.vc = pattn_inputs(case, seed)
    s.out = torch.zeros(M, H * hd, device=DEV)
    s.ws = Owned(Workspace(), L.vxh_workspace_free)
    ok(L.vxh_workspace_alloc(s.ws.ref, 32, L.vxh_attention_workspace_floats(M, past + M, case["cap"], H, KV, hd)))
    s.args = (ptr(s.q), M, past, past + M, H, KV, hd, case["cap"], ptr(s.kc), ptr(s.vc), ptr(s.out), H * hd, s.ws.ref,
              None)
    return s


def run_pattn(s):
    ok(_lib.vxh_attention(*s.args))
    return s.out


def exact_pattn(case, seed):
    M, H, KV, hd, past = case["rows"], case["heads"], case["kv_heads"], case["hd"], case["past"]
    q, kc, vc = pattn_inputs(case, seed)
    return attend64(q.double().view(M, H, hd), kc.double().view(-1, KV, hd), vc.double().view(-1, KV, hd), past,
                    case["cap"]).reshape(M, -1)


def work_pattn(c):
    M, H, KV, hd, past = c["rows"], c["heads"], c["kv_heads"], c["hd"], c["past"]
    cap = c["cap"] or 1 << 30
    return {"bytes": 8 * KV * hd * min(past + M, cap) + 8 * M * H * hd,
            "flops": 4 * H * hd * sum(min(past + m + 1, cap) for m in range(M))}


# --------------------------------------------------------------------------
# decide: a draft token drawn from its logits row, and the verify decision
# over k drafts (row statistics, acceptance, resample)
# --------------------------------------------------------------------------
def prepare_decide(case, seed):
    L = lib()
    g = gen(seed)
    V, k, T, top_p = case["vocab"], case["drafts"], case["temp"], case["top_p"]
    s = GemmState()
    s.l = 2.5 * normal(g, k + 1, V)
    s.d = s.l[:k] + 0.3 * normal(g, k, V)
    s.u = torch.rand(2 * k + 1, generator=g, device=DEV)
    s.drafts = torch.zeros(k, device=DEV, dtype=torch.int32)
    s.nuc = torch.zeros(k, 8, device=DEV)
    s.keep = torch.zeros(V, device=DEV)
    s.stats = torch.zeros(k + 1, 3, device=DEV)
    s.out = torch.zeros(k + 3, device=DEV, dtype=torch.int32)
    s.tok, s.desc = torch.zeros(1, device=DEV, dtype=torch.int32), torch.zeros(8, device=DEV)
    s.ws = Owned(VocabWs(), L.vxh_vocab_ws_free)
    ok(L.vxh_vocab_ws_alloc(s.ws.ref, 16))
    for i in range(k):
        ok(L.vxh_sample_keep_mc(ptr(s.d[i]), V, T, top_p, ptr(s.u[k + 1 + i:]), ptr(s.drafts[i:]), ptr(s.nuc[i]),
                                None, s.ws.ref, None))
    torch.cuda.synchronize()
    s.a0 = (ptr(s.d), V, T, top_p, ptr(s.u[k + 1:]), ptr(s.tok), ptr(s.desc), ptr(s.keep), s.ws.ref, None)
    s.a1 = (ptr(s.l), V, k + 1, V, T, ptr(s.stats), s.ws.ref, None)
    s.a2 = (ptr(s.l), V, V, ptr(s.stats), ptr(s.d), V, V, ptr(s.nuc), ptr(s.drafts), k, T, ptr(s.u), ptr(s.out),
            s.ws.ref, None)
    return s


def run_decide(s):
    ok(_lib.vxh_sample_keep_mc(*s.a0))
    ok(_lib.vxh_row_stats_mc(*s.a1))
    ok(_lib.vxh_accept_mc(*s.a2))
    return [s.tok, s.keep, s.stats[:, :2], s.out]


def exact_decide(case, seed):
    g = gen(seed)
    V, k = case["vocab"], case["drafts"]
    l = 2.5 * normal(g, k + 1, V)
    d = l[:k] + 0.3 * normal(g, k, V)
    m = l.double().amax(dim=1)
    z = torch.exp((l.double() - m[:, None]) / case["temp"]).sum(dim=1)
    return [None, d[0].double(), torch.stack([m, z], dim=1), None]


def work_decide(c):
    V, k = c["vocab"], c["drafts"]
    return {"bytes": 4 * V * (1 + 1 + (k + 1) + k), "flops": 10 * V * (2 * k + 2)}


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
OPS = {
    "decode": (ModelState, run_model, exact_model, work_model),
    "verify": (ModelState, run_model, exact_model, work_model),
    "prompt": (ModelState, run_model, exact_model, work_model),
    "gemm": (prepare_gemm, run_gemm, exact_gemm, work_gemm),
    "ffn": (prepare_ffn, run_ffn, exact_ffn, work_ffn),
    "rows": (prepare_rows, run_rows, exact_gemm, work_gemm),
    "attn": (prepare_attn, run_attn, exact_attn, work_attn),
    "pattn": (prepare_pattn, run_pattn, exact_pattn, work_pattn),
    "decide": (prepare_decide, run_decide, exact_decide, work_decide),
}

DRAFT = {"layers": 22, "d": 2048, "heads": 32, "kv_heads": 4, "ff": 5632, "vocab": 32000}
TARGET = {"layers": 32, "d": 4096, "heads": 32, "kv_heads": 32, "ff": 11008, "vocab": 32000}


def listed():
    q4 = {"weights": "q4_0", "output": "q4_0", "kv16": False}
    return [
        # one token of the 22-layer draft at a 2K context: eight of these make
        # most of a speculative round
        dict(DRAFT, name="decode_draft", op="decode", rows=1, past=2047, **q4),
        # the target's verify step of k = 8 drafts at a 2K context
        dict(TARGET, name="verify_target", op="verify", rows=9, past=2048, **q4),
        # a 2048-token prompt through two decoder blocks of the target and its head
        dict(TARGET, name="prompt_blocks", op="prompt", layers=2, rows=2048, past=0, **q4),
        # the smallest matrix of a draft layer, one row: launches and latency
        {"name": "gemm_one_row", "op": "gemm", "weights": "q4_0", "n": 2048, "k": 2048, "rows": 1, "resid": False},
        # the target's FFN matrix at a verify batch of nine rows
        {"name": "gemm_verify", "op": "gemm", "weights": "q4_0", "n": 11008, "k": 4096, "rows": 9, "resid": False},
        # a Q8_0 long-K matrix at five rows with the residual add
        {"name": "gemm_q8_long", "op": "gemm", "weights": "q8_0", "n": 4096, "k": 11008, "rows": 5, "resid": True},
        # the FFN block of a 28-layer GQA model's verify batch
        {"name": "ffn_verify", "op": "ffn", "weights": "q4_0", "d": 3584, "ff": 18944, "rows": 9},
        # a full prompt chunk through gate/up of the target
        {"name": "rows_chunk", "op": "rows", "weights": "q4_0", "n": 22016, "k": 4096, "rows": 512, "resid": False},
        # a short, ragged prompt through a Q8_0 down projection with the residual
        {"name": "rows_ragged_q8", "op": "rows", "weights": "q8_0", "n": 4096, "k": 11008, "rows": 77, "resid": True},
        # the attention of a verify batch over an 8K context of the GQA model
        {"name": "attn_gqa_8k", "op": "attn", "heads": 28, "kv_heads": 4, "hd": 128, "rows": 9, "past": 8183, "cap": 0,
         "kv16": False},
        # the last chunk of a 2K prompt through the draft's attention
        {"name": "attn_prompt", "op": "pattn", "heads": 32, "kv_heads": 4, "hd": 64, "rows": 500, "past": 1536,
         "cap": 4096},
        # drawing a draft token and the decision over eight drafts, large vocabulary
        {"name": "decide_large_vocab", "op": "decide", "vocab": 152064, "drafts": 8, "temp": 1.0, "top_p": 1.0},
    ]


def spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    op = rng.choice(["decode", "verify", "prompt", "gemm", "gemm", "ffn", "rows", "rows", "attn", "attn", "pattn",
                     "pattn", "decide"])
    weights = rng.choice(["q4_0", "q4_0", "q8_0"])
    if op in ("decode", "verify", "prompt"):
        hd = rng.choice([64, 128])
        kv = rng.choice([1, 2, 4, 8])
        heads = kv * rng.choice([1, 2, 3, 4, 7])
        while heads * hd > 4096:
            heads -= kv
        rows = {"decode": 1, "verify": rng.randint(2, 16), "prompt": spread(rng, 48, 1100)}[op]
        return {"op": op, "layers": rng.randint(1, 4), "d": heads * hd, "heads": heads, "kv_heads": kv,
                "ff": 32 * spread(rng, 8, 344), "vocab": spread(rng, 300, 32000), "rows": rows,
                "past": 0 if op == "prompt" and rng.random() < 0.5 else spread(rng, 1, 3000), "weights": weights,
                "output": rng.choice(["q4_0", "q8_0"]), "kv16": op != "prompt" and rng.random() < 0.3}
    if op == "gemm":
        return {"op": op, "weights": weights, "n": spread(rng, 96, 32000), "k": 32 * spread(rng, 4, 344),
                "rows": rng.randint(1, 16), "resid": rng.random() < 0.4}
    if op == "ffn":
        return {"op": op, "weights": weights, "d": 32 * spread(rng, 8, 128), "ff": 32 * spread(rng, 16, 592),
                "rows": rng.randint(3, 16)}
    if op == "rows":
        return {"op": op, "weights": weights, "n": spread(rng, 96, 22016), "k": 32 * spread(rng, 4, 344),
                "rows": spread(rng, 17, 512), "resid": rng.random() < 0.5}
    if op in ("attn", "pattn"):
        kv = rng.choice([1, 2, 4, 8, 32])
        c = {"op": op, "heads": kv * rng.choice([1, 2, 4, 7] if kv < 32 else [1]), "kv_heads": kv,
             "hd": rng.choice([64, 128]), "rows": rng.randint(1, 16) if op == "attn" else spread(rng, 17, 512),
             "past": spread(rng, 1, 8000 if op == "attn" else 3000), "cap": rng.choice([0, 4096])}
        if op == "attn":
            c["kv16"] = rng.random() < 0.4
        return c
    return {"op": op, "vocab": spread(rng, 1000, 152064), "drafts": rng.randint(1, 15),
            "temp": rng.choice([0.5, 0.8, 1.0]), "top_p": rng.choice([0.9, 1.0])}


class State:
    def __init__(self, run_one, inner):
        self.run_one, self.inner = run_one, inner


def prepare(case, seed):
    make, run_one, _, _ = OPS[case["op"]]
    return State(run_one, make(case, seed))


def run(state):
    return state.run_one(state.inner)


def exact(case, seed):
    lib()
    return OPS[case["op"]][2](case, seed)


def work(case):
    return OPS[case["op"]][3](case)


def tolerance(case):
    # activations enter the matrix products as two fp16 parts (22 bits), the
    # sums are fp32: about four times the error measured against 64 bits
    op = case["op"]
    if op in ("decode", "verify", "prompt"):
        # roundings travel through the layers (1.5e-6 to 5e-6 seen); in an
        # fp16 cache a new row may round to the neighbouring half
        return {"rel": 1e-3 if case["kv16"] else 3e-5}
    if op == "attn":
        return {"rel": 5e-4 if case["kv16"] else 2e-6}
    return {"rel": {"gemm": 1e-6, "ffn": 2e-6, "rows": 5e-6, "pattn": 2e-6, "decide": 1e-6}[op]}
