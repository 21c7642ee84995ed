"""The prompt prefill's buffers when device memory runs out (CPU).

host/*.c is built against a stand-in for the device layer: every function of
vxh.h does nothing, except that allocations count against a budget and the
prompt attention records its rows.  Checked: which chunks a prompt runs in and
which allocations fail, never a result."""
import ctypes as C
import glob
import os
import re
import subprocess

import numpy as np
import pytest

import _native as N

PRELUDE = """
#include <stdlib.h>
#include <string.h>
#include "vxh.h"
size_t st_budget, st_used;
int st_failed, st_n, st_rows[4096];
"""
# what the stand-in does instead of nothing
BODIES = {
    "vxh_malloc": """size_t *p = st_used + bytes > st_budget ? NULL : (size_t *)malloc(16);
    *dptr = p;
    if (!p) { st_failed++; return VXH_ERR_ALLOC; }
    *p = bytes; st_used += bytes; return 0;""",
    "vxh_free": "if (dptr) { st_used -= *(size_t *)dptr; free(dptr); } return 0;",
    "vxh_workspace_alloc": """memset(w, 0, sizeof *w);
    if (vxh_malloc((void **)&w->part, 4 * part_floats)) return VXH_ERR_ALLOC;
    w->part_floats = part_floats; return 0;""",
    "vxh_workspace_free": "vxh_free(w->part); memset(w, 0, sizeof *w); return 0;",
    "vxh_rows_panel_bytes": "return (size_t)M * K * 4;",
    "vxh_attention_workspace_floats": "return 1000;",
    "vxh_attention_rows_workspace_floats": "return (size_t)M * (cap && cap < n_ctx ? cap : n_ctx);",
    "vxh_attention_rows": "st_rows[st_n++] = M; return 0;",
    "vxh_last_error": 'return "";',
}


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    text = open(os.path.join(N.REPO, "include", "vxh.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    src, bodies = PRELUDE, dict(BODIES)
    for ret, name, args in re.findall(r"^(int|size_t|void|const char \*) ?(vxh_\w+)\(([^;]*)\);", text, flags=re.M):
        src += "%s %s(%s) { %s }\n" % (ret, name, args, bodies.pop(name, "" if ret == "void" else "return 0;"))
    assert not bodies, f"not in vxh.h: {sorted(bodies)}"
    (d / "stub.c").write_text(src)
    so = str(d / "host.so")
    host = sorted(glob.glob(os.path.join(N.REPO, "veltrix-engine_amd", "host", "*.c")))
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-shared", "-fPIC", "-I", os.path.join(N.REPO, "include"), "-o", so,
                    str(d / "stub.c")] + host + ["-lm", "-Wl,-z,defs"], check=True)
    lib = C.CDLL(so)
    lib.vx_model_create_synthetic.argtypes = [C.POINTER(N.VxModelConfig), C.POINTER(N.VxSynthSpec),
                                              C.POINTER(C.POINTER(N.VxModelDev))]
    return lib


class Model:
    """A one-layer model and the memory left for its prefill buffers (per_row
    bytes each)."""

    def __init__(self, L, n_ctx, hd=64, **opt):
        self.L, self.m = L, C.POINTER(N.VxModelDev)()
        self.V, self.d, self.n_ctx = 64, 2 * hd, n_ctx
        self.budget, self.used = C.c_size_t.in_dll(L, "st_budget"), C.c_size_t.in_dll(L, "st_used")
        self.failed, self.n = C.c_int.in_dll(L, "st_failed"), C.c_int.in_dll(L, "st_n")
        self.rows = (C.c_int * 4096).in_dll(L, "st_rows")
        self.budget.value = 1 << 40
        cfg = N.VxModelConfig()
        cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.n_embd = 1, 2, 2, self.d
        cfg.n_ff, cfg.n_vocab, cfg.n_ctx = 256, self.V, n_ctx
        spec = N.VxSynthSpec(seed=1, std=0.02, matrix_type=2, embd_type=2, output_type=2)
        assert L.vx_model_create_synthetic(C.byref(cfg), C.byref(spec), C.byref(self.m)) == 0
        self.options(**opt)
        self.prompt(1)
        self.base = self.used.value

    def options(self, **opt):
        o = N.VxModelOptions()
        self.L.vx_model_get_options(self.m, C.byref(o))
        for k, v in opt.items():
            setattr(o, k, v)
        assert self.L.vx_model_set_options(self.m, C.byref(o)) == 0

    def room(self, rows):
        """Memory for prefill buffers of `rows` rows from now on."""
        self.budget.value = self.base + rows * self.per_row

    def prompt(self, n, want=0):
        """(rows of every prompt chunk, failed allocations) of a prompt of n tokens from an empty cache."""
        self.L.vx_model_kv_truncate(self.m, 0)
        self.n.value = self.failed.value = 0
        logits = np.zeros(self.V, np.float32)
        rc = self.L.vx_model_forward(self.m, np.zeros(n, np.int32).ctypes.data_as(C.c_void_p), n,
                                     logits.ctypes.data_as(C.c_void_p))
        assert (rc == 0) == (want == 0), rc
        if rc == 0:
            assert self.m.contents.cache_len == n
        return self.rows[:self.n.value], self.failed.value

    def close(self):
        self.L.vx_model_destroy(self.m)


@pytest.fixture
def make(L):
    models = []

    def f(n_ctx, **opt):
        probe = Model(L, n_ctx, **opt)
        probe.prompt(1024)
        per_row = (probe.used.value - probe.base) // 1024
        probe.close()
        m = Model(L, n_ctx, **opt)
        m.per_row = per_row
        models.append(m)
        return m
    yield f
    for m in models:
        m.close()


def test_chunks_with_room(make):
    m = make(8000)
    assert m.prompt(60) == ([60], 0)
    assert m.prompt(5000) == ([2048, 2048, 904], 0)
    used = m.used.value
    assert m.prompt(1300) == ([1300], 0) and m.used.value == used


def test_growth_stops_at_what_fits_and_stays_there(make):
    """1100 rows fit: chunks of 1024, and the two sizes that failed are not
    tried again by the following chunks and prompts."""
    m = make(8000)
    m.room(1100)
    assert m.prompt(5000) == ([1024] * 4 + [904], 2)
    assert m.prompt(5000) == ([1024] * 4 + [904], 0)
    assert m.prompt(60) == ([60], 0)


def test_failed_growth_keeps_the_size_that_worked(make):
    m = make(8000)
    m.room(1600)
    assert m.prompt(1500) == ([1500], 0)
    assert m.prompt(4000) == ([1536, 1536, 928], 1)
    assert m.prompt(4000) == ([1536, 1536, 928], 0)


def test_larger_cap_falls_back_to_fewer_rows(make):
    """A cap that makes the workspace outgrow the device: fewer rows, no error,
    also for a short prompt; with the old cap the old size comes back."""
    m = make(4000, attn_cap=256)
    assert m.prompt(2048) == ([2048], 0)
    m.budget.value = m.used.value + 4096
    m.options(attn_cap=0)
    rows, failed = m.prompt(60)
    assert rows == [60] and failed >= 1
    rows, _ = m.prompt(2048)
    assert sum(rows) == 2048 and max(rows) == 512
    assert m.prompt(2048) == (rows, 0)
    m.options(attn_cap=256)
    assert m.prompt(3000) == ([2048, 952], 0)


def test_chunks_cut_below_the_minimum_take_the_batched_forward(make):
    """prefill_min_rows also holds for a chunk that the room or the head size
    cuts short."""
    m = make(8000, prefill_min_rows=1000)
    m.room(600)
    rows, failed = m.prompt(3000)
    assert rows == [] and failed >= 1
    assert m.prompt(3000) == ([], 0)
    m = make(8000, hd=96, prefill_min_rows=600)
    assert m.prompt(3000) == ([], 0)
    m.options(prefill_min_rows=500)
    assert m.prompt(3000) == ([512] * 5, 0)


def test_no_room_at_all_is_an_error_until_there_is(make):
    m = make(8000)
    m.room(100)
    m.prompt(3000, want=1)
    assert m.used.value == m.base
    m.room(2048)
    assert m.prompt(3000) == ([2048, 952], 0)
