"""Device blocks kept between handles: rebuilding layouts in turn, from several
threads and contexts, gives the same layouts as a first build, and the memory
goes back with the last context."""
from __future__ import annotations

import subprocess
import sys
import threading
from pathlib import Path

import numpy as np
import pytest

from smaxkernels_amd import capi, matgen

pytestmark = pytest.mark.gpu
FIELDS = ("chunk_ptr", "chunk_lengths", "col", "val", "perm", "src_index")


def layout(ctx, d, A, sigma):
    s = ctx.scs_from_crs(A.n_rows, A.n_cols, A.nnz, *d, 8, 64, sigma)
    a = s.arrays(np.float64)
    s.destroy()
    return a


def test_rebuilt_layouts_in_reused_blocks(ctx):
    """Two matrices of different sizes and two window lengths, rebuilt in turn:
    every rebuild lands in blocks that held another layout."""
    mats = [matgen.lomax_band(60_000), matgen.lomax_band(90_000, seed=5)]
    dev = [[ctx.upload(a) for a in (A.row_ptr, A.col, A.val)] for A in mats]
    first = {}
    for _ in range(3):
        for i, A in enumerate(mats):
            for sigma in (4096, 65536):
                got = layout(ctx, dev[i], A, sigma)
                want = first.setdefault((i, sigma), got)
                for f in FIELDS:
                    assert np.array_equal(got[f], want[f]), (i, sigma, f)
    for ds in dev:
        for d in ds:
            d.free()


def test_threads_with_contexts_of_their_own():
    A = matgen.lomax_band(60_000)
    want, errors = [], []

    def work(n):
        try:
            with capi.Context(0) as c:
                d = [c.upload(a) for a in (A.row_ptr, A.col, A.val)]
                for _ in range(n):
                    got = layout(c, d, A, 4096)
                    want.append(got)
                    assert all(np.array_equal(got[f], want[0][f]) for f in FIELDS)
        except Exception as e:  # reported in the test's thread
            errors.append(e)

    work(1)
    threads = [threading.Thread(target=work, args=(4,)) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_handle_destroyed_after_its_context():
    """A handle may be destroyed without a context (null): its blocks are freed."""
    A = matgen.lomax_band(60_000)
    c = capi.Context(0)
    s = c.scs_from_crs(A.n_rows, A.n_cols, A.nnz, c.upload(A.row_ptr), c.upload(A.col),
                       c.upload(A.val), 8, 64, 4096)
    lib, h = c.lib, s.handle
    c.close()
    assert lib.smax_hip_scs_destroy(None, h) == capi.SUCCESS


def test_handle_destroyed_during_a_capture(ctx):
    """In relaxed mode freeing memory is allowed while a stream is captured:
    a handle that goes then, as by garbage collection, leaves the capture be."""
    import torch
    A = matgen.lomax_band(60_000)
    d = [ctx.upload(a) for a in (A.row_ptr, A.col, A.val)]
    S, T = (ctx.scs_from_crs(A.n_rows, A.n_cols, A.nnz, *d, 8, 64, 4096) for _ in range(2))
    x, y = ctx.upload(matgen.uniform_f64(3, A.n_cols)), ctx.zeros(A.n_rows, np.float64)
    S.apply(capi.F64, x, y, unpermuted=True)
    want = ctx.download(y)
    st, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    ctx.set_stream(st.cuda_stream)
    try:
        with torch.cuda.graph(g, stream=st, capture_error_mode="relaxed"):
            S.apply(capi.F64, x, y, unpermuted=True)
            # without the context: its stream, which is being captured, is not waited for
            assert ctx.lib.smax_hip_scs_destroy(None, T.handle) == capi.SUCCESS
            S.apply(capi.F64, x, y, unpermuted=True)
        for _ in range(3):
            ctx._check(ctx.lib.smax_hip_zero(ctx.handle, y.ptr, y.nbytes))
            ctx.sync()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(ctx.download(y), want)
    finally:
        ctx.set_stream(None)
    S.destroy()
    for a in (*d, x, y):
        a.free()


# Its own process: no other context of the device keeps the blocks.
MEMORY = """
import sys, torch
sys.path.insert(0, sys.argv[1])
from smaxkernels_amd import capi

MB, GB = 1 << 20, 1 << 30
free = lambda: torch.cuda.mem_get_info()[0]

def handle(c, n):  # 28 bytes a row, and the conversion's scratch
    ptr = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    col, val = ptr[:n], torch.ones(n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    h = c.scs_from_crs(n, n, n, ptr, col, val, 8, 64, 4096)
    del ptr, col, val
    torch.cuda.empty_cache()
    return h

with capi.Context(0) as c:  # what the first use of everything takes
    handle(c, 4_000_000).destroy()

start = free()
def held():
    return start - free()
def back(what):
    assert held() < 64 * MB, (what, held())
def keep(c):
    handle(c, 8_000_000).destroy()
    assert held() > 200 * MB, held()

with capi.Context(0) as c:
    back("a new context")
    keep(c)
    c.trim()
    back("trim")
    keep(c)
    p = capi.vp()
    assert c.lib.smax_hip_malloc(c.handle, capi.C.byref(p), 1 << 50) == capi.ERROR_OUT_OF_MEMORY
    back("a failed allocation")
    keep(c)
    d = capi.Context(0)
assert held() > 200 * MB, "the other context"
d.close()
back("the last context")

with capi.Context(0) as c:
    hs = [handle(c, 70_000_000) for _ in range(3)]
    in_use = held()
    assert in_use > 5.5 * GB, in_use
    for h in hs:
        h.destroy()
    assert 2 * GB < held() < 4 * GB + 64 * MB, held()
back("the last context")
print("done")
"""


def test_memory_goes_back():
    """By free device memory: kept blocks go by trim, a failed allocation (of
    a size that no device has) and the last context, and what is kept stays
    within 4 GiB when 5.5 GB are freed."""
    root = Path(__file__).resolve().parents[1]
    p = subprocess.run([sys.executable, "-c", MEMORY, str(root)], capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0 and "done" in p.stdout, p.stdout + p.stderr
