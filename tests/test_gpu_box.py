"""The whole-box stencil kernels and the stages that read every face in place
(GPU).

7-point stages (amr_dev_stage_fused) read each ghost plane from where its
values come from -- same-level, boundary, coarse and fine neighbours -- and
need no exchange.  Cells (ghosts included, once they are asked for) must be
the CPU oracle's plain stages bit for bit in FP64, and the device's own plain
stages in the narrow storage forms.  Shapes: the smallest block, vectors of
two and of four cells, quarters that a vector straddles, more vectors than
threads, faces with as many cells as the interior, boxes too large for LDS
(the plane-by-plane kernels).  27-point blocks take the same kernels with the
exchange in front.
"""
import numpy as np
import pytest

import amrcheck as A
import meshgen
import miniamr_amd as M
from conftest import require

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (4, 4, 4), (6, 6, 6), (8, 8, 8), (10, 10, 10), (6, 10, 14), (12, 4, 8),
          (2, 20, 4), (16, 16, 16), (16, 2, 12), (14, 14, 14), (18, 18, 18), (4, 30, 30)]


def pair(n, nv, st, prec, other):
    kw = dict(nx=n[0], ny=n[1], nz=n[2], num_vars=nv, max_blocks=14, stencil=st, precision=prec)
    return M.Device(lib=M.load_library(M.LIB_PATH), **kw), M.Device(lib=other, **kw)


@pytest.mark.parametrize("prec", [M.PREC_F64, M.PREC_F32, M.PREC_BF16], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("st", [7, 27])
@pytest.mark.parametrize("n", SHAPES, ids=["%dx%dx%d" % n for n in SHAPES])
def test_stages_match(n, st, prec, monkeypatch):
    require(M.LIB_PATH, "run __graft_entry__.build()")
    require(A.ORACLE_SO, "run __graft_entry__.build()")
    print("case: box stencil=%d block=%s precision=%d" % (st, n, prec), flush=True)
    if st == 27:
        monkeypatch.setenv("MINIAMR_FUSED", "2")
    other = M.load_library(A.ORACLE_SO if prec == M.PREC_F64 else M.LIB_PATH)
    nv = 3
    g, c = pair(n, nv, st, prec, other)
    rng = np.random.default_rng(3 + n[0] + 10 * st)
    order = list(rng.permutation(11))
    plan = meshgen.random_plan(rng, 5, 6)
    for s in range(11):
        cells = rng.random(g.shape)
        g.upload(s, cells)
        c.upload(s, cells)
    for d in (g, c):
        d.set_mesh(order, plan)
        d.reserve_sums(3)
    for k in range(3):                      # an odd number of moves between the copies
        g.stage_fused(0, nv, stage=k, permute=st == 7 and k == 1, sum_row=k)
        c.stage(0, nv, stage=k, permute=st == 7 and k == 1, sum_row=k)
    g.stage_fused(1, 1, stage=3)            # one variable: the copies differ between variables
    c.stage(1, 1, stage=3)
    g.stage_fused(0, 1, stage=3)
    c.stage(0, 1, stage=3)
    g.stage_fused(2, 1, stage=3)
    c.stage(2, 1, stage=3)
    np.testing.assert_allclose(g.read_sums(0, 3), c.read_sums(0, 3), rtol=1e-13)
    for s in range(11):
        assert np.array_equal(g.download(s), c.download(s)), s
    # some variables one stage ahead: read them, then go on with all of them
    for k, (start, num) in enumerate([(0, 1), (0, nv), (1, 2), (0, nv)]):
        g.stage_fused(start, num, stage=k)
        c.stage(start, num, stage=k)
        if k < 3:
            assert np.array_equal(g.download(order[k]), c.download(order[k])), k
    for s in range(11):
        assert np.array_equal(g.download(s), c.download(s)), s


def test_inactive_slots_and_saved_states():
    """Slots outside the active list keep their cells while fused stages move
    the active blocks' cells to the other interior copy, and a saved state is
    the same whatever stages ran before."""
    require(M.LIB_PATH, "run __graft_entry__.build()")
    print("case: inactive slots, saved states", flush=True)
    lib = M.load_library(M.LIB_PATH)
    kw = dict(nx=4, ny=6, nz=8, num_vars=3, max_blocks=24, stencil=7)
    g, c = M.Device(lib=lib, **kw), M.Device(lib=lib, **kw)
    rng = np.random.default_rng(8)
    for s in range(24):
        cells = rng.random(g.shape)
        g.upload(s, cells)
        c.upload(s, cells)
    plan = meshgen.random_plan(rng, 5, 6)
    for d, stage in ((g, g.stage_fused), (c, c.stage)):
        d.set_mesh(range(11), plan)
        for k in range(3):
            stage(0, 3, stage=k)
        # an inactive parent's children, one of them a slot that was active
        d.split([(15, 16 + o, o, 0) for o in range(7)] + [(15, 10, 7, 0)])
        stage(0, 3, stage=3)
    for s in (12, 15, 16, 22, 10, 3):
        assert np.array_equal(g.download(s), c.download(s)), s
    # slots 11 and up become active and are read
    jobs = [np.array([(M.FACE_SAME, 2 * d, s, (s + 1) % 24, 0, 0) for s in range(24)],
                     dtype=M.FACE_JOB) for d in range(3)]
    for d, stage in ((g, g.stage_fused), (c, c.stage)):
        d.set_mesh(range(24), jobs)
        stage(0, 3, stage=0)
    import ctypes
    size = ctypes.c_size_t()
    lib.amr_dev_state_bytes(g.h, ctypes.byref(size))
    state = np.zeros(size.value, dtype=np.uint8)
    ptr = state.ctypes.data_as(ctypes.c_void_p)
    assert lib.amr_dev_save_state(g.h, ptr) == 0
    want = [c.download(s) for s in range(24)]
    fresh = M.Device(lib=lib, **kw)
    assert lib.amr_dev_load_state(fresh.h, ptr) == 0
    g.stage_fused(0, 3, stage=1)
    assert lib.amr_dev_load_state(g.h, ptr) == 0
    for s in range(24):
        assert np.array_equal(fresh.download(s), want[s]), s
        assert np.array_equal(g.download(s), want[s]), s


@pytest.mark.parametrize("prec", [M.PREC_F64, M.PREC_F32, M.PREC_BF16], ids=["f64", "f32", "bf16"])
def test_download_into_page_locked_memory(prec):
    """A download into page-locked memory (written by the conversion kernel
    itself) gives the values of one into pageable memory, at the start, in the
    middle and at the end of the allocation, and leaves its neighbours alone."""
    require(M.LIB_PATH, "run __graft_entry__.build()")
    import ctypes
    lib = M.load_library(M.LIB_PATH)
    hip = ctypes.CDLL("libamdhip64.so")
    d = M.Device(nx=6, ny=4, nz=10, num_vars=3, max_blocks=2, stencil=7, precision=prec, lib=lib)
    rng = np.random.default_rng(2)
    d.upload(1, rng.random(d.shape))
    want = d.download(1)
    n, lead = want.size, 5
    ptr = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(8 * (3 * n + lead)), 0) == 0
    buf = np.ctypeslib.as_array((ctypes.c_double * (3 * n + lead)).from_address(ptr.value))
    try:
        for at in (0, lead, n + lead, 2 * n + lead):
            buf[:] = -1.0
            out = ctypes.cast(ptr.value + 8 * at, ctypes.POINTER(ctypes.c_double))
            assert lib.amr_dev_download_block(d.h, 1, out) == 0
            assert np.array_equal(buf[at:at + n], want.ravel())
            assert np.all(buf[:at] == -1.0) and np.all(buf[at + n:] == -1.0)
    finally:
        d.close()
        hip.hipHostFree(ptr)
