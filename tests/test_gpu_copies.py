"""Calls that meet the cells a fused stage has moved to the other interior
copy, or the ghost planes it has left unwritten (GPU).

The context under test runs amr_dev_stage_fused; its twin -- the CPU oracle,
or a context of the library where the oracle has no such call -- runs the
plain stages.  All cells, ghosts included, must be the same bits.
"""
import ctypes

import numpy as np
import pytest

import amrcheck as A
import meshgen
import miniamr_amd as M
from conftest import require

pytestmark = pytest.mark.gpu

N, NV, SLOTS = (4, 6, 8), 3, 32


def pair(stencil, other=None, n=N, nv=NV, slots=SLOTS, seed=1):
    """A context and its twin with the same random cells in every slot."""
    require(M.LIB_PATH, "run __graft_entry__.build()")
    require(A.ORACLE_SO, "run __graft_entry__.build()")
    kw = dict(nx=n[0], ny=n[1], nz=n[2], num_vars=nv, max_blocks=slots, stencil=stencil)
    g = M.Device(lib=M.load_library(M.LIB_PATH), **kw)
    c = M.Device(lib=M.load_library(other or A.ORACLE_SO), **kw)
    rng = np.random.default_rng(seed)
    for s in range(slots):
        cells = rng.random(g.shape)
        for d in (g, c):
            d.upload(s, cells)
    return g, c, rng


def stages(g, c, start, num, first=0, count=1, permute=False):
    for k in range(first, first + count):
        g.stage_fused(start, num, stage=k, permute=permute)
        c.stage(start, num, stage=k, permute=permute)


def same(g, c, slots=range(SLOTS)):
    for s in slots:
        assert np.array_equal(g.download(s), c.download(s)), s


@pytest.mark.parametrize("st", [7, 27])
def test_inactive_slots_while_variables_are_in_different_copies(st):
    """One fused stage of one variable, then a look at slots outside the active
    list: a download, a packed message."""
    print("case: inactive slots, mixed copies, stencil %d" % st, flush=True)
    import torch
    g, c, rng = pair(st)
    plan = meshgen.random_plan(rng, 5, 6)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, 1)
    same(g, c, [12, 3, 12, 13])
    stages(g, c, 1, 2, 1)
    stages(g, c, 2, 1, 2)
    p = M.Device(lib=g.lib, nx=N[0], ny=N[1], nz=N[2], num_vars=NV, max_blocks=SLOTS, stencil=st)
    msgs = np.zeros(2, dtype=M.FACE_MSG)
    msgs["slot"] = [14, 3]
    out = []
    for s in (14, 3):
        p.upload(s, c.download(s))
    length = g.face_msg_len(0, 1, 0)
    msgs["offset"] = [0, NV * length]
    for d in (g, p):
        buf = torch.full((2 * NV * length,), -1.0, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        d.pack_faces(0, 1, 0, NV, msgs, buf)
        d.sync()
        out.append(buf.cpu().numpy())
    assert np.array_equal(out[0], out[1])
    same(g, c)


@pytest.mark.parametrize("how", ["split", "split_noalloc", "consolidate"])
@pytest.mark.parametrize("st", [7, 27])
def test_refinement_while_variables_are_in_different_copies(st, how):
    """Children (a merged block) written after a fused stage of one variable
    keep their cells through the set_mesh that makes them active; parents
    (children) are read whether they are active or not."""
    print("case: %s, mixed copies, stencil %d" % (how, st), flush=True)
    g, c, rng = pair(st)
    plan, after = meshgen.random_plan(rng, 5, 6), meshgen.random_plan(rng, 5, 24)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, 1)
    # an active source with inactive targets, and inactive sources
    jobs = [(3, 16 + o, o, 0) for o in range(8)] + [(12, 24 + o, o, 0) for o in range(8)]
    if how == "consolidate":
        jobs = [(16, o, o, 0) for o in range(8)] + [(12, 24 + o, o, 0) for o in range(8)]
    for d in (g, c):
        getattr(d, how)(jobs)
        d.set_mesh(range(29), after)
    same(g, c)
    stages(g, c, 0, NV, 1, 2)
    same(g, c)


@pytest.mark.parametrize("st", [7, 27])
def test_inactive_sources_while_variables_are_in_different_copies(st):
    """A plan whose jobs read slots outside the active list, after a fused stage
    of one variable: plain stages read those slots' cells."""
    print("case: inactive sources, mixed copies, stencil %d" % st, flush=True)
    g, c, rng = pair(st)
    plan, reads = meshgen.random_plan(rng, 5, 6), meshgen.random_plan(rng, 5, 6)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, 1)
    for d in (g, c):
        d.set_mesh(range(5, 11), reads)
    stages(g, c, 0, NV, 1, 3)
    same(g, c)


def test_compare_cells_while_variables_are_in_different_copies():
    print("case: compare_cells, mixed copies", flush=True)
    g, c, rng = pair(7, other=M.LIB_PATH)
    plan = meshgen.random_plan(rng, 5, 6)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, 1)
    stages(g, c, 2, 1, 1)
    worst = (ctypes.c_double * NV)(*[-1.0] * NV)
    assert g.lib.amr_dev_compare_cells(g.h, c.h, 0, NV, worst) == 0
    assert list(worst) == [0.0] * NV
    same(g, c)


@pytest.mark.parametrize("what", ["stage", "comm"])
@pytest.mark.parametrize("st", [7, 27])
def test_permuted_exchange_after_fused_stages(st, what):
    """With y or z first, a 27-point exchange copies ghost cells that the stage
    before wrote: after a fused stage they are brought up to date first.  Every
    block of a box is its neighbours' source, the domain boundary included."""
    print("case: permuted exchange after fused stages, %s, stencil %d" % (what, st), flush=True)
    g, c, _ = pair(st)
    order, plan = meshgen.box_plan(3, 2, 2)
    for d in (g, c):
        d.set_mesh(order, plan)
    for k in range(6):
        stages(g, c, 0, NV, 0, 1 + k % 2)
        if what == "comm":
            g.comm(0, NV, stage=k, permute=True)
            c.comm(0, NV, stage=k, permute=True)
        else:
            stages(g, c, 0, NV, k, 1, permute=True)
        same(g, c, order)


@pytest.mark.parametrize("st", [7, 27])
def test_upload_after_fused_stages(st):
    """An upload's ghost cells stay as uploaded, and the stencil reads them."""
    print("case: upload after fused stages, stencil %d" % st, flush=True)
    g, c, rng = pair(st)
    plan = meshgen.random_plan(rng, 5, 6)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, NV, 0, 3)
    for s in (2, 7, 10):
        cells = rng.random(g.shape)
        for d in (g, c):
            d.upload(s, cells)
    same(g, c)
    stages(g, c, 0, NV, 3)
    cells = rng.random(g.shape)
    for d in (g, c):
        d.upload(8, cells)
        for v in range(NV):
            d.stencil(v)
    same(g, c)


@pytest.mark.parametrize("st", [7, 27])
def test_clear_block_after_fused_stages(st):
    """A cleared slot is zero, ghost planes too, and its neighbours' ghost
    planes keep the cells they had from it."""
    print("case: clear_block after fused stages, stencil %d" % st, flush=True)
    g, c, rng = pair(st, other=M.LIB_PATH)
    plan = meshgen.random_plan(rng, 5, 6)
    for d in (g, c):
        d.set_mesh(range(11), plan)
    stages(g, c, 0, NV)
    for s in (1, 2, 3, 8, 20):
        for d in (g, c):
            assert d.lib.amr_dev_clear_block(d.h, s) == 0
    assert not g.download(8).any() and not g.download(20).any()
    same(g, c)
