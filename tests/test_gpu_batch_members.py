"""Members of a batch (include/amr_batch.h) between their own amr_dev_* calls
(GPU).

Every member must come out as a context of its own that runs the plain stages
on the CPU oracle: cells and ghosts bit for bit in FP64.
"""
import ctypes

import numpy as np
import pytest

import amrcheck as A
import meshgen
import miniamr_amd as M
from conftest import require

pytestmark = pytest.mark.gpu


class Batch:
    """A batch and, per member, a device context of the oracle."""

    def __init__(self, stencil, shape=None):
        require(M.LIB_PATH, "run __graft_entry__.build()")
        require(A.ORACLE_SO, "run __graft_entry__.build()")
        self.lib, self.cpu = M.load_library(M.LIB_PATH), M.load_library(A.ORACLE_SO)
        self.stencil, self.pairs = stencil, []
        self.h = ctypes.c_void_p()
        self.ok(self.lib.amr_batch_create(0, M.PREC_F64, stencil, ctypes.byref(self.h)))
        if shape:
            self.ok(self.lib.amr_batch_set_shape(self.h, ctypes.byref(M.BatchShape(*shape))))

    def ok(self, rc):
        assert rc == 0, self.lib.amr_batch_last_error(self.h)

    def add(self, n, nv, slots):
        kw = dict(nx=n[0], ny=n[1], nz=n[2], num_vars=nv, max_blocks=slots, stencil=self.stencil)
        m = M.Device.__new__(M.Device)          # the batch owns the context
        m.lib, m.cfg = self.lib, M.Config(*n, nv, slots, self.stencil, M.PREC_F64, 0)
        m.shape = (nv, n[0] + 2, n[1] + 2, n[2] + 2)
        m.h = ctypes.c_void_p()
        self.ok(self.lib.amr_batch_add(self.h, ctypes.byref(m.cfg), ctypes.byref(m.h)))
        c = M.Device(lib=self.cpu, **kw)
        self.pairs.append((m, c))
        return m, c

    def timestep(self, stage0, nstages, permute=False):
        self.ok(self.lib.amr_batch_timestep(self.h, stage0, nstages, 0, int(permute)))
        for _, c in self.pairs:
            for s in range(stage0, stage0 + nstages):
                c.stage(0, c.cfg.num_vars, stage=s, permute=permute)

    def check(self, what):
        for q, (m, c) in enumerate(self.pairs):
            for s in range(c.cfg.max_blocks):
                assert np.array_equal(m.download(s), c.download(s)), (what, q, s)

    def close(self):
        for m, c in self.pairs:
            m.h = ctypes.c_void_p()
            c.close()
        self.lib.amr_batch_destroy(self.h)


def fill(rng, pair, slots):
    for s in range(slots):
        cells = rng.random(pair[0].shape)
        for d in pair:
            d.upload(s, cells)


@pytest.mark.parametrize("exchange_vars", [4, 8, 16])
def test_wavefront_exchange_items(exchange_vars):
    """Coarse/fine jobs of one wavefront each copy the plane's present cells to
    the ring beside a boundary face before any lane writes the new ones: faces
    below, at and above the 64 lanes, partial groups of variables."""
    print("case: batch, wavefront exchange items of %d variables" % exchange_vars, flush=True)
    rng = np.random.default_rng(exchange_vars)
    b = Batch(27, (1, 0, 0, 0, exchange_vars, 64))
    try:
        for n, nv in (((4, 4, 4), 3), ((6, 10, 14), 5), ((8, 8, 8), 17), ((2, 16, 16), 9)):
            pair = b.add(n, nv, 12)
            fill(rng, pair, 12)
            plan = meshgen.random_plan(rng, 5, 6, kinds=(M.FACE_BC, M.FACE_PROLONG,
                                                         M.FACE_RESTRICT, M.FACE_SAME))
            for d in pair:
                d.set_mesh(range(11), plan)
        for k in range(3):
            b.timestep(2 * k, 2)
        b.check("wavefront items")
    finally:
        b.close()


@pytest.mark.parametrize("st", [7, 27])
def test_members_cells_in_the_other_copy(st):
    """The batch steps a member's present cells after calls that left them in
    the other interior copy: an odd number of fused stages, of all variables
    and of one, and a saved state."""
    print("case: batch, members moved between timesteps, stencil %d" % st, flush=True)
    rng = np.random.default_rng(st)
    b = Batch(st)
    try:
        for n, nv in (((4, 6, 8), 3), ((8, 8, 8), 2)):
            pair = b.add(n, nv, 12)
            fill(rng, pair, 12)
            plan = meshgen.random_plan(rng, 5, 6)
            for d in pair:
                d.set_mesh(range(11), plan)
        m, c = b.pairs[0]
        b.timestep(0, 2)
        for k in range(3):
            m.stage_fused(0, 3, stage=k)
            c.stage(0, 3, stage=k)
        b.timestep(2, 2)
        m.stage_fused(1, 1)
        c.stage(1, 1)
        b.timestep(4, 2)
        b.timestep(6, 2)
        for d in (m, c):
            d.stage_fused(0, 3)
        b.timestep(8, 1)
        b.check("stages of a member")
        for d in (m, c):
            d.stage_fused(0, 3)
        b.timestep(10, 2)                       # the member now steps from the other copy
        size = ctypes.c_size_t()
        assert b.lib.amr_dev_state_bytes(m.h, ctypes.byref(size)) == 0
        state = np.empty(size.value, dtype=np.uint8)
        assert b.lib.amr_dev_save_state(m.h, state.ctypes.data_as(ctypes.c_void_p)) == 0
        b.timestep(12, 2)
        b.check("a saved state")
    finally:
        b.close()


@pytest.mark.parametrize("st", [7, 27])
def test_members_plan_reads_inactive_slots(st):
    """A member whose jobs read slots outside its active list: those cells stay
    where they are, in every stage of a timestep."""
    print("case: batch, inactive sources, stencil %d" % st, flush=True)
    rng = np.random.default_rng(st)
    b = Batch(st)
    try:
        for n, nv in (((4, 6, 8), 3), ((8, 8, 8), 2)):
            pair = b.add(n, nv, 12)
            fill(rng, pair, 12)
            plan = meshgen.random_plan(rng, 5, 6)
            for d in pair:
                d.set_mesh(range(5 if nv == 3 else 0, 11), plan)
        b.timestep(0, 4)
        b.check("inactive sources")
    finally:
        b.close()


@pytest.mark.parametrize("st", [7, 27])
def test_permuted_stages_after_fused_timesteps(st):
    """Permuted stages copy ghost cells that the stage before wrote; a fused
    timestep leaves them unwritten."""
    print("case: batch, permuted after fused, stencil %d" % st, flush=True)
    rng = np.random.default_rng(st)
    b = Batch(st)
    try:
        for n, box in (((4, 6, 8), (3, 2, 2)), ((8, 8, 8), (2, 1, 3))):
            order, plan = meshgen.box_plan(*box)
            pair = b.add(n, 2, len(order))
            fill(rng, pair, len(order))
            for d in pair:
                d.set_mesh(order, plan)
        for k in range(1, 6):
            b.timestep(0, 2)
            if k % 2:
                b.timestep(k, 1, permute=True)
            else:
                b.ok(b.lib.amr_batch_stage(b.h, k, 1, -1))
                for _, c in b.pairs:
                    c.stage(0, 2, stage=k, permute=True)
            b.check("permutation %d" % k)
    finally:
        b.close()
