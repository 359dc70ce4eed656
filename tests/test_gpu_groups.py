"""Whole --stencil 0 stages by groups of variables (GPU).

A stage over all variables updates the groups (u, mat+u, 2*mat+u, 3*mat+u)
independently; cells and clamp counts must be those of the variables one
after another -- the CPU oracle's in FP64, the device's own variable by
variable in the narrow forms -- over all six calculation stages.  Variable
counts: one material (variable 1 is then class 1), several, and variables
left over for the plain average; blocks that fit in LDS and ones that do not.
"""
import numpy as np
import pytest

import amrcheck as A
import meshgen
import miniamr_amd as M
from conftest import require

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [M.PREC_F64, M.PREC_F32, M.PREC_BF16], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("nv", [4, 7, 9, 13])
@pytest.mark.parametrize("n", [(4, 4, 4), (12, 12, 12), (6, 14, 10), (16, 16, 16), (2, 30, 4)],
                         ids=lambda n: "%dx%dx%d" % n)
def test_grouped_stages_match(n, nv, prec):
    require(M.LIB_PATH, "run __graft_entry__.build()")
    require(A.ORACLE_SO, "run __graft_entry__.build()")
    print("case: groups block=%s vars=%d precision=%d" % (n, nv, prec), flush=True)
    f64 = prec == M.PREC_F64
    kw = dict(nx=n[0], ny=n[1], nz=n[2], num_vars=nv, max_blocks=12, stencil=0, precision=prec)
    g = M.Device(lib=M.load_library(M.LIB_PATH), **kw)
    c = M.Device(lib=M.load_library(A.ORACLE_SO if f64 else M.LIB_PATH), **kw)
    rng = np.random.default_rng(50 + nv)
    a1, a0 = float(rng.random()), rng.random(nv // 4)
    plan = meshgen.random_plan(rng, 5, 6)
    for s in range(11):
        cells = 2.0 * rng.random(g.shape)
        for d in (g, c):
            d.upload(s, cells)
    for d in (g, c):
        d.set_materials(a1, a0)
        d.set_mesh(range(11), plan)
    for stage in range(7):
        g.stage(0, nv, stage=stage)
        if f64:
            c.stage(0, nv, stage=stage)
        else:
            c.comm(0, nv, stage=stage)
            for v in range(nv):
                c.stencil_stage(v, stage)
    for s in range(11):
        assert np.array_equal(g.download(s), c.download(s)), s
    assert g.check_counts() == c.check_counts()
