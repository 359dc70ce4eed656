"""The workloads whose speed is watched: what users of this framework run.

A case is a dict of plain values; its "kind" says which public entry points
one pass goes through:

  grid     miniamr_amd.Device, driven by a caller's own loop: a uniform grid
           of blocks, `stages` stages (exchange, stencil, checksums every
           fifth), then the cells and the checksums;
  amr      miniamr_amd.Run, the drop-in driver: `steps` timesteps of 20
           stages on a refined mesh around one sphere, then the cells of
           every active block and the last timestep's checksums;
  refine   the same driver with a sphere that crosses the domain and comes
           back while the mesh is refined after every timestep of 5 stages;
           one pass is one whole period, so every pass meets the same meshes;
  batch    miniamr_amd.BatchRun: independent runs stepped together;
  reverse  the reverse pass of a taped run (include/amr_adjoint.h): weights on
           the final cells in, gradient of the initial cells out.

Cells come back the way every caller gets them, block by block through
amr_dev_download_block, into page-locked memory kept from pass to pass; the
stages between two such outputs are as many as between two outputs of a
real run.  The runs keep on from where the last pass left them.
"""
import ctypes
import functools
import math
import os

import numpy as np
import torch

import miniamr_amd as M

PRECISION = {"f64": M.PREC_F64, "f32": M.PREC_F32, "bf16": M.PREC_BF16}
BYTES = {"f64": 8, "f32": 4, "bf16": 2}
CHECKSUM_FREQ = 5          # stages between two checksums
STAGES = 20                # stages of a driver timestep (amr, batch, reverse)
REFINE_STAGES = 5          # the same where the mesh is refined every timestep
PERIOD = 32                # timesteps after which the moving sphere is back
ENDLESS = 1000000000       # timesteps of a run that a caller steps as it likes


def _case(name, kind, n, num_vars, stencil, precision, **more):
    c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "num_vars": num_vars,
         "stencil": stencil, "precision": precision}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    cube = lambda n: (n, n, n)  # noqa: E731
    return [
        # The smallest meshes in use (the differentiation form's block size):
        # a stage is a few microseconds of work, so launches and gaps count.
        _case("grid_8_7pt_f64", "grid", cube(8), 4, 7, "f64", bx=4, by=4, bz=4, stages=400),
        # Uneven blocks, an odd number of variables, a mesh that fits in cache.
        _case("grid_6x10x14_27pt_f32", "grid", (6, 10, 14), 11, 27, "f32", bx=5, by=3, bz=4,
              stages=200),
        # The reference's default block, variables and stencil on a medium mesh.
        _case("amr_10_7pt_f64", "amr", cube(10), 40, 7, "f64", init=2, levels=3, radius=0.25,
              max_blocks=900, code=0, steps=20),
        # The bandwidth-scale configuration's block, variables and stencil in
        # FP64, the precision the reference computes in; the largest case.
        _case("amr_16_27pt_f64", "amr", cube(16), 40, 27, "f64", init=3, levels=3, radius=0.2,
              max_blocks=1600, code=0, steps=20),
        # The same stage in the two narrow storage forms.
        _case("amr_16_27pt_f32", "amr", cube(16), 20, 27, "f32", init=2, levels=4, radius=0.2,
              max_blocks=2600, code=0, steps=20),
        _case("amr_16_27pt_bf16", "amr", cube(16), 40, 27, "bf16", init=2, levels=3,
              radius=0.25, max_blocks=900, code=0, steps=20),
        # The default stencil on the larger block.
        _case("amr_16_7pt_f32", "amr", cube(16), 40, 7, "f32", init=4, levels=2, radius=0.2,
              max_blocks=800, code=0, steps=20),
        # Whole ghost planes (--code 1) on uneven blocks.
        _case("amr_6x10x14_code1_f64", "amr", (6, 10, 14), 11, 27, "f64", init=2, levels=3,
              radius=0.25, max_blocks=900, code=1, steps=10),
        # The variable-work stencils (--stencil 0): six calculation stages.
        _case("amr_12_stencil0_f64", "amr", cube(12), 20, 0, "f64", init=2, levels=2,
              radius=0.25, max_blocks=500, code=0, steps=6),
        # A moving object: refinement (marking, split, consolidate, new plans)
        # between short timesteps.
        _case("refine_16_27pt_f64", "refine", cube(16), 12, 27, "f64", init=2, levels=3,
              radius=0.15, max_blocks=1200, code=0, steps=PERIOD),
        # Many small independent runs on one GPU, three block sizes.
        _case("batch_12_runs_f32", "batch", (0, 0, 0), 0, 27, "f32", runs=12, pick=0, steps=10),
        # Gradients: the adjoint kernels over a whole tape.
        _case("reverse_16_27pt_f32", "reverse", cube(16), 20, 27, "f32", init=2, levels=2,
              radius=0.25, max_blocks=500, code=0, steps=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any even block sizes, any number of
    variables, both stencils and codes, the three storage types."""
    kind = rng.choice(("grid", "grid", "grid", "amr", "amr", "amr", "amr", "refine", "batch",
                       "reverse"))
    precision = rng.choice(("f64", "f64", "f32", "bf16"))
    stencil = rng.choice((7, 27))
    n = [2 * rng.randint(2, 10) for _ in range(3)]
    if rng.random() < 0.5:
        n = [n[0]] * 3
    num_vars = _log_int(rng, 1, 40)
    radius = round(rng.uniform(0.1, 0.3), 3)
    cells = n[0] * n[1] * n[2]
    if kind == "grid":
        b = [_log_int(rng, 1, 8) for _ in range(3)]
        num_vars = max(1, min(num_vars, int(2e7 / (b[0] * b[1] * b[2] * cells))))
        return _case(None, kind, n, num_vars, stencil, precision, bx=b[0], by=b[1], bz=b[2],
                     stages=2 * rng.randint(20, 200))
    if kind == "batch":
        return _case(None, kind, (0, 0, 0), 0, 27, "f32", runs=rng.randint(4, 12),
                     pick=rng.randint(0, 50), steps=10)
    init, levels = rng.randint(1, 3), rng.randint(1, 3)
    if kind == "reverse":
        precision = rng.choice(("f64", "f32"))
        num_vars, levels = min(num_vars, 20), min(levels, 2)
    elif kind == "amr" and rng.random() < 0.15:
        stencil, num_vars, levels = 0, min(max(num_vars, 4), 20), min(levels, 2)
    code = rng.choice((0, 0, 0, 1)) if kind == "amr" else 0
    if kind == "refine":
        num_vars = min(num_vars, 12)
    # at most about a gigabyte of cells
    num_vars = max(4 if stencil == 0 else 1,
                   min(num_vars, int(4e8 / (_room(init, levels, radius) * cells))))
    return _case(None, kind, n, num_vars, stencil, precision, init=init, levels=levels,
                 radius=radius, max_blocks=_room(init, levels, radius), code=code,
                 steps={"amr": rng.randint(6, 20), "refine": PERIOD, "reverse": 10}[kind]
                 if stencil else 6)


def _room(init, levels, radius):
    """Block slots that a mesh around a sphere surface never runs out of: the
    estimate of configs/make_batch64.py, three times."""
    return max(64 + 8 * init ** 3,
               int(3 * (45.0 * (init * 2 ** levels * radius) ** 2 + 8 * init ** 3)))


# ------------------------------------------------------------- the driver
def _arguments(case, seed, tiny=False):
    """The driver's command line of an amr, refine or reverse case; tiny: the
    same mesh with the smallest blocks (the mesh depends on the objects only)."""
    moving = case["kind"] == "refine"
    # a sphere's centre crosses the unit domain in 16 steps and bounces
    sphere = ("--object 2 1 0.5 0.45 0.55 0.0625 0 0 {r} {r} {r} 0 0 0" if moving else
              "--object 2 0 0.5 0.45 0.55 0 0 0 {r} {r} {r} 0 0 0").format(r=case["radius"])
    size = [2, 2, 2] if tiny else [case["nx"], case["ny"], case["nz"]]
    return ("--init_x {i} --init_y {i} --init_z {i} --nx {n[0]} --ny {n[1]} --nz {n[2]} "
            "--num_vars {v} --stencil {s} --code {c} --num_refine {l} --max_blocks {b} "
            "--num_tsteps {t} --stages_per_ts {st} --checksum_freq {cf} --refine_freq {rf} "
            "--error_tol -10 --report_perf 0 --seed {seed} --precision {p} --num_objects 1 "
            "{sphere}").format(
                i=case["init"], n=size, v=1 if tiny else case["num_vars"],
                s=7 if tiny else case["stencil"], c=case["code"], l=case["levels"],
                b=case["max_blocks"],
                t=case["steps"] if case["kind"] == "reverse" else ENDLESS,
                st=REFINE_STAGES if moving else STAGES, cf=CHECKSUM_FREQ,
                rf=1 if moving else 4, seed=seed, p="f64" if tiny else case["precision"],
                sphere=sphere)


@functools.lru_cache(maxsize=None)
def _batch_lines(runs, pick):
    """Command lines of a batch: rows of the 64-run workload in small meshes
    (1,000 block slots at most), with static spheres and no end."""
    rows = []
    with open(os.path.join(M.PKG, "configs", "batch64.txt")) as f:
        for line in f:
            t = line.split()
            if not t or t[0] == "#":
                continue
            if int(t[t.index("--max_blocks") + 1]) > 1000:
                continue
            o = t.index("--object")
            t[o + 6:o + 9] = ["0", "0", "0"]
            t[t.index("--num_tsteps") + 1] = str(ENDLESS)
            rows.append(t)
    return [rows[(pick + i) % len(rows)] for i in range(runs)]


def _batch_arguments(case, seed):
    out = []
    for i, t in enumerate(_batch_lines(case["runs"], case["pick"])):
        t = list(t)
        t[t.index("--seed") + 1] = str((seed * 64 + i) % (1 << 31))
        out.append(" ".join(t) + " --report_perf 0")
    return out


class _Held:
    """What a program keeps between passes; frees it when dropped."""

    def __init__(self):
        self.ends = []

    def __del__(self):
        for end in reversed(self.ends):
            end()


def _host_cells(blocks, num_vars, n):
    """Page-locked room for `blocks` blocks, ghost cells included."""
    return torch.zeros((blocks, num_vars, n[0] + 2, n[1] + 2, n[2] + 2), dtype=torch.float64,
                       pin_memory=True)


def _inner(cells):
    return cells[..., 1:-1, 1:-1, 1:-1]


def _addresses(cells):
    """The address of each block's cells, as the C interface takes it."""
    base, step = cells.data_ptr(), cells.stride(0) * 8
    return [ctypes.cast(base + i * step, ctypes.POINTER(ctypes.c_double))
            for i in range(cells.shape[0])]


class _Cells:
    """The cells and checksums of one run of the driver."""

    def __init__(self, host, dev, run):
        self.host, self.dev, self.run = host, dev, run
        st = M.RunStats()
        host.amr_run_stats_get(run, ctypes.byref(st))
        self.st = st
        self.device = ctypes.c_void_p(host.amr_run_device(run))
        self.n = (st.nx, st.ny, st.nz)
        self.slot, self.level = ctypes.c_int32(), ctypes.c_int32()
        self.lo, self.hi = (ctypes.c_double * 3)(), (ctypes.c_double * 3)()

    def slots(self):
        out = []
        for i in range(self.host.amr_run_active(self.run)):
            self.host.amr_run_block(self.run, i, ctypes.byref(self.slot),
                                    ctypes.byref(self.level), self.lo, self.hi)
            out.append(self.slot.value)
        return out

    def read(self, slots, at):
        for s, p in zip(slots, at):
            if self.dev.amr_dev_download_block(self.device, s, p):
                raise M.AmrError(self.dev.amr_dev_last_error(self.device).decode())

    def sums(self, stages):
        rows = -(-stages // CHECKSUM_FREQ)
        out = np.empty((rows, self.st.num_vars))
        if self.dev.amr_dev_read_sums(self.device, 0, rows,
                                      out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))):
            raise M.AmrError(self.dev.amr_dev_last_error(self.device).decode())
        return out


# ----------------------------------------------------------- uniform grids
def _grid_jobs(case):
    """The exchange plan of a uniform bx x by x bz grid of blocks (slot
    numbers x fastest): a same-level copy or a reflecting boundary per face."""
    b = (case["bx"], case["by"], case["bz"])
    slot = lambda p: p[0] + b[0] * (p[1] + b[1] * p[2])  # noqa: E731
    plan = []
    for d in range(3):
        jobs = []
        for z in range(b[2]):
            for y in range(b[1]):
                for x in range(b[0]):
                    for hi in (0, 1):
                        q = [x, y, z]
                        q[d] += 1 if hi else -1
                        here = slot((x, y, z))
                        if 0 <= q[d] < b[d]:
                            jobs.append((M.FACE_SAME, 2 * d + hi, here, slot(q), 0, 0))
                        else:
                            jobs.append((M.FACE_BC, 2 * d + hi, here, here, 0, 0))
        plan.append(np.array(jobs, dtype=M.FACE_JOB))
    return plan


def _grid_values(case, seed):
    """Initial cells of each block, uniform in [0, 1) as the driver's, with
    the ghost cells of a new block (zero)."""
    nb = case["bx"] * case["by"] * case["bz"]
    g = torch.Generator().manual_seed(int(seed))
    cells = torch.zeros((nb, case["num_vars"], case["nx"] + 2, case["ny"] + 2, case["nz"] + 2),
                        dtype=torch.float64)
    _inner(cells)[:] = torch.rand((nb, case["num_vars"], case["nx"], case["ny"], case["nz"]),
                                  generator=g, dtype=torch.float64)
    return cells


# ------------------------------------------------------------- the cases
def prepare(case, seed):
    kind, s = case["kind"], _Held()
    s.case = case
    if kind == "grid":
        nb = case["bx"] * case["by"] * case["bz"]
        s.dev = M.Device(case["nx"], case["ny"], case["nz"], case["num_vars"], nb,
                         stencil=case["stencil"], precision=PRECISION[case["precision"]])
        for slot, cells in enumerate(_grid_values(case, seed).numpy()):
            s.dev.upload(slot, cells)
        s.dev.set_mesh(range(nb), _grid_jobs(case))
        s.dev.reserve_sums(-(-case["stages"] // CHECKSUM_FREQ))
        s.cells = _host_cells(nb, case["num_vars"], (case["nx"], case["ny"], case["nz"]))
        s.at = _addresses(s.cells)
        s.ends.append(s.dev.close)
        s.dev.sync()
        return s
    host, dev = M.load_host_library(), M.load_library()
    if kind == "batch":
        s.batch = M.BatchRun(_batch_arguments(case, seed), autotune=True, host=host)
        s.ends.append(s.batch.close)
        s.members, s.out, s.slots, s.at = [], [], [], []
        for i in range(case["runs"]):
            c = _Cells(host, dev, ctypes.c_void_p(host.amr_batch_run_get(s.batch.h, i)))
            s.members.append(c)
            s.slots.append(c.slots())
            s.out.append(_host_cells(len(s.slots[-1]), c.st.num_vars, c.n))
            s.at.append(_addresses(s.out[-1]))
        return s
    args = _arguments(case, seed % (1 << 31))
    s.run = M.Run(args + (" --tape" if kind == "reverse" else ""), host=host)
    s.ends.append(s.run.close)
    s.c = _Cells(host, dev, ctypes.c_void_p(s.run.h))
    if kind != "reverse":
        # the active blocks change only where the object moves
        s.slots = s.c.slots() if kind == "amr" else None
        s.cells = _host_cells(len(s.slots) if kind == "amr" else case["max_blocks"],
                              case["num_vars"], s.c.n)
        s.at = _addresses(s.cells)
        return s
    while s.run.step() == 0:
        pass
    dev.amr_dev_tape(s.c.device, 0)
    length = ctypes.c_int()
    dev.amr_dev_tape_length(s.c.device, ctypes.byref(length))
    s.length, s.uploads = length.value, []
    op = (ctypes.c_int32 * 8)()
    for i in range(s.length):
        dev.amr_dev_tape_op(s.c.device, i, op)
        if op[0] != 1:             # the uploads come first
            break
        s.uploads.append(op[1])
    s.adj = ctypes.c_void_p()
    if dev.amr_adj_create(s.c.device, ctypes.byref(s.adj)):
        raise M.AmrError(dev.amr_adj_last_error(s.adj).decode())
    s.ends.append(functools.partial(dev.amr_adj_destroy, s.adj))
    # N(0, 1) weights on the cells of the final blocks that meet the sphere
    g, r, c = torch.Generator().manual_seed(int(seed)), case["radius"], (0.5, 0.45, 0.55)
    s.slots = []
    for slot, _, lo, hi in s.run.blocks():
        near = [min(max(x, lo[d]), hi[d]) for d, x in enumerate(c)]
        if sum((near[d] - c[d]) ** 2 for d in range(3)) <= r * r:
            s.slots.append(slot)
    s.weights = _host_cells(len(s.slots), case["num_vars"], s.c.n)
    _inner(s.weights)[:] = torch.randn(_inner(s.weights).shape, generator=g, dtype=torch.float64)
    s.weights_at = _addresses(s.weights)
    s.cells = _host_cells(len(s.uploads), case["num_vars"], s.c.n)
    s.at = _addresses(s.cells)
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "grid":
        d, last = s.dev, case["stages"] - 1
        nv = case["num_vars"]
        for stage in range(last):
            d.stage_fused(0, nv, stage, sum_row=-1 if stage % CHECKSUM_FREQ
                          else stage // CHECKSUM_FREQ)
        d.stage(0, nv, last, sum_row=-1 if last % CHECKSUM_FREQ else last // CHECKSUM_FREQ)
        for slot, at in enumerate(s.at):
            d._check(d.lib.amr_dev_download_block(d.h, slot, at), "download")
        return {"cells": _inner(s.cells), "sums": d.read_sums(0, -(-case["stages"]
                                                                   // CHECKSUM_FREQ))}
    if kind == "batch":
        for _ in range(case["steps"]):
            s.batch.step()
        for m, slots, at in zip(s.members, s.slots, s.at):
            m.read(slots, at)
        return {"cells": [_inner(x) for x in s.out], "sums": [m.sums(STAGES) for m in s.members]}
    if kind in ("amr", "refine"):
        for _ in range(case["steps"]):
            s.run.step()
        slots = s.c.slots() if s.slots is None else s.slots
        s.c.read(slots, s.at)
        return {"cells": _inner(s.cells[:len(slots)]),
                "sums": s.c.sums(REFINE_STAGES if kind == "refine" else STAGES)}
    lib, bad = s.c.dev, 0
    bad |= lib.amr_adj_zero(s.adj)
    for slot, at in zip(s.slots, s.weights_at):
        bad |= lib.amr_adj_set_block(s.adj, slot, at)
    bad |= lib.amr_adj_run(s.adj, len(s.uploads), s.length)
    for slot, at in zip(s.uploads, s.at):
        bad |= lib.amr_adj_get_block(s.adj, slot, at)
    if bad:
        raise M.AmrError(lib.amr_adj_last_error(s.adj).decode())
    return {"gradient": _inner(s.cells)}


@functools.lru_cache(maxsize=None)
def _block_stages(args, steps):
    """(sum over the stages of one pass of the active blocks, active blocks at
    its end) of a driver command line, from the driver itself."""
    r = M.Run(args)
    for _ in range(steps):
        r.step()
    st = r.stats()
    r.close()
    return int(st.block_stages), int(st.active_blocks)


def work(case):
    """Every stage reads and writes each cell of each variable once and does
    the stencil's additions and division; the cells that come back are read
    once and written as 64-bit values."""
    kind, eb = case["kind"], BYTES[case["precision"]]
    flops = {7: 7, 27: 27, 0: 20}
    if kind == "batch":
        b = f = 0.0
        for t in _batch_lines(case["runs"], case["pick"]):
            t = list(t)
            n, v = int(t[t.index("--nx") + 1]), int(t[t.index("--num_vars") + 1])
            for x, y in (("--nx", "2"), ("--ny", "2"), ("--nz", "2"), ("--num_vars", "1")):
                t[t.index(x) + 1] = y
            bs, blocks = _block_stages(" ".join(t) + " --report_perf 0", case["steps"])
            b += n ** 3 * v * (2.0 * eb * bs + (eb + 8.0) * blocks)
            f += n ** 3 * v * 27.0 * bs
        return {"bytes": b, "flops": f}
    cells = case["nx"] * case["ny"] * case["nz"] * case["num_vars"]
    if kind == "grid":
        blocks = case["bx"] * case["by"] * case["bz"]
        bs = blocks * case["stages"]
    else:
        bs, blocks = _block_stages(_arguments(case, 1, tiny=True), case["steps"])
        if kind == "reverse":      # weights in, gradient of the initial blocks out
            blocks = case["init"] ** 3
    return {"bytes": cells * (2.0 * eb * bs + (eb + 8.0) * blocks),
            "flops": cells * float(flops[case["stencil"]]) * bs}


def exact(case, seed):
    """Uniform grids: the same cells and checksums from torch in 64 bits, the
    whole domain as one array with reflecting ends.  The driver's meshes and
    initial values are its own: no other code here gives them."""
    if case["kind"] != "grid":
        return None
    bx, by, bz = case["bx"], case["by"], case["bz"]
    nx, ny, nz, nv = case["nx"], case["ny"], case["nz"], case["num_vars"]
    u = _inner(_grid_values(case, seed)).cuda()
    u = u.reshape(bz, by, bx, nv, nx, ny, nz).permute(3, 2, 4, 1, 5, 0, 6)
    u = u.reshape(nv, bx * nx, by * ny, bz * nz)
    if case["precision"] != "f64":    # the values as the blocks hold them
        u = u.to(torch.float32 if case["precision"] == "f32" else torch.bfloat16).double()
    sums = []
    for stage in range(case["stages"]):
        p = torch.nn.functional.pad(u[None], (1, 1, 1, 1, 1, 1), mode="replicate")[0]
        if case["stencil"] == 27:
            for d in (1, 2, 3):
                k = p.shape[d] - 2
                p = p.narrow(d, 0, k) + p.narrow(d, 1, k) + p.narrow(d, 2, k)
            u = p / 27.0
        else:
            c = p[:, 1:-1, 1:-1, 1:-1]
            u = (c + p[:, :-2, 1:-1, 1:-1] + p[:, 2:, 1:-1, 1:-1] + p[:, 1:-1, :-2, 1:-1] +
                 p[:, 1:-1, 2:, 1:-1] + p[:, 1:-1, 1:-1, :-2] + p[:, 1:-1, 1:-1, 2:]) / 7.0
        if stage % CHECKSUM_FREQ == 0:
            sums.append(u.sum(dim=(1, 2, 3)))
    u = u.reshape(nv, bx, nx, by, ny, bz, nz).permute(5, 3, 1, 0, 2, 4, 6)
    return {"cells": u.reshape(bx * by * bz, nv, nx, ny, nz).cpu(),
            "sums": torch.stack(sums).cpu().numpy()}
