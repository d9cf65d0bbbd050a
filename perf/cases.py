"""Performance cases of the CK-MPM engine: what a program has it do, over the sizes, materials
and drivers that it has.

Four families, by the field "kind":

* ``scene``   one engine: "path" plain (``Substep`` calls), frame (``Simulate``, the frame loop
              with its dt rules) or graph (``MPMBatch`` of one engine, replayed hipGraphs);
              a pass is some substeps and the export of the positions, and of the whole
              particle state where "state" is set (a checkpoint).
* ``batch``   many engines advanced together as fused launches, then their positions.
* ``grad``    ``autodiff.simulate`` forward and backward: final positions and the gradients
              of log E and v0, all in input order.
* ``hash``    the sparse block table: build and find ("form" lds, cooperative or scalar) or
              the build into the caller's memory ("form" noalloc), on device arrays.

Bodies are boxes of cells at 8 particles per cell with jitter (columns with 4 to 16 per cell
for "mixed"), with a smooth initial strain given through ``import_state``.  The order in
which particles come back follows when they cross the faces of the 4^3-cell blocks.  Small
scenes move fast and cross them; in large ones and batches, where FP32 rounding would decide
a crossing somewhere in nearly every pass, bodies start almost at rest with no particle
within 0.1 cells of a face.
"""
import ctypes
import math
import random

import numpy as np
import torch

from ckmpm_amd import autodiff, native, scenes
from ckmpm_amd.engine import MPMBatch, engine_from_scene
from ckmpm_amd.hashtable import BlockHashTable, build_noalloc, table_sizes

RHO = 1000.0
KINDS = {"fc": scenes.FIXED_COROTATED, "nh": scenes.NEO_HOOKEAN, "dp": scenes.DRUCKER_PRAGER,
         "fluid": scenes.FLUID, "vm": scenes.VON_MISES, "cc": scenes.CAM_CLAY}
YOUNG = {"fc": (1e4, 0.3), "nh": (5e4, 0.4), "dp": (3.5e5, 0.3), "vm": (2e5, 0.3), "cc": (2e5, 0.3)}
# initial strain amplitude: soft solids in contact strain by percents, sand and metal by tenths
# of a percent (past their yield surfaces), a consolidated clay too (inside its own, whose
# hardening variable jumps at the surface), a weakly compressible fluid by less
STRAIN = {"fc": 0.04, "nh": 0.02, "dp": 2e-3, "vm": 1e-3, "cc": 1e-3, "fluid": 1e-3}
ATTRS = {"fc": 12, "nh": 12, "dp": 13, "fluid": 4, "vm": 12, "cc": 13}
DT = {32: 1e-4, 64: 1e-4, 128: 1e-4, 256: 5e-5, 512: 2e-5}


def listed():
    return [
        # two small elastic bodies, plain calls: the engine's launch latency
        {"name": "two_elastic_15k", "kind": "scene", "materials": "fc,fc", "cells": "12x13x12", "grid": 64,
         "path": "plain", "substeps": 20, "state": True, "walls": "sticky"},
        # the frame loop with its CFL rule and a host decision per substep, one frame out
        {"name": "frame_jelly_64k", "kind": "scene", "materials": "nh", "cells": "20x20x20", "grid": 128,
         "path": "frame", "substeps": 10, "state": True, "walls": "sticky"},
        # ragged fluid and sand against slip walls (the boundary hook), plain calls
        {"name": "fluid_sand_slip_ragged", "kind": "scene", "materials": "fluid,dp", "cells": "19x23x21", "grid": 64,
         "path": "plain", "substeps": 16, "state": True, "walls": "slip"},
        # metal yielding and stiff clay, checkpointed state
        {"name": "plastic_250k", "kind": "scene", "materials": "vm,cc", "cells": "25x25x25", "grid": 128,
         "path": "graph", "substeps": 32, "state": True, "walls": "sticky"},
        # a soft elastic block of mid size
        {"name": "elastic_330k", "kind": "scene", "materials": "fc", "cells": "37x33x34", "grid": 128,
         "path": "graph", "substeps": 32, "state": True, "walls": "sticky"},
        # one jelly of a million particles
        {"name": "jelly_1m", "kind": "scene", "materials": "nh", "cells": "50x50x50", "grid": 256,
         "path": "graph", "substeps": 40, "state": True, "walls": "sticky"},
        # the benchmark's scene type and size: fluid column and sand heap, uneven cells
        {"name": "dam_sand_8m", "kind": "scene", "materials": "mixed", "fluid": 5_000_000, "sand": 3_000_000,
         "grid": 512, "path": "graph", "substeps": 40, "state": False, "walls": "sticky"},
        # many independent scenes of mixed materials and sizes
        {"name": "batch_64", "kind": "batch", "scenes": 64, "lo": 8_000, "hi": 120_000, "substeps": 20},
        # gradient loop of the cantilever, checkpoints every 25 substeps
        {"name": "gradient_104k", "kind": "grad", "material": "fc", "cells": "77x13x13", "grid": 128, "substeps": 50,
         "segment": 25},
        # a small gradient with the whole tape kept
        {"name": "gradient_9k_tape", "kind": "grad", "material": "nh", "cells": "23x7x7", "grid": 64, "substeps": 24,
         "segment": 0},
        # the block table over a large scene's block list: rebuild, then the 27 neighbours of each
        {"name": "table_25k", "kind": "hash", "keys": 25_090, "per_key": 27, "side": 128, "form": "lds"},
        # a larger table into the caller's memory
        {"name": "table_200k_noalloc", "kind": "hash", "keys": 200_003, "per_key": 0, "side": 256, "form": "noalloc"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["scene", "scene", "scene", "scene", "mixed", "batch", "grad", "hash"])
    if kind == "mixed":
        g = rng.choice([128, 256, 512])
        total = _log(rng, {128: 6e4, 256: 4e5, 512: 2e6}[g], {128: 4e5, 256: 2e6, 512: 7e6}[g])
        part = rng.uniform(0.3, 0.7)
        return {"kind": "scene", "materials": "mixed", "fluid": int(total * part), "sand": int(total * (1 - part)),
                "grid": g, "path": "graph", "substeps": rng.randrange(12, 41), "state": False, "walls": "sticky"}
    if kind == "scene":
        g = rng.choice([64, 128, 256])
        mats = rng.choice(["fc", "nh", "dp", "fluid", "vm", "cc", "fc,fc", "fluid,dp", "vm,cc", "nh,fluid"])
        side = _log(rng, 9, {64: 21, 128: 38, 256: 50}[g])
        cells = "x".join(str(max(7, round(side * rng.uniform(0.8, 1.2)))) for _ in range(3))
        path = rng.choice(["plain", "plain", "graph", "graph", "frame"])
        return {"kind": "scene", "materials": mats, "cells": cells, "grid": g, "path": path,
                "substeps": rng.randrange(8, 33), "state": rng.random() < 0.7,
                "walls": rng.choice(["sticky", "sticky", "slip"])}
    if kind == "batch":
        lo = _log(rng, 4e3, 2e4)
        return {"kind": "batch", "scenes": rng.randrange(3, 65), "lo": int(lo), "hi": int(lo * _log(rng, 2, 6)),
                "substeps": rng.randrange(6, 21)}
    if kind == "grad":
        g = rng.choice([64, 128])
        k = {64: 1.0, 128: 1.7}[g]
        steps = rng.randrange(11, 45)
        return {"kind": "grad", "material": rng.choice(["fc", "nh"]),
                "cells": "%dx%dx%d" % (rng.randrange(12, int(36 * k)), rng.randrange(5, int(8 * k)), rng.randrange(5, int(8 * k))),
                "grid": g, "substeps": steps, "segment": rng.choice([0, 10, 25])}
    form = rng.choice(["lds", "cooperative", "scalar", "noalloc"])
    keys = int(_log(rng, 300, 28_000 if form == "lds" else 250_000))
    return {"kind": "hash", "keys": keys, "per_key": 0 if form == "noalloc" else rng.choice([1, 8, 27]),
            "side": rng.choice([128, 200, 256]), "form": form}


# ------------------------------------------------------------------ bodies
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _cells(lo, ext):
    r = [torch.arange(a, a + e, device="cuda") for a, e in zip(lo, ext)]
    return torch.stack(torch.meshgrid(*r, indexing="ij"), -1).reshape(-1, 3).float()


def _box(gen, lo, ext, dx):
    """8 particles per cell on stratified sub-cells with jitter; a few dropped so that the
    count is odd."""
    cells = _cells(lo, ext)
    sub = _cells((0, 0, 0), (2, 2, 2)) * 0.5
    x = (cells[:, None] + sub[None] + 0.5 * _rand(gen, cells.shape[0], 8, 3)).reshape(-1, 3) * dx
    return x[: x.shape[0] - 3]


def _column(gen, lo, ext_x, ext_z, n, dx):
    """n particles at log-uniform 4 to 16 per cell, bottom layer first."""
    rows = int(math.ceil(n / (8.2 * ext_x * ext_z))) + 2
    c = _cells((lo[1], lo[0], lo[2]), (rows, ext_x, ext_z))[:, [1, 0, 2]]
    cnt = torch.exp(math.log(4.0) + _rand(gen, c.shape[0]) * math.log(4.0)).round().long()
    at = torch.repeat_interleave(torch.arange(c.shape[0], device="cuda"), cnt)[:n]
    return (c[at] + _rand(gen, at.shape[0], 3)) * dx


def _off_faces(x, dx, m=0.1):
    """Particles closer than m cells to a block face (cell 4 k + 1.75, by the binning rule)
    move m cells away from it."""
    d = torch.remainder(x / dx - 1.75 + 2.0, 4.0) - 2.0
    return x + torch.where(d.abs() < m, torch.where(d < 0, -m * dx, m * dx), 0.0)


class _Body:
    """One model's inputs: material name, FP32 positions and velocities, a smooth strain."""

    def __init__(self, mat, x, gen, dx, speed=0.02):
        self.mat, self.dx = mat, dx
        self.x = (x if speed > 0.1 else _off_faces(x, dx)).contiguous()
        self.wave = (_rand(gen, 9, 3) - 0.5).double() * 60.0
        self.phase = _rand(gen, 9).double() * 6.28
        vw, vp = (_rand(gen, 3, 3) - 0.5).double() * 30.0, _rand(gen, 3).double() * 6.28
        self.v = (speed * torch.sin(self.x.double() @ vw.T + vp)).float().contiguous()

    def strain(self, x):
        """E = F - I (n, 9) in FP32 at the FP32 positions x; for a fluid J - 1 (n,)."""
        a = STRAIN[self.mat]
        s = a * torch.sin(x.double() @ self.wave.T + self.phase)
        s[:, [0, 4, 8]] -= 0.5 * a
        return (s[:, 0] if self.mat == "fluid" else s).float()


def _material(mat):
    if mat == "fluid":
        return scenes.Material(scenes.FLUID, bulk=1e5, gamma=7.0, viscosity=0.1, J0=1.0)
    lam, mu = scenes.lame(*YOUNG[mat])
    if mat == "vm":
        return scenes.Material(scenes.VON_MISES, lam, mu, yield_stress=30.0)
    if mat == "cc":
        return scenes.Material(scenes.CAM_CLAY, lam, mu, alpha0=-0.02, beta=0.5, hardening_factor=0.8, m=2.36)
    return scenes.Material(KINDS[mat], lam, mu)


def _bodies(case, seed):
    gen, g = _generator(seed), case["grid"]
    dx = 1.0 / g
    y0 = 5 if case.get("walls") == "slip" else 10
    if case["materials"] == "mixed":
        y0 = max(9, int(0.035 * g))
        xf = _column(gen, (int(0.0625 * g), y0, int(0.45 * g)), g // 4, g // 10, case["fluid"], dx)
        w = int(0.22 * g)
        xs = _column(gen, (int(0.58 * g), y0, (g - w) // 2), w, w, case["sand"], dx)
        return [_Body("fluid", xf, gen, dx, 0.0), _Body("dp", xs, gen, dx, 0.0)]
    mats = case["materials"].split(",")
    ext = [int(e) for e in case["cells"].split("x")]
    width = ext[0] * len(mats) + 2 * (len(mats) - 1)
    small = 8 * math.prod(ext) * len(mats) < 40_000 and case.get("path") is not None  # one small scene
    speed = 0.3 if small else 0.02
    out = []
    for i, m in enumerate(mats):
        lo = ((g - width) // 2 + i * (ext[0] + 2), y0, (g - ext[2]) // 2)
        out.append(_Body(m, _box(gen, lo, ext, dx), gen, dx, speed))
    return out


def _boundary(case):
    if case.get("walls") != "slip":
        return None
    return scenes.Boundary(scenes.WALLS_SLIP, [scenes.Region((0, 0, 0), (case["grid"], 6, case["grid"]), scenes.REGION_FIXED)])


def _engine(bodies, grid, boundary=None, fps=None):
    dx = 1.0 / grid
    vol = dx ** 3 / 8
    models = [scenes.ModelSpec(_material(b.mat), RHO * vol, vol, b.x.cpu().numpy(), b.v.cpu().numpy()) for b in bodies]
    sc = scenes.Scene("case", (grid // 4,) * 3, (0, 0, 0), dx, -9.8, DT[grid], 0, models, boundary=boundary)
    # the frame loop's rate and CFL number as the scene's program sets them
    eng = engine_from_scene(sc, fps=fps, cfl=0.5 if fps else None)
    for i, b in enumerate(bodies):
        st = eng.state(i)
        e = b.strain(torch.from_numpy(eng.positions(i)).cuda()).cpu().numpy()
        if b.mat == "fluid":
            st[3] = e
        else:
            st[3:12] = e.T
        eng.set_state(i, st)
    return eng


def _fps(case):
    """Frames of about "substeps" substeps of the default dt."""
    return int(round(1.0 / (DT[case["grid"]] * case["substeps"])))


def _pinned(*shape):
    return torch.empty(*shape, dtype=torch.float32, pin_memory=True)


def _floats(buf):
    return ctypes.cast(buf.data_ptr(), ctypes.POINTER(ctypes.c_float))


def _positions_into(eng, model, buf):
    """ckmpm_get_positions into a buffer that the program keeps."""
    n = ctypes.c_uint64()
    rc = native.load().ckmpm_get_positions(eng._h, model, _floats(buf), buf.shape[0], ctypes.byref(n))
    if rc != native.OK:
        raise RuntimeError("ckmpm_get_positions: %d" % rc)
    return buf


def _state_into(eng, model, buf):
    """ckmpm_export_state into a buffer that the program keeps."""
    rc = native.load().ckmpm_export_state(eng._h, model, _floats(buf))
    if rc != native.OK:
        raise RuntimeError("ckmpm_export_state: %d" % rc)
    return buf


def _batch_cases(case):
    """The scenes of a batch: a grid, a material and a box each, sizes spread over their logarithm."""
    r = random.Random(case["scenes"] * 1_000_003 + case["lo"])
    out = []
    for i in range(case["scenes"]):
        g = r.choice([64, 128])
        side = min((_log(r, case["lo"], case["hi"]) / 8) ** (1 / 3), 0.5 * g)
        out.append({"materials": ["fc", "nh", "dp", "fluid"][i % 4], "grid": g,
                    "cells": "x".join(str(max(6, round(side * r.uniform(0.8, 1.2)))) for _ in range(3))})
    return out


def _bar(case, seed):
    """The clamped bar of the gradient cases: positions of the scene, inputs of the seed."""
    g = case["grid"]
    dx = 1.0 / g
    ext = [int(e) for e in case["cells"].split("x")]
    lo = (max(2, int(0.03 * g)), (g - ext[1]) // 2, (g - ext[2]) // 2)
    x = _box(_generator(12345), lo, ext, dx)
    n, gen = x.shape[0], _generator(seed)
    nu = 0.3
    log_e = math.log(1e4) + 0.3 * torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
    v0 = 0.05 * torch.randn(n, 3, generator=gen, device="cuda", dtype=torch.float64)
    gx = torch.randn(n, 3, generator=gen, device="cuda", dtype=torch.float64) / n
    return x, log_e, v0, gx, nu


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "scene":
        bodies = _bodies(case, seed)
        eng = _engine(bodies, case["grid"], _boundary(case), _fps(case) if case["path"] == "frame" else None)
        dt = DT[case["grid"]]
        st = {"kind": kind, "path": case["path"], "eng": eng, "dt": dt, "substeps": case["substeps"],
              "state": case["state"], "models": len(bodies)}
        if case["path"] == "plain":
            eng.Substep(0.0, dt)  # the reference's first iteration has dt = 0
        if case["path"] == "graph":
            st["batch"] = MPMBatch([eng])
            st["batch"].Run(1)
            st["out"] = [_pinned(b.x.shape[0], 3) for b in bodies]
            st["out_state"] = [_pinned(ATTRS[b.mat], b.x.shape[0]) if case["state"] else None for b in bodies]
        return st
    if kind == "batch":
        engs, outs = [], []
        for i, c in enumerate(_batch_cases(case)):
            b = _bodies(c, seed * 1009 + i)
            engs.append(_engine(b, c["grid"]))
            outs.append(b[0].x.shape[0])
        batch = MPMBatch(engs)
        batch.Run(1)
        buf = _pinned(sum(outs), 3)
        return {"kind": kind, "batch": batch, "engs": engs, "substeps": case["substeps"], "buf": buf,
                "parts": list(torch.split(buf, outs))}
    if kind == "grad":
        x, log_e, v0, gx, nu = _bar(case, seed)
        dx = 1.0 / case["grid"]
        lam, mu = scenes.lame(1e4, nu)
        vol = dx ** 3 / 8
        m = scenes.ModelSpec(scenes.Material(KINDS[case["material"]], lam, mu), RHO * vol, vol, x.cpu().numpy(),
                             np.zeros((x.shape[0], 3), np.float32))
        sc = scenes.Scene("bar", (case["grid"] // 4,) * 3, (0, 0, 0), dx, -9.8, DT[case["grid"]], case["substeps"], [m])
        return {"kind": kind, "log_e": log_e.requires_grad_(), "v0": v0.requires_grad_(), "gx": gx, "scene": sc, "nu": nu,
                "substeps": case["substeps"], "segment": case["segment"] or None}
    gen, n, side = _generator(seed), case["keys"], case["side"]
    keys = torch.randperm(side ** 3, generator=gen, device="cuda")[:n].to(torch.int32)
    vals = torch.arange(n, device="cuda", dtype=torch.int32)
    st = {"kind": kind, "form": case["form"], "dim": (side,) * 3, "n": n, "keys": keys, "vals": vals}
    if case["form"] == "noalloc":
        slots, stash = table_sizes(n)
        st["slots"] = torch.zeros(slots, dtype=torch.int64, device="cuda")
        st["stash"] = torch.zeros(stash, dtype=torch.int64, device="cuda")
        st["nstash"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    else:
        # neighbours of the listed blocks: about as many present as absent keys
        off = torch.tensor([(i * side + j) * side + k for i in (-1, 0, 1) for j in (-1, 0, 1) for k in (-1, 0, 1)],
                           device="cuda", dtype=torch.int32)[:: 27 // case["per_key"]][: case["per_key"]]
        st["queries"] = ((keys[:, None] + off[None]).reshape(-1) % side ** 3).contiguous()
        st["found"] = torch.empty_like(st["queries"])
        st["table"] = BlockHashTable(st["dim"], n)
    torch.cuda.synchronize()
    return st


def run(st):
    kind = st["kind"]
    if kind == "scene":
        eng = st["eng"]
        if st["path"] == "plain":
            for _ in range(st["substeps"]):
                eng.Substep(st["dt"], st["dt"])
        elif st["path"] == "frame":
            eng.Simulate(1)
        else:
            st["batch"].Run(st["substeps"])
        out = {}
        for i in range(st["models"]):
            out["x%d" % i] = _positions_into(eng, i, st["out"][i]) if "out" in st else eng.positions(i)
            if st["state"]:
                out["state%d" % i] = _state_into(eng, i, st["out_state"][i]) if "out" in st else eng.state(i)
        return out
    if kind == "batch":
        st["batch"].Run(st["substeps"])
        for eng, part in zip(st["engs"], st["parts"]):
            _positions_into(eng, 0, part)
        return st["buf"]
    if kind == "grad":
        x = autodiff.simulate(st["log_e"], st["v0"], st["scene"], st["substeps"], segment=st["segment"], nu=st["nu"])
        g_e, g_v = torch.autograd.grad(x, (st["log_e"], st["v0"]), st["gx"])
        # the library computes in FP32
        return {"x": x.detach().float(), "log_e_bar": g_e.float(), "v0_bar": g_v.float()}
    if st["form"] == "noalloc":
        rc = build_noalloc(st["dim"], st["n"], st["keys"].data_ptr(), st["vals"].data_ptr(), st["n"],
                           st["slots"].data_ptr(), st["stash"].data_ptr(), st["nstash"].data_ptr())
        if rc != native.OK:
            raise RuntimeError("build_noalloc: %d" % rc)
        return {"slots": st["slots"], "stash": st["stash"], "nstash": st["nstash"]}
    t, q = st["table"], st["queries"]
    t.InsertDevice(st["keys"].data_ptr(), st["vals"].data_ptr(), st["n"])
    form = {"lds": t.LDS, "cooperative": t.COOPERATIVE, "scalar": t.SCALAR}[st["form"]]
    t.FindDevice(q.data_ptr(), q.numel(), st["found"].data_ptr(), form)
    t.Synchronize()
    return st["found"]


# ------------------------------------------------------------------ work
def _particles(case):
    """(material, particles, grid blocks) of each body of a scene."""
    if case["materials"] == "mixed":
        return [(m, n, (n / 8.66 / 64) * 1.5) for m, n in (("fluid", case["fluid"]), ("dp", case["sand"]))]
    ext = [int(e) for e in case["cells"].split("x")]
    blocks = math.prod(e / 4 + 2 for e in ext)
    return [(m, 8 * math.prod(ext) - 3, blocks) for m in case["materials"].split(",")]


def work(case):
    # a substep: each particle's state read and written and its order kept (12 bytes), each
    # grid block's mass, momentum (2048 bytes, deposited, read and cleared) and velocity
    # (1536 bytes, written) once; flops: two stencils, G2P and P2G over 16 nodes, 3x3
    # algebra, the stress
    def substep(parts):
        b = sum(n * (2 * 4 * ATTRS[m] + 12) + blocks * 7168 for m, n, blocks in parts)
        f = sum(n * (1300 if m == "fluid" else 1500 if m == "nh" else 1900) for m, n, _ in parts)
        return b, f

    kind = case["kind"]
    if kind == "scene":
        parts = _particles(case)
        b, f = substep(parts)
        steps = case["substeps"]
        out = sum(n * (12 + (4 * ATTRS[m] if case["state"] else 0)) for m, n, _ in parts)
        return {"bytes": steps * b + out, "flops": steps * f}
    if kind == "batch":
        parts = [p for c in _batch_cases(case) for p in _particles(c)]
        b, f = substep(parts)
        return {"bytes": case["substeps"] * b + sum(12 * n for _, n, _ in parts), "flops": case["substeps"] * f}
    if kind == "grad":
        parts = _particles({"materials": case["material"], "cells": case["cells"]})
        b, f = substep(parts)
        n = parts[0][1]
        # forward, and a backward that reads state and adjoints and writes adjoints; about
        # three times the forward's arithmetic (recompute and transpose)
        return {"bytes": case["substeps"] * (3 * b) + n * 4 * 13, "flops": case["substeps"] * 4 * f}
    n, q = case["keys"], case["keys"] * case["per_key"]
    buckets = -(-n * 10 // 112)
    return {"bytes": 8 * n + 128 * buckets + 8 * q, "flops": 0}


# ------------------------------------------------------------------ exact
# The same substep in FP64 torch, from the published method: two staggered grids, compact
# kernel w0 = 1 - t + sin(2 pi t) / (2 pi), APIC with the closed-form moment matrix, and
# the canonical block and particle order (whole numbers, from FP64 positions after the
# setup, whose FP32 cell rule is part of the input).
def _mm(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _t(A):
    return A.transpose(1, 2)


def _det(A):
    return (A[:, 0] * torch.linalg.cross(A[:, 1], A[:, 2])).sum(1)


def _inv(A):
    r0, r1, r2 = A[:, 0], A[:, 1], A[:, 2]
    adj = torch.stack([torch.linalg.cross(r1, r2), torch.linalg.cross(r2, r0), torch.linalg.cross(r0, r1)], 2)
    return adj / (r0 * adj[:, :, 0]).sum(1)[:, None, None]


def _stencil(x, dx, g):
    shift = 0.25 if g == 0 else -0.25
    xs = x / dx
    c = torch.floor(xs.detach() + shift)
    t = xs - c + shift
    w0 = 1.0 - t + torch.sin(2 * math.pi * t) / (2 * math.pi)
    return c.long(), t, torch.stack([w0, 1.0 - w0], 0)  # w[o][n, axis]


def _moment(x, dx):
    """The moment matrix of the compact kernel over both grids, in units of dx^2: second
    moments on the diagonal, products of first moments off it."""
    D = 0
    for g in (0, 1):
        _, t, w = _stencil(x, dx, g)
        m1 = w[1] - t
        diag = w[0] * t * t + w[1] * (1 - t) ** 2
        off = m1[:, :, None] * m1[:, None, :]
        eye = torch.eye(3, device=x.device, dtype=torch.bool)
        D = D + torch.where(eye, torch.diag_embed(diag), off)
    return D


class _Grid:
    """Nodes of both sub-grids in the cells' bounding box."""

    def __init__(self, xs, dx):
        allx = torch.cat([x.detach() for x in xs])
        self.lo = torch.floor(allx.min(0).values / dx).long() - 3
        self.size = torch.floor(allx.max(0).values / dx).long() + 5 - self.lo
        self.n = int(self.size.prod())

    def index(self, c, o, g):
        q = c + torch.tensor(o, device=c.device) - self.lo
        return ((q[:, 0] * self.size[1] + q[:, 1]) * self.size[2] + q[:, 2]) + g * self.n

    def cells(self):
        r = [torch.arange(int(s), device=self.lo.device) + l for s, l in zip(self.size, self.lo)]
        c = torch.stack(torch.meshgrid(*r, indexing="ij"), -1).reshape(-1, 3)
        return torch.cat([c, c])


_OFFS = [(i, j, k) for i in (0, 1) for j in (0, 1) for k in (0, 1)]


def _weight(w, o):
    return w[o[0]][:, 0] * w[o[1]][:, 1] * w[o[2]][:, 2]


def _p2g(grid, M, x, dx, mass, mom, K):
    """Adds w m and w (m v + K (x_i - x_p)) of one model to M (2 n, 4)."""
    for g in (0, 1):
        c, t, w = _stencil(x, dx, g)
        for o in _OFFS:
            d = (torch.tensor(o, device=x.device) - t) * dx
            p = mom if K is None else mom + (K * d[:, None, :]).sum(-1)
            wi = _weight(w, o)[:, None]
            M = M.index_add(0, grid.index(c, o, g), torch.cat([wi * mass, wi * p], 1))
    return M


def _g2p(grid, V, x, dx):
    v = 0
    B = 0
    for g in (0, 1):
        c, t, w = _stencil(x, dx, g)
        for o in _OFFS:
            wv = _weight(w, o)[:, None] * V[grid.index(c, o, g)]
            v = v + 0.5 * wv
            B = B + wv[:, :, None] * (torch.tensor(o, device=x.device) - t)[:, None, :]
    return v, _mm(B, _inv(_moment(x, dx))) / dx


def _grid_velocity(grid, M, dt, gravity, dim, slip):
    m = M[:, :1]
    on = m > 0
    v = torch.where(on, M[:, 1:] / torch.where(on, m, torch.ones_like(m)), torch.zeros_like(M[:, 1:]))
    v = v + torch.where(on, 1.0, 0.0) * torch.tensor([0.0, gravity * dt, 0.0], device=M.device, dtype=M.dtype)
    c = grid.cells()
    if not slip:
        b = c >> 2
        stuck = ((b < 2) | (b + 2 >= dim)).any(1, keepdim=True)
        return torch.where(stuck, torch.zeros_like(v), v)
    n = (c < 8).double() - (c >= 4 * dim - 8).double()
    n = n / n.norm(dim=1, keepdim=True).clamp_min(1e-30)
    v = v - (v * n).sum(1, keepdim=True) * n
    return torch.where((c[:, 1:2] < 6) & (c[:, 1:2] >= 0), torch.zeros_like(v), v)


def _eigen(S):
    """Cyclic Jacobi of symmetric 3x3 matrices: eigenvalues (n, 3), eigenvectors in columns."""
    S = S.clone()
    Q = torch.eye(3, device=S.device, dtype=S.dtype).expand_as(S).clone()
    for _ in range(7):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            b, dm = S[:, p, q], S[:, q, q] - S[:, p, p]
            den = dm.abs() + torch.sqrt(dm * dm + 4 * b * b)
            t = torch.where(den > 0, 2 * b * torch.where(dm >= 0, 1.0, -1.0) / den.clamp_min(1e-300), torch.zeros_like(b))
            c = 1 / torch.sqrt(1 + t * t)
            s = t * c
            R = torch.zeros_like(S)
            R[:, p, p], R[:, q, q], R[:, p, q], R[:, q, p] = c, c, s, -s
            R[:, 3 - p - q, 3 - p - q] = 1
            S = _mm(_t(R), _mm(S, R))
            Q = _mm(Q, R)
    return torch.diagonal(S, dim1=1, dim2=2), Q


def _principal(F):
    """Principal stretches - 1 and directions of F = (stretch) (rotation)."""
    E = F - torch.eye(3, device=F.device, dtype=F.dtype)
    m, U = _eigen(E + _t(E) + _mm(E, _t(E)))
    return m / (1 + torch.sqrt(1 + m)), U


def _sym(U, k):
    return _mm(U * k[:, None, :], _t(U))


def _stress(mat, F, hard, lam, mu, mp):
    """(F, hardening variable, Kirchhoff stress) after the return map."""
    eye = torch.eye(3, device=F.device, dtype=F.dtype)
    if mat == "nh":
        lnJ = torch.log(_det(F))
        return F, hard, mu * (_mm(F, _t(F)) - eye) + (lam * lnJ)[:, None, None] * eye
    d, U = _principal(F)
    s = 1 + d
    J = s.prod(1)
    if mat == "fc":
        return F, hard, _sym(U, 2 * mu * s * d + (lam * J * (J - 1))[:, None])
    stretch = lambda ns: _mm(_sym(U, ns / s), F)  # noqa: E731  (F with singular values ns)
    if mat in ("dp", "vm"):
        eps = torch.log1p(d)
        tr = eps.sum(1)
        if mat == "vm":
            dev = eps - tr[:, None] / 3
            nrm = dev.norm(dim=1)
            over = nrm - mp.yield_stress / (2 * mu)
            H = torch.where((over > 0)[:, None], eps - (over / nrm)[:, None] * dev, eps)
            F = torch.where((over > 0)[:, None, None], stretch(torch.exp(H)), F)
        else:
            sphi = math.sin(math.radians(mp.friction_deg))
            alpha = math.sqrt(2 / 3) * 2 * sphi / (3 - sphi)
            trt = tr + hard
            dev = eps - trt[:, None] / 3
            nrm = dev.norm(dim=1)
            dg = nrm + (3 * lam + 2 * mu) / (2 * mu) * trt * alpha
            opened = trt >= 0
            H = torch.where((dg > 0)[:, None], eps - (dg / nrm)[:, None] * dev, eps)
            H = torch.where(opened[:, None], torch.zeros_like(H), H)
            hard = torch.where(opened, trt, torch.zeros_like(trt))
            F = torch.where((opened | (dg > 0))[:, None, None], stretch(torch.exp(H)), F)
        return F, hard, _sym(U, 2 * mu * H + (lam * H.sum(1))[:, None])
    # non-associated Cam-clay
    kappa, beta, msq = 2 * mu / 3 + lam, mp.beta, mp.m ** 2
    p0 = kappa * (1e-5 + torch.sinh(mp.hardening_factor * (-hard).clamp_min(0)))
    pmin = -beta * p0
    b2 = s * s
    mean = b2.mean(1)
    devf = mu * J ** (-2 / 3)
    sh = devf[:, None] * (b2 - mean[:, None])
    p = -0.5 * kappa * (J * J - 1)
    ysh = 1.5 * (1 + 2 * beta)
    yph = msq * (p - pmin) * (p - p0)
    sn2 = (sh * sh).sum(1)
    cap = (p > p0) | (p < pmin)
    shear = ~cap & (ysh * sn2 + yph >= 1e-4)
    pc = torch.where(p > p0, p0, pmin)
    jc = torch.sqrt(1 - 2 * pc / kappa)
    scale = J ** (2 / 3) / mu * torch.sqrt((-yph).clamp_min(0) / ysh) / torch.sqrt(sn2).clamp_min(1e-300)
    bs = sh * scale[:, None] + mean[:, None]
    newb = torch.where(cap[:, None], (jc ** (2 / 3))[:, None].expand_as(bs), torch.where(shear[:, None], bs, b2))
    # hardening on the shear branch: the ray from the ellipse's centre through (p, q)
    ctr = 0.5 * (1 - beta) * p0
    d0, d1 = ctr - p, -torch.sqrt(1.5 * sn2)
    dn = torch.sqrt(d0 * d0 + d1 * d1).clamp_min(1e-300)
    d0, d1 = d0 / dn, d1 / dn
    A = msq * d0 * d0 + (1 + 2 * beta) * d1 * d1
    B = msq * d0 * (2 * ctr - p0 - pmin)
    C = msq * (ctr - pmin) * (ctr - p0)
    disc = torch.sqrt((B * B - 4 * A * C).clamp_min(0))
    p1, p2 = ctr + (-B + disc) / (2 * A) * d0, ctr + (-B - disc) / (2 * A) * d0
    pf = torch.where((p - ctr) * (p1 - ctr) > 0, p1, p2)
    jf = torch.sqrt((1 - 2 * pf / kappa).abs())
    band = shear & (p0 > 1e-4) & (p < p0 - 1e-4) & (p > 1e-4 + pmin) & (jf > 1e-4)
    hard = torch.where(cap, hard + torch.log(J / jc), torch.where(band, hard + 9 * torch.log(J / jf), hard))
    F = torch.where((cap | shear)[:, None, None], stretch(torch.sqrt(newb)), F)
    j2 = newb.prod(1)
    return F, hard, _sym(U, devf[:, None] * (newb - newb.mean(1)[:, None]) + (0.5 * kappa * (j2 - 1))[:, None])


def _fluid_stress(J, C, mp):
    p = mp.bulk * (J ** -mp.gamma - 1)
    eye = torch.eye(3, device=J.device, dtype=J.dtype)
    return J[:, None, None] * (mp.viscosity * (C + _t(C)) - p[:, None, None] * eye)


def _block_key(b, dim):
    return (b[:, 0] * dim[1] + b[:, 1]) * dim[2] + b[:, 2]


def _coords(k, dim):
    return torch.stack([k // (dim[1] * dim[2]), k // dim[2] % dim[1], k % dim[2]], 1)


def _extend(A, dim):
    """Particle blocks A (in list order), then the new blocks of A + {0,1}^3 and of
    A + {-1,0,1}^3, each in ascending key order."""
    out = A
    for lo in (0, -1):
        offs = torch.tensor([(i, j, k) for i in range(lo, 2) for j in range(lo, 2) for k in range(lo, 2)], device=A.device)
        q = (_coords(A, dim)[:, None] + offs[None]).reshape(-1, 3)
        q = q[((q >= 0) & (q < dim)).all(1)]
        k = torch.unique(_block_key(q, dim))
        out = torch.cat([out, k[~torch.isin(k, out)]])
    return out


class _Reference:
    """FP64 engine over the bodies, with the canonical order."""

    def __init__(self, bodies, grid, slip=False):
        self.dx, self.g = 1.0 / grid, grid
        dev = bodies[0].x.device
        self.dim = torch.full((3,), grid // 4, device=dev)
        self.slip, self.vol = slip, self.dx ** 3 / 8
        self.mass = float(np.float32(RHO * self.vol))
        self.vol = float(np.float32(self.vol))
        self.gravity = float(np.float32(-9.8))
        self.models = []
        keys = []
        for b in bodies:
            c = torch.floor(b.x * grid + 0.25).long()  # FP32, two roundings
            blk = (c - 2) >> 2
            cell = (((c - 2) & 3) * torch.tensor([16, 4, 1], device=dev)).sum(1)
            key = _block_key(blk, self.dim)
            ck = key * 64 + cell
            s, perm = torch.sort(ck, stable=True)
            head = torch.cat([torch.ones(1, dtype=torch.bool, device=dev), s[1:] != s[:-1]])
            at = torch.arange(s.shape[0], device=dev)
            rank = at - torch.cummax(torch.where(head, at, torch.zeros_like(at)), 0).values
            order = perm[torch.argsort(((s >> 6) << 38) | (rank << 6) | (s & 63), stable=True)]
            x = b.x[order]
            e = b.strain(x).double()
            mp = _material(b.mat)
            m = {"mat": b.mat, "mp": mp, "x": x.double(), "v": b.v[order].double(), "blk": key[order],
                 "lam": float(np.float32(mp.lam)), "mu": float(np.float32(mp.mu)),
                 "hard": torch.full((x.shape[0],), float(np.float32(mp.alpha0)) if b.mat == "cc" else 0.0, device=dev, dtype=torch.float64),
                 "F": 1 + e if b.mat == "fluid" else e.reshape(-1, 3, 3) + torch.eye(3, device=dev, dtype=torch.float64)}
            self.models.append(m)
            keys.append(key)
        self.blocks = _extend(torch.unique(torch.cat(keys)), self.dim)
        self.grid = _Grid([m["x"] for m in self.models], self.dx)
        M = torch.zeros(2 * self.grid.n, 4, device=dev, dtype=torch.float64)
        for m in self.models:
            M = _p2g(self.grid, M, m["x"], self.dx, self.mass, self.mass * m["v"], None)
        self.M = M

    def substep(self, dt, next_dt):
        """next_dt: a number, or a function of the grid's largest speed."""
        dt = float(np.float32(dt))
        V = _grid_velocity(self.grid, self.M, dt, self.gravity, self.dim, self.slip)
        if callable(next_dt):
            heavy = self.M[:, 0] >= math.ldexp(self.mass, -20)
            next_dt = next_dt(float(V[heavy].norm(dim=1).max()))
        nd = float(np.float32(next_dt))
        index = torch.full((int(self.dim.prod()),), -1, device=V.device, dtype=torch.long)
        index[self.blocks] = torch.arange(self.blocks.shape[0], device=V.device)
        deposits, occupied = [], []
        for m in self.models:
            v, C = _g2p(self.grid, V, m["x"], self.dx)
            m["x"] = m["x"] + dt * v
            if m["mat"] == "fluid":
                m["F"] = m["F"] * (1 + dt * torch.diagonal(C, dim1=1, dim2=2).sum(1))
                tau = _fluid_stress(m["F"], C, m["mp"])
            else:
                F = m["F"] + dt * _mm(C, m["F"])
                m["F"], m["hard"], tau = _stress(m["mat"], F, m["hard"], m["lam"], m["mu"], m["mp"])
            Dh = 2 * _inv(_moment(m["x"], self.dx)) / self.dx ** 2
            deposits.append((m["x"], self.mass * v, self.mass * C - nd * self.vol * _mm(Dh, tau)))
            m["from"] = m["blk"]
            new = (torch.floor(m["x"] / self.dx + 0.25).long() - 2) >> 2
            move = ((new - _coords(m["blk"], self.dim) + 1) * torch.tensor([9, 3, 1], device=V.device)).sum(1)
            m["new"] = _block_key(new, self.dim)
            m["order"] = torch.argsort(index[m["new"]] * 27 + move, stable=True)
            occupied.append(m["new"])
        self.grid = _Grid([d[0] for d in deposits], self.dx)
        M = torch.zeros(2 * self.grid.n, 4, device=V.device, dtype=torch.float64)
        for x, mom, K in deposits:
            M = _p2g(self.grid, M, x, self.dx, self.mass, mom, K)
        self.M = M
        keep = torch.isin(self.blocks, torch.cat(occupied))
        self.blocks = _extend(self.blocks[keep], self.dim)
        return next_dt

    def advance(self):
        """The stored state moves to the order of the next substep."""
        for m in self.models:
            if "order" in m:
                o = m.pop("order")
                for k in ("x", "F", "hard"):
                    m[k] = m[k][o]
                m["blk"] = m["new"][o]

    def outputs(self, i):
        m = self.models[i]
        u = m["x"] - 4 * _coords(m["from"], self.dim) * self.dx
        if m["mat"] == "fluid":
            st = [u, (m["F"] - 1)[:, None]]
        else:
            st = [u, (m["F"] - torch.eye(3, device=u.device, dtype=u.dtype)).reshape(-1, 9)]
            if ATTRS[m["mat"]] == 13:
                st.append(m["hard"][:, None])
        return m["x"], torch.cat(st, 1).T.contiguous()


def _run_reference(bodies, grid, steps, slip=False, fps=None):
    r = _Reference(bodies, grid, slip)
    dt = float(np.float32(DT[grid]))
    if fps is None:
        r.substep(0.0, dt)
        for _ in range(steps):
            r.advance()
            r.substep(dt, dt)
        return r
    dx = float(np.float32(1.0 / grid))
    vmax = max(float(b.v.double().norm(dim=1).max()) for b in bodies)
    top = min(dt, 1.0 / fps, dx * 0.5 / vmax if vmax else dt)
    time, cur, end = 0.0, 0.0, 1.0 / fps
    while time < end:
        r.advance()
        cur = r.substep(cur, lambda v: min(top, end - time, dx * 0.5 / v if v > 0 else top))
        time += cur
    return r


def _polar(F):
    R = F
    for _ in range(9):  # Newton: quadratic from a gradient near a rotation
        R = 0.5 * (R + _t(_inv(R)))
    return R


def _exact_grad(case, seed):
    x, log_e, v0, gx, nu = _bar(case, seed)
    g = case["grid"]
    dx = 1.0 / g
    dim = torch.full((3,), g // 4, device=x.device)
    vol = float(np.float32(dx ** 3 / 8))
    mass = float(np.float32(RHO * dx ** 3 / 8))
    log_e = log_e.clone().requires_grad_()
    v0 = v0.clone().requires_grad_()
    E = torch.exp(log_e)
    # the library takes FP32 moduli and velocities: their values, the exact derivative
    lam = E * (nu / ((1 + nu) * (1 - 2 * nu)))
    lam = lam + (lam.detach().float().double() - lam.detach())
    mu = E * (1 / (2 * (1 + nu)))
    mu = mu + (mu.detach().float().double() - mu.detach())
    v = v0 + (v0.detach().float().double() - v0.detach())
    p = x.double()
    eye = torch.eye(3, device=x.device, dtype=torch.float64)
    F = eye.expand(p.shape[0], 3, 3)
    gravity = float(np.float32(-9.8))
    grid = _Grid([p], dx)
    M = torch.zeros(2 * grid.n, 4, device=x.device, dtype=torch.float64)
    M = _p2g(grid, M, p, dx, mass, mass * v, None)
    for k in range(case["substeps"]):
        nd = float(np.float32(DT[g]))
        dt = 0.0 if k == 0 else nd
        V = _grid_velocity(grid, M, dt, gravity, dim, False)
        vp, C = _g2p(grid, V, p, dx)
        p = p + dt * vp
        F = F + dt * _mm(C, F)
        J = _det(F)[:, None, None]
        if case["material"] == "fc":
            tau = 2 * mu[:, None, None] * _mm(F - _polar(F), _t(F)) + lam[:, None, None] * J * (J - 1) * eye
        else:
            tau = mu[:, None, None] * (_mm(F, _t(F)) - eye) + lam[:, None, None] * torch.log(J) * eye
        Dh = 2 * _inv(_moment(p, dx)) / dx ** 2
        K = mass * C - nd * vol * _mm(Dh, tau)
        grid = _Grid([p], dx)
        M = torch.zeros(2 * grid.n, 4, device=x.device, dtype=torch.float64)
        M = _p2g(grid, M, p, dx, mass, mass * vp, K)
    g_e, g_v = torch.autograd.grad(p, (log_e, v0), gx.float().double())
    return {"x": p.detach(), "log_e_bar": g_e, "v0_bar": g_v}


def exact(case, seed):
    kind = case["kind"]
    if kind == "hash":
        return None  # whole numbers
    if kind == "grad":
        n = 8 * math.prod(int(e) for e in case["cells"].split("x"))
        return _exact_grad(case, seed) if n * case["substeps"] <= 6_000_000 else None
    if kind == "batch":
        parts = _batch_cases(case)
        if sum(p[1] for c in parts for p in _particles(c)) * case["substeps"] > 400_000_000:
            return None
        rs = [_run_reference(_bodies(c, seed * 1009 + i), c["grid"], case["substeps"]) for i, c in enumerate(parts)]
        return torch.cat([r.outputs(0)[0] for r in rs])
    if sum(p[1] for p in _particles(case)) * case["substeps"] > 400_000_000:
        return None  # takes too long
    r = _run_reference(_bodies(case, seed), case["grid"], case["substeps"], case["walls"] == "slip",
                       _fps(case) if case["path"] == "frame" else None)
    out = {}
    for i in range(len(r.models)):
        out["x%d" % i], st = r.outputs(i)
        if case["state"]:
            out["state%d" % i] = st
    return out
