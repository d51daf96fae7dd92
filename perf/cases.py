"""Timed workloads of the SPH / hash-grid path, each through the package's public entry points.

    step    Pipeline.step: one substep of the dam-break pipeline (sph_fused, gravity, integrate,
            box) from particles in caller order, as an interactive host drives it
    frame   Pipeline.run: the substeps of one output frame in one call
    unfused Pipeline.step of the separate density, pressure and viscosity modules with gravity,
            integrate and box (a manifest that does not name all three, or a host that reads the
            velocities between them)
    force   SphFusedModule.execute_force: the force pass over a grid and densities the host holds
    counts  HashGrid.build and HashGrid.neighbor_counts of all points
    query   HashGrid.query_neighbors_batch: neighbour lists of arbitrary points
    sort    RadixSorter.sort of (u32 key, u32 value) pairs, with find_cell_boundaries after it
            where the keys are cells

Every pass starts from the same inputs: what a call updates in place is copied back first, in one
device copy.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "forge-gpu_amd"))

import forge_hip as fh  # noqa: E402
from forge_hip.workloads import particle_mass  # noqa: E402

RHO0, GAS, MU, DT = 1000.0, 2000.0, 0.01, 1e-4
GRAVITY, RESTITUTION = (0.0, -9.81, 0.0), 0.3


def listed():
    return [
        # the smallest scene: launches and latency, not work
        {"name": "step_small", "kind": "step", "fill": "block", "n": 2197, "exact": False},
        # the 50,000-particle dam break, a frame of 10 substeps
        {"name": "frame_50k", "kind": "frame", "fill": "block", "n": 50_000, "substeps": 10},
        # the 1,048,576-particle dam break, a frame of 10 substeps
        {"name": "frame_1m", "kind": "frame", "fill": "block", "n": 1_048_576, "substeps": 10},
        # the same size after the block has burst with the manifest's mass rule: particles on the
        # walls and edges, thousands at each corner point, a sparse interior
        {"name": "step_walls_1m", "kind": "step", "fill": "walls", "n": 1_048_576,
         "exact": False},
        # skewed occupancy: Gaussian clumps, cells of up to several thousand particles, with the
        # options for dense clumps (sub-cells, 8 parts)
        {"name": "step_clumps_2m", "kind": "step", "fill": "clumps", "n": 2_097_152,
         "exact": False},
        # bit-reproducible mode of the fused module
        {"name": "step_exact_260k", "kind": "step", "fill": "block", "n": 262_144, "exact": True},
        # separate modules, an odd size
        {"name": "unfused_150k", "kind": "unfused", "fill": "block", "n": 150_001},
        {"name": "force_400k", "kind": "force", "fill": "block", "n": 400_000},
        # grid build and neighbour counts of 4,194,304 uniform points, ~30 neighbours each
        {"name": "counts_4m", "kind": "counts", "n": 4_194_304, "near": 31.9, "aos": False},
        # neighbour lists of a batch of probes in a cloud of points (12-byte records)
        {"name": "query_120k", "kind": "query", "n": 600_000, "nq": 120_000, "near": 30.0,
         "aos": True},
        # the standalone sort: 24-bit cells of a 256^3 grid, sorted on all 32 bits
        {"name": "sort_16m", "kind": "sort", "n": 16_777_216, "bits": 32, "key_bits": 24,
         "cells": 0},
        # cells of one frame: sort and cell ranges, an odd size
        {"name": "sort_cells_300k", "kind": "sort", "n": 300_007, "bits": 20, "key_bits": 20,
         "cells": 1_000_000},
    ]


def draw(rng):
    def size(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    kind = rng.choice(["step", "step", "frame", "unfused", "force", "counts", "query", "sort",
                       "sort"])
    if kind == "step":
        fill = rng.choice(["block", "walls", "clumps", "block"])
        exact = fill == "block" and rng.random() < 0.4
        return {"kind": kind, "fill": fill, "exact": exact,
                "n": size(2_000, 262_144 if exact else 1_048_576)}
    if kind == "frame":
        return {"kind": kind, "fill": "block", "n": size(2_000, 1_048_576),
                "substeps": rng.randint(2, 10)}
    if kind in ("unfused", "force"):
        return {"kind": kind, "fill": "block", "n": size(2_000, 400_000)}
    if kind == "counts":
        return {"kind": kind, "n": size(4_000, 4_194_304), "near": round(rng.uniform(20, 32), 1),
                "aos": rng.random() < 0.5}
    if kind == "query":
        return {"kind": kind, "n": size(4_000, 1_000_000), "nq": size(1_000, 120_000),
                "near": round(rng.uniform(15, 40), 1), "aos": rng.random() < 0.5}
    if rng.random() < 0.5:
        bits = rng.randint(12, 22)
        return {"kind": kind, "n": size(4_000, 4_194_304), "bits": bits, "key_bits": bits,
                "cells": (1 << bits) - rng.randint(0, 1 << (bits - 2))}
    return {"kind": kind, "n": size(4_000, 16_777_216), "bits": 32,
            "key_bits": rng.choice([24, 28, 32]), "cells": 0}


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _block_spacing(n):
    """Spacing of a block twice as wide and high as deep, 0.64 wide (0.005 at 1,048,576)."""
    return 0.64 / math.ceil((2 * n) ** (1 / 3) - 1e-6)


def _radius(case):
    """h: two spacings in the block; 0.01 at 1,048,576 particles spread over the box."""
    if case["fill"] == "block":
        return 2.0 * _block_spacing(case["n"])
    return 0.01 * (1_048_576 / case["n"]) ** (1 / 3) if case["n"] < 1_048_576 else 0.01


def _dims(h):
    return [math.ceil(1.0 / h - 1e-4)] * 3


def _mass(case):
    if case["fill"] == "block":
        return RHO0 * _block_spacing(case["n"]) ** 3
    return particle_mass(RHO0, case["n"])


def _clumps(g):
    centres = torch.rand(64, 3, generator=g, device="cuda")
    sigma = 0.005 + 0.045 * torch.rand(64, 1, generator=g, device="cuda")
    return centres, sigma


def _positions(case, g):
    n = case["n"]
    if case["fill"] == "block":
        s = _block_spacing(n)
        cols = round(0.64 / s)
        i = torch.arange(n, device="cuda")
        at = torch.stack([i % cols, (i // cols) % cols, i // (cols * cols)])
        jitter = 0.16 * torch.rand(3, n, generator=g, device="cuda") - 0.08
        return ((at + 0.5 + jitter) * s).float()
    p = torch.rand(3, n, generator=g, device="cuda")
    if case["fill"] == "clumps":
        centres, sigma = _clumps(g)
        m = (9 * n) // 10
        k = torch.arange(m, device="cuda") % 64
        q = centres[k] + sigma[k] * torch.randn(m, 3, generator=g, device="cuda")
        p[:, :m] = q.T.clamp(0.0, 1.0 - 2.0 ** -24)
        return p
    # walls: 4 % at the corners, 12 % on the edges, 40 % on the faces, the rest inside
    fixed = torch.zeros(n, dtype=torch.long, device="cuda")
    fixed[: int(0.56 * n)] = 1
    fixed[: int(0.16 * n)] = 2
    fixed[: int(0.04 * n)] = 3
    first = torch.randint(0, 3, (n,), generator=g, device="cuda")
    side = torch.randint(0, 2, (3, n), generator=g, device="cuda").float()
    for a in range(3):
        p[a] = torch.where((a - first) % 3 < fixed, side[a], p[a])
    return p[:, torch.randperm(n, generator=g, device="cuda")].contiguous()


def _fields(case, seed):
    """A FieldSet whose state fields are rows of one buffer (padded to 256 bytes), and a copy."""
    g = _gen(seed)
    n = case["n"]
    f = fh.FieldSet(n)
    buf = torch.zeros(6, (n + 63) // 64 * 64, device="cuda")
    buf[:3, :n] = _positions(case, g)
    buf[3:, :n] = torch.randn(3, n, generator=g, device="cuda") * 0.1
    for row, name in enumerate(("pos_x", "pos_y", "pos_z", "vel_x", "vel_y", "vel_z")):
        f.f32_fields[name] = buf[row, :n]
    f.f32_fields["density"] = torch.zeros(n, device="cuda")
    return f, buf, buf.clone()


def _options(ctx, case):
    clumps = case.get("fill") == "clumps"
    for option, value in ((fh.FH_OPT_SPH_EXACT, int(bool(case.get("exact")))),
                          (fh.FH_OPT_SUBCELL, 8 if clumps else 0),
                          (fh.FH_OPT_HEAVY_PARTS, 8 if clumps else 0),
                          (fh.FH_OPT_HEAVY_WORK, 384 if clumps else 0),
                          (fh.FH_OPT_HEAVY_SLOTS, 1 << 30 if clumps else 0)):
        ctx.set_option(option, value)


def _points(case, g):
    p = torch.rand(3, case["n"], generator=g, device="cuda")
    return p.T.contiguous() if case["aos"] else tuple(a.contiguous() for a in p)


def _reach(case):
    """Radius (and cell) that `near` uniform points fall into on average."""
    return (case["near"] / case["n"] * 3.0 / (4.0 * math.pi)) ** (1 / 3)


def _keys(case, g):
    if case["cells"]:
        return torch.randint(0, case["cells"], (case["n"],), generator=g, device="cuda",
                             dtype=torch.int32)
    full = torch.randint(-(1 << 31), 1 << 31, (case["n"],), generator=g, device="cuda",
                         dtype=torch.int32)
    if case["key_bits"] == 32:
        return full
    return full & ((1 << case["key_bits"]) - 1)


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "sort":
        k0 = _keys(case, _gen(seed))
        pairs = torch.stack([k0, torch.arange(n, device="cuda", dtype=torch.int32)])
        cells = [torch.empty(case["cells"], device="cuda", dtype=torch.int32) for _ in range(2)]
        return {"kind": kind, "case": case, "start": pairs, "pairs": [k0.clone(), k0.clone()],
                "sorter": fh.RadixSorter(n), "cells": cells}
    if kind in ("counts", "query"):
        g = _gen(seed)
        r = _reach(case)
        state = {"kind": kind, "points": _points(case, g), "radius": r,
                 "grid": fh.HashGrid(r, _dims(r), max_particles=n)}
        if kind == "query":
            state["grid"].build(state["points"])
            q = 1.04 * torch.rand(3, case["nq"], generator=g, device="cuda") - 0.02
            state["queries"] = q.T.contiguous() if case["aos"] else tuple(a.contiguous() for a in q)
            # the program's buffer of neighbour lists, which its next kernel reads
            state["lists"] = torch.zeros(int(1.1 * case["near"] * case["nq"]) + 4096,
                                         device="cuda", dtype=torch.int32)
        return state
    h = _radius(case)
    dims, mass = _dims(h), _mass(case)
    fields, buf, start = _fields(case, seed)
    state = {"kind": kind, "fields": fields, "buf": buf, "start": start}
    ctx = fields.context(dims[0] ** 3)
    _options(ctx, case)
    fused = fh.SphFusedModule(h, h, dims, mass, GAS, RHO0, MU)
    pipe = fh.Pipeline()
    if kind == "unfused":
        pipe.add(fh.SphDensityModule(h, h, dims, mass))
        pipe.add(fh.SphPressureModule(GAS, RHO0, h, h, dims, mass))
        pipe.add(fh.SphViscosityModule(MU, h, h, dims, mass))
    else:
        if kind != "frame":
            fused.accel = torch.zeros(3, n, device="cuda")
        pipe.add(fused)
    if kind == "force":
        p = buf[:3, :n].double()
        order, starts, key = _cells64(p, h, dims, torch.float32)
        fields.f32_fields["density"] = _density64(p, h, mass, dims).float()
        fields.u32_fields["cell_start"] = starts.int()
        fields.u32_fields["sorted_indices"] = order.int()
    pipe.add(fh.GravityModule(*GRAVITY))
    pipe.add(fh.IntegrateModule())
    pipe.add(fh.BoxColliderModule(0.0, 0.0, 0.0, 1.0, 1.0, 1.0, RESTITUTION))
    state.update(fused=fused, pipe=pipe, substeps=case.get("substeps", 1))
    if kind == "unfused":
        pipe.modules[0].prepare(fields)
    return state


def run(state):
    kind = state["kind"]
    if kind == "sort":
        keys, vals = state["pairs"]
        case = state["case"]
        keys.copy_(state["start"][0])
        vals.copy_(state["start"][1])
        state["sorter"].sort(keys, vals, case["n"], case["bits"])
        if case["cells"]:
            fh.find_cell_boundaries(keys, *state["cells"], case["n"], case["cells"],
                                    ctx=state["sorter"].ctx)
        return [keys, vals, *state["cells"]]
    if kind == "counts":
        grid = state["grid"]
        grid.build(state["points"])
        counts, weights = grid.neighbor_counts(state["radius"], state["points"])
        return [weights, counts, grid.cell_start, grid.sorted_indices, grid.cell_indices]
    if kind == "query":
        counts, offsets, found = state["grid"].query_neighbors_batch(
            state["queries"], state["radius"], state["points"])
        state["lists"][:found.numel()].copy_(found)
        return [counts, offsets, state["lists"]]
    fields = state["fields"]
    f = fields.f32_fields
    if kind == "force":
        ctx = fields.context()
        with torch.cuda.stream(ctx.torch_stream()):
            state["buf"].copy_(state["start"])
        state["fused"].execute_force(fields, DT)
        ctx.sync()
        return [state["fused"].accel, f["vel_x"], f["vel_y"], f["vel_z"]]
    state["buf"].copy_(state["start"])
    if kind == "frame":
        state["pipe"].run(fields, DT, state["substeps"])
    else:
        state["pipe"].step(fields, DT)
    out = [f[k] for k in ("density", "pos_x", "pos_y", "pos_z", "vel_x", "vel_y", "vel_z")]
    if kind == "step":
        out.append(state["fused"].accel)
    return out


# ---- what a pass cannot do without ----------------------------------------------------------

# float operations of one pair: distance 8; density weight 5; pressure and viscosity terms 24
_DIST, _DENSITY, _FORCE = 8, 5, 24


def _neighbours(case):
    """Mean number of particles within h of a particle."""
    n = case["n"]
    if case["fill"] == "block":
        return 33.5
    h = _radius(case)
    ball = 4.0 / 3.0 * math.pi * h ** 3
    if case["fill"] == "clumps":  # mean over the clumps, sigma uniform in [0.005, 0.05]
        per, total = 0.9 * n / 64, 0.0
        for k in range(64):
            s = 0.005 + 0.045 * (k + 0.5) / 64
            total += per * min(1.0, ball / ((4.0 * math.pi) ** 1.5 * s ** 3))
        return 0.9 * total / 64 + 0.1 * n * ball
    # (corner points collapse to one particle each)
    return 0.44 * 0.44 * n * ball + 0.4 * 0.4 * n / 6 * math.pi * h * h + 0.12 * 0.12 * n / 12 * 2 * h


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "sort":
        return {"bytes": 16 * n + 8 * case["cells"], "flops": 0}
    if kind in ("counts", "query"):
        cells = _dims(_reach(case))[0] ** 3
        pair = (_DIST + 5) * case["near"]
        if kind == "counts":
            return {"bytes": 12 * n + 8 * n + 8 * n + 4 * cells, "flops": pair * n}
        # the cells around each query, its point and its list
        return {"bytes": case["nq"] * (12 + 8 + case["near"] * (12 + 4 + 4)),
                "flops": _DIST * case["near"] * case["nq"]}
    pairs = _neighbours(case) * n
    state = 24 * n + 24 * n + 4 * n
    if kind == "force":
        return {"bytes": 24 * n + 8 * n + 24 * n, "flops": pairs * (_DIST + _FORCE)}
    per_step = pairs * (2 * _DIST + _DENSITY + _FORCE)
    if kind == "unfused":
        per_step = pairs * (3 * _DIST + _DENSITY + _FORCE)
        state += 4 * n + 4 * _dims(_radius(case))[0] ** 3
    return {"bytes": state + (12 * n if kind == "step" else 0),
            "flops": per_step * case.get("substeps", 1)}


def tolerance(case):
    """About four times what the fused module's two arithmetic modes (other sums, other order)
    and 64-bit arithmetic were seen to differ by."""
    if case["kind"] in ("sort", "query"):
        return "exact"
    if case["kind"] == "counts":
        return {"rel": 1e-6, "max": 5e-6}
    if case["kind"] == "frame":  # ten substeps carry a rounding on: seen 6.5e-5 and 5e-3
        return {"rel": 3e-4, "max": 0.02}
    if case.get("fill") == "walls":  # thousands of equal terms per corner: seen 2.1e-5 and 8e-5
        return {"rel": 1e-4, "max": 4e-4}
    return {"rel": 5e-6, "max": 5e-5}  # seen 1.3e-6 and 1.3e-5


# ---- the same results in 64 bits ------------------------------------------------------------


def _cells64(p, cell, dims, kind=torch.float64):
    """(order, starts, keys) of the cells of points (3, n): keys floor(p / cell) clamped."""
    c = torch.tensor(cell, dtype=torch.float32).to(kind).item()
    at = [torch.floor(p[a].to(kind) / c).long().clamp(0, dims[a] - 1) for a in range(3)]
    key = at[0] + dims[0] * (at[1] + dims[1] * at[2])
    order = torch.argsort(key, stable=True)
    starts = torch.zeros(dims[0] * dims[1] * dims[2] + 1, dtype=torch.long, device=p.device)
    starts[1:] = torch.cumsum(torch.bincount(key, minlength=starts.numel() - 1), 0)
    return order, starts, key


def _pairs64(p, cell, dims, chunk=1 << 24):
    """All candidate pairs (i, j) of the 27-cell neighbourhoods, in pieces."""
    order, starts, key = _cells64(p, cell, dims)
    x, y, z = key % dims[0], key // dims[0] % dims[1], key // (dims[0] * dims[1])
    lo, hi = (x - 1).clamp(min=0), (x + 1).clamp(max=dims[0] - 1)
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            ny, nz = y + dy, z + dz
            ok = (ny >= 0) & (ny < dims[1]) & (nz >= 0) & (nz < dims[2])
            row = (ny + dims[1] * nz).clamp(0, dims[1] * dims[2] - 1) * dims[0]
            b = starts[row + lo]
            cnt = torch.where(ok, starts[row + hi + 1] - b, torch.zeros_like(b))
            # particles in sorted order, so that neighbouring ones read the same candidates
            b, cnt = b[order], cnt[order]
            ends = torch.cumsum(cnt, 0)
            total, at = int(ends[-1]), 0
            while at < total:
                i0 = int(torch.searchsorted(ends, at, right=True))
                i1 = max(i0 + 1, int(torch.searchsorted(ends, at + chunk, right=True)))
                c = cnt[i0:i1]
                i = torch.repeat_interleave(torch.arange(i0, i0 + c.numel(), device=p.device), c)
                first = ends[i0:i1] - c
                j = torch.arange(at, int(ends[i0 + c.numel() - 1]), device=p.device)
                j = j - torch.repeat_interleave(first - b[i0:i1], c)
                at = int(ends[i0 + c.numel() - 1])
                yield order[i], order[j]


def _near64(p, h, dims):
    """The pairs within h: (i, j, p_i - p_j, squared distance)."""
    h2 = _f32(_f32(h) * _f32(h))
    for i, j in _pairs64(p, h, dims):
        d = p[:, i] - p[:, j]
        r2 = (d * d).sum(0)
        keep = r2 < h2
        yield i[keep], j[keep], d[:, keep], r2[keep]


def _f32(v):
    return torch.tensor(v, dtype=torch.float32).item()


def _density64(p, h, mass, dims):
    h, mass = _f32(h), _f32(mass)
    rho = torch.zeros(p.shape[1], dtype=torch.float64, device=p.device)
    for i, _, _, r2 in _near64(p, h, dims):
        rho.index_add_(0, i, (h * h - r2) ** 3)
    return rho * (mass * 315.0 / (64.0 * math.pi * h ** 9))


def _force64(p, v, rho, h, mass, dims, pressure=True, viscosity=True):
    """Acceleration (pressure + viscosity) / rho of every particle."""
    h, mass = _f32(h), _f32(mass)
    out = torch.zeros_like(p)
    coef = 45.0 / (math.pi * h ** 6)
    pr = GAS * (rho - RHO0)
    for i, j, d, r2 in _near64(p, h, dims):
        keep = (r2 > 1e-12) & (rho[j] >= 1e-6)
        i, j, d, r2 = i[keep], j[keep], d[:, keep], r2[keep]
        r = r2.sqrt()
        term = torch.zeros_like(d)
        if pressure:
            term += mass * (pr[i] + pr[j]) / (2.0 * rho[j]) * coef * (h - r) ** 2 / r * d
        if viscosity:
            term += _f32(MU) * mass / rho[j] * coef * (h - r) * (v[:, j] - v[:, i])
        for a in range(3):
            out[a].index_add_(0, i, term[a])
    return torch.where(rho >= 1e-6, out / rho, torch.zeros_like(out))


def _epilogue64(p, v):
    dt = _f32(DT)
    v = v + torch.tensor([_f32(g) for g in GRAVITY], dtype=torch.float64, device=p.device)[:, None] * dt
    p = p + v * dt
    low, high = p < 0.0, p > 1.0
    e = _f32(RESTITUTION)
    v = torch.where(low, v.abs() * e, torch.where(high, -v.abs() * e, v))
    return p.clamp(0.0, 1.0), v


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind in ("sort", "query"):
        return None  # whole numbers only
    if case.get("fill") == "clumps" and n > 400_000:
        return None  # 78 s at 2,097,152
    if kind == "counts":
        pts = _points(case, _gen(seed))
        p = (pts.T if case["aos"] else torch.stack(pts)).double()
        r = _f32(_reach(case))
        w = torch.zeros(n, dtype=torch.float64, device="cuda")
        for i, _, _, r2 in _near64(p, r, _dims(_reach(case))):
            w.index_add_(0, i, (r * r - r2) ** 3)
        return [w * (315.0 / (64.0 * math.pi * r ** 9)), None, None, None, None]
    h = _radius(case)
    dims, mass = _dims(h), _mass(case)
    g = _gen(seed)
    p = _positions(case, g).double()
    v = (torch.randn(3, n, generator=g, device="cuda") * 0.1).double()
    if kind == "force":
        rho = _density64(p, h, mass, dims).float().double()
        a = _force64(p, v, rho, h, mass, dims)
        v = v + a * _f32(DT)
        return [a, v[0], v[1], v[2]]
    for _ in range(case.get("substeps", 1)):
        rho = _density64(p, h, mass, dims)
        if kind == "unfused":
            v = v + _force64(p, v, rho, h, mass, dims, viscosity=False) * _f32(DT)
            v = v + _force64(p, v, rho, h, mass, dims, pressure=False) * _f32(DT)
        else:
            a = _force64(p, v, rho, h, mass, dims)
            v = v + a * _f32(DT)
        p, v = _epilogue64(p, v)
    out = [rho, p[0], p[1], p[2], v[0], v[1], v[2]]
    return out + [a] if kind == "step" else out
