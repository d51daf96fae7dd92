"""GPU parity of hashing, HashGrid::build and the neighbour queries (C ABI fh_hash_cells,
fh_hashgrid_build, fh_query_neighbors, fh_neighbor_query) against the oracle and the
reference's hash-grid known answers.  Bar: bit-exact cells, cell ranges, sorted indices,
neighbour lists and counts; weight sums within rel 1e-4."""
import json
from pathlib import Path

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
KATS = json.loads((Path(__file__).parent / "golden" / "reference_kats.json").read_text())


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def test_hashgrid_basic(fh, gpu_ctx):
    kat = KATS["hashgrid_basic"]
    grid = fh.HashGrid(kat["cell_size"], kat["dims"], kat["origin"], 100, ctx=gpu_ctx)
    pos = dev(kat["positions"])
    grid.build(pos)
    nb = grid.query_neighbors(kat["query"], kat["radius"], pos)
    for i in kat["must_contain"]:
        assert i in nb
    for i in kat["must_not_contain"]:
        assert i not in nb
    assert nb == kat["neighbors"]


def test_hashgrid_uniform_distribution(fh, gpu_ctx):
    kat = KATS["hashgrid_uniform"]
    i = np.arange(1000)
    pos = np.stack([(i % 10) + 0.5, ((i // 10) % 10) + 0.5, (i // 100) + 0.5], 1)
    grid = fh.HashGrid(kat["cell_size"], kat["dims"], kat["origin"], 1000, ctx=gpu_ctx)
    p = dev(pos)
    grid.build(p)
    nb = grid.query_neighbors(kat["query"], kat["radius"], p)
    assert len(nb) >= kat["reference_asserts_at_least"]
    assert sorted(nb) == kat["neighbors_sorted"] and len(nb) == kat["count"]


def edge_positions(n, rng, lo=-0.2, hi=1.2):
    p = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    specials = np.array([np.nan, np.inf, -np.inf, -0.0, 0.0, 1.0, 0.5, 3e38, -3e38, 1e-45,
                         0.25, 0.75, 0.999999], np.float32)
    k = min(n, 400)
    p[:k] = rng.choice(specials, (k, 3))
    return p


@pytest.mark.parametrize("layout", ["aos", "soa"])
@pytest.mark.parametrize("n,cs,dims,origin", [
    (5000, 0.05, (20, 20, 20), (0.0, 0.0, 0.0)),
    (100_000, 0.0122, (82, 82, 82), (0.0, 0.0, 0.0)),
    (70_001, 0.1, (7, 13, 3), (-0.1, 0.2, 0.05)),
    (1, 1.0, (1, 1, 1), (0.0, 0.0, 0.0)),
    (20_000, 1.0, (1, 1, 1), (0.0, 0.0, 0.0)),      # one cell: no sort pass moves keys
    (20_000, 0.5, (2, 1, 1), (0.0, 0.0, 0.0)),      # one 1-bit pass
])
def test_build_matches_oracle(fh, gpu_ctx, oracle, layout, n, cs, dims, origin):
    rng = np.random.default_rng(n)
    p = edge_positions(n, rng)
    grid = fh.HashGrid(cs, dims, origin, n, ctx=gpu_ctx)
    if layout == "aos":
        grid.build(dev(p))
    else:
        grid.build(tuple(dev(p[:, a].copy()) for a in range(3)))
    ocs, osi, oci = oracle.hashgrid_build(p[:, 0], p[:, 1], p[:, 2], grid.cell_size, grid.origin, dims)
    assert np.array_equal(fh.to_u32(grid.cell_start), ocs)
    assert np.array_equal(fh.to_u32(grid.sorted_indices)[:n], osi)
    assert np.array_equal(fh.to_u32(grid.cell_indices)[:n], oci)


def test_build_empty(fh, gpu_ctx):
    grid = fh.HashGrid(0.1, (4, 4, 4), (0, 0, 0), 0, ctx=gpu_ctx)
    grid.build(torch.zeros((0, 3), dtype=torch.float32, device="cuda"))
    assert np.all(fh.to_u32(grid.cell_start) == 0)


def test_position_to_cell_matches_oracle(fh, gpu_ctx, oracle):
    grid = fh.HashGrid(0.3, (5, 6, 7), (0.1, -0.2, 0.0), 16, ctx=gpu_ctx)
    for q in [(0.1, -0.2, 0.0), (float("nan"), 0.5, 0.5), (1e30, -1e30, 2.0), (0.4, 0.1, 0.3),
              (0.39999998, 0.09999999, 0.29999998), (-0.0, 0.0, 2.1)]:
        assert grid.position_to_cell(q) == oracle.position_to_cell(q, grid.cell_size, grid.origin,
                                                                   grid.dims)


def test_query_batch_matches_oracle(fh, gpu_ctx, oracle):
    rng = np.random.default_rng(11)
    n, cs, dims = 20_000, 0.05, (20, 20, 20)
    p = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    q = rng.uniform(-0.15, 1.15, (3000, 3)).astype(np.float32)  # some queries outside the grid
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    P = dev(p)
    grid.build(P)
    counts, offsets, idx = grid.query_neighbors_batch(dev(q), 0.04, P)
    counts, offsets, idx = fh.to_u32(counts), fh.to_u32(offsets), fh.to_u32(idx)
    ocs, osi, _ = oracle.hashgrid_build(p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims)
    for t in range(q.shape[0]):
        exp = oracle.query_neighbors(q[t], 0.04, p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims, ocs, osi)
        got = idx[offsets[t]:offsets[t + 1]]
        assert counts[t] == exp.size
        assert np.array_equal(got, exp), t


@pytest.mark.parametrize("layout", ["aos", "soa"])
@pytest.mark.parametrize("n,nq", [(1, 1), (40, 1025), (3000, 63), (40_000, 1024), (40_000, 1249),
                                  (40_000, 1300)])
def test_query_batch_sizes_match_oracle(fh, gpu_ctx, oracle, layout, n, nq):
    """Rows shorter and longer than a step of 16 candidates, queries outside the grid, partial waves; a
    context too small for the grid's points reads them in place."""
    rng = np.random.default_rng(n + nq)
    cs, dims = 0.05, (20, 20, 20)
    p = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    p[: n // 2] = 0.4 + 0.1 * p[: n // 2]  # dense: rows of several steps
    q = rng.uniform(-0.1, 1.1, (nq, 3)).astype(np.float32)
    q[: nq // 2] = 0.35 + 0.2 * q[: nq // 2]
    pack = dev if layout == "aos" else lambda a: tuple(dev(a[:, k].copy()) for k in range(3))
    P, Q = pack(p), pack(q)
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    grid.build(P)
    ocs, osi, _ = oracle.hashgrid_build(p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims)
    small = fh.Context(max_n=16, max_cells=8000)
    try:
        for ctx in (gpu_ctx, small):
            grid.ctx = ctx
            counts, offsets, idx = (fh.to_u32(t) for t in grid.query_neighbors_batch(Q, 0.04, P))
            for t in range(0, nq, max(1, nq // 150)):
                exp = oracle.query_neighbors(q[t], 0.04, p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0),
                                             dims, ocs, osi)
                assert counts[t] == exp.size
                assert np.array_equal(idx[offsets[t]:offsets[t + 1]], exp), t
    finally:
        grid.ctx = gpu_ctx
        small.close()


@pytest.mark.parametrize("n,nq", [(300, 3555), (300, 3556), (6000, 1100), (6000, 3555),
                                  (30_000, 3556), (262_143, 3555), (262_143, 3556),
                                  (262_144, 1024)])
def test_query_batch_rules_match_oracle(fh, gpu_ctx, oracle, n, nq):
    """On either side of the copy's rule (12 candidates per point, 2.5 from 2^18 points on) and of the
    walk over rows that hold points only: few points per row, empty rows, full ones."""
    rng = np.random.default_rng(n + nq)
    cs, dims = 0.05, (20, 20, 20)
    p = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    q = rng.uniform(-0.05, 1.05, (nq, 3)).astype(np.float32)
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    P = dev(p)
    grid.build(P)
    ocs, osi, _ = oracle.hashgrid_build(p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims)
    counts, offsets, idx = (fh.to_u32(t) for t in grid.query_neighbors_batch(dev(q), 0.03, P))
    for t in range(0, nq, max(1, nq // 150)):
        exp = oracle.query_neighbors(q[t], 0.03, p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims,
                                     ocs, osi)
        assert counts[t] == exp.size
        assert np.array_equal(idx[offsets[t]:offsets[t + 1]], exp), t


@pytest.mark.parametrize("where", ["points", "elsewhere", "all over"])
@pytest.mark.parametrize("nq", [1249, 1250, 3000])
def test_query_batch_of_points_in_a_corner(fh, gpu_ctx, oracle, where, nq):
    """40,000 points in a corner of the grid: batches of a 32nd of the points on count the candidates of
    a few of their queries, which are many, none, or some, to decide for the copy; a second batch on
    the same context decides anew."""
    rng = np.random.default_rng(nq)
    cs, dims, n = 0.05, (20, 20, 20), 40_000
    p = rng.uniform(0.0, 0.25, (n, 3)).astype(np.float32)
    q = rng.uniform(0.0, 1.0, (nq, 3))
    q = (q if where == "all over" else 0.25 * q + (0.0 if where == "points" else 0.6))
    q = q.astype(np.float32)
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    P = dev(p)
    grid.build(P)
    ocs, osi, _ = oracle.hashgrid_build(p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims)
    for batch in (q, q[::-1].copy()):
        got = grid.query_neighbors_batch(dev(batch), 0.01, P)
        counts, offsets, idx = (fh.to_u32(t) for t in got)
        for t in range(0, nq, max(1, nq // 100)):
            exp = oracle.query_neighbors(batch[t], 0.01, p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0),
                                         dims, ocs, osi)
            assert counts[t] == exp.size
            assert np.array_equal(idx[offsets[t]:offsets[t + 1]], exp), t
        grid.query_neighbors_batch(dev(batch + 0.3), 0.01, P)


@pytest.mark.parametrize("kind", ["subset", "far"])
def test_query_batch_over_part_of_the_points(fh, gpu_ctx, oracle, kind):
    """A batch that copies the positions reads no more of the caller's arrays than it may: a grid
    over some of the points (ids beyond the grid's own count), and entries that hold no id at all in
    cells that no query comes near."""
    rng = np.random.default_rng(17)
    cs, dims, total, n = 0.05, (20, 20, 20), 60_000, 40_000
    p = rng.uniform(0.0, 1.0, (total, 3)).astype(np.float32)
    ids = np.sort(rng.permutation(total)[:n]) if kind == "subset" else np.arange(n)
    sub = p[ids]
    ocs, osi, cell = oracle.hashgrid_build(sub[:, 0], sub[:, 1], sub[:, 2], cs, (0, 0, 0), dims)
    near = ids[osi].astype(np.uint32)
    q = rng.uniform(0.0, 1.0, (4000, 3)).astype(np.float32)  # enough for the copy
    given = near.copy()
    if kind == "far":
        q[:, 0] *= 0.5  # cells x < 10, rows up to x = 10
        given[cell[osi] % 20 >= 12] = 0xFFFFFFF0
        p = p[:n]
    P = tuple(dev(p[:, k].copy()) for k in range(3))
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    grid.build(tuple(dev(sub[:, k].copy()) for k in range(3)))
    grid.sorted_indices[:n] = fh.from_u32(given)
    torch.cuda.synchronize()
    counts, offsets, idx = (fh.to_u32(t) for t in grid.query_neighbors_batch(dev(q), 0.04, P))
    for t in range(0, len(q), 13):
        exp = oracle.query_neighbors(q[t], 0.04, p[:, 0], p[:, 1], p[:, 2], cs, (0, 0, 0), dims,
                                     ocs, near)
        assert counts[t] == exp.size
        assert np.array_equal(idx[offsets[t]:offsets[t + 1]], exp), t


@pytest.mark.parametrize("n", [50_000, 4_194_304])
def test_neighbor_counts_matches_oracle(fh, gpu_ctx, oracle, n):
    """c2 workload (uniform points, r = cs = 0.0122, 82^3 cells); full size at n = 4,194,304."""
    from forge_hip import workloads
    c = workloads.config2(n=n)
    grid = fh.HashGrid(c["cell_size"], c["dims"], c["origin"], n, ctx=gpu_ctx)
    P = tuple(dev(c[a]) for a in "xyz")
    print(f"c2 n={n}", flush=True)
    grid.build(P)
    cnt, w = grid.neighbor_counts(c["radius"], P)
    ocs, osi, _ = oracle.hashgrid_build(c["x"], c["y"], c["z"], c["cell_size"], c["origin"], c["dims"])
    assert np.array_equal(fh.to_u32(grid.cell_start), ocs)
    assert np.array_equal(fh.to_u32(grid.sorted_indices), osi)
    ocnt, ow = oracle.neighbor_counts(c["x"], c["y"], c["z"], c["cell_size"], c["origin"],
                                      c["dims"], ocs, osi, c["radius"])
    g_cnt, g_w = fh.to_u32(cnt), w.cpu().numpy()
    assert np.array_equal(g_cnt, ocnt)
    # the configuration's bar for the weight sums is rel 1e-4; the kernel keeps the reference's
    # arithmetic and visiting order, so they are bit-identical
    rel = np.abs(g_w - ow) / np.maximum(np.abs(ow), 1e-30)
    assert rel.max() <= 1e-4
    assert np.array_equal(g_w, ow)
    print(f"c2 n={n}: mean count {g_cnt.mean():.2f}, weight sums bit-exact")


@pytest.mark.parametrize("case", ["outside", "clustered"])
def test_neighbor_counts_edge_cases_match_oracle(fh, gpu_ctx, oracle, case):
    """Points outside a non-cubic grid (sorted into clamped cells, queried around their
    unclamped cell like the reference), and tight clusters whose cells hold hundreds of points
    (candidate streams several LDS windows long): counts and weight sums bit-exact."""
    rng = np.random.default_rng(29 if case == "outside" else 30)
    cs, dims = 0.025, (40, 30, 20)
    if case == "outside":
        n = 60_000
        lo, hi = np.array([-0.05, -0.05, -0.05]), np.array([1.05, 0.8, 0.55])
        p = (lo + (hi - lo) * rng.uniform(0, 1, (n, 3))).astype(np.float32)
    else:
        n = 100_000
        p = rng.uniform(0, 1, (n, 3)) * np.array([1.0, 0.75, 0.5])
        centres = rng.uniform(0.1, 0.4, (6, 3))
        k = n // 2
        p[:k] = centres[rng.integers(0, 6, k)] + rng.normal(0, 0.01, (k, 3))
        p = p.astype(np.float32)
    x, y, z = (np.ascontiguousarray(p[:, a]) for a in range(3))
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    P = (dev(x), dev(y), dev(z))
    print(f"neighbour counts: {case}, n={n}", flush=True)
    grid.build(P)
    cnt, w = grid.neighbor_counts(cs, P)
    ocs, osi, _ = oracle.hashgrid_build(x, y, z, cs, (0, 0, 0), dims)
    assert np.array_equal(fh.to_u32(grid.sorted_indices), osi)
    ocnt, ow = oracle.neighbor_counts(x, y, z, cs, (0, 0, 0), dims, ocs, osi, cs)
    assert np.array_equal(fh.to_u32(cnt), ocnt)
    assert np.array_equal(w.cpu().numpy(), ow)
    print(f"{case}: max count {ocnt.max()}, mean {ocnt.mean():.1f}")


@pytest.mark.parametrize("n", [1, 255, 257, 30_001])
def test_neighbor_counts_of_records_match_oracle(fh, gpu_ctx, oracle, n):
    """Positions as 12-byte records, gathered without a packed copy: bit-exact as from arrays."""
    rng = np.random.default_rng(n)
    cs, dims = 0.05, (20, 20, 20)
    p = rng.uniform(-0.02, 1.02, (n, 3)).astype(np.float32)
    grid = fh.HashGrid(cs, dims, (0, 0, 0), n, ctx=gpu_ctx)
    P = dev(p)
    grid.build(P)
    cnt, w = grid.neighbor_counts(cs, P)
    x, y, z = (np.ascontiguousarray(p[:, a]) for a in range(3))
    ocs, osi, _ = oracle.hashgrid_build(x, y, z, grid.cell_size, (0, 0, 0), dims)
    ocnt, ow = oracle.neighbor_counts(x, y, z, grid.cell_size, (0, 0, 0), dims, ocs, osi, cs)
    assert np.array_equal(fh.to_u32(cnt), ocnt)
    assert np.array_equal(w.cpu().numpy(), ow)
