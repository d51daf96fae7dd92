"""GPU parity of the unfused SPH modules (C ABI fh_sph_pressure, fh_sph_viscosity, and the grid
that fh_sph_density leaves in the FieldSet) against the oracle.  These kernels evaluate the
reference expressions term by term in the reference's neighbour order (sph_pressure.rs:28-112,
sph_viscosity.rs:27-106), so from identical inputs every velocity is bit-identical."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def u32(t):
    return t.cpu().numpy().view(np.uint32)


def state(cfg, seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(-0.5, 0.5, cfg.n).astype(np.float32) for _ in range(3)]


def clumps():
    """Wall-pinned particles (y = 0), a clump of 300 at one point and 200 at the corner."""
    from forge_hip import workloads
    cfg = workloads.small_sph(n=30_000, cols=24)
    rng = np.random.default_rng(21)
    k = cfg.n // 3
    cfg.x[:k] = rng.uniform(0.0, 0.03, k).astype(np.float32)
    cfg.y[:k] = 0.0
    cfg.z[:k] = rng.uniform(0.0, 0.05, k).astype(np.float32)
    cfg.x[k:k + 300], cfg.y[k:k + 300], cfg.z[k:k + 300] = 0.31, 0.42, 0.27
    cfg.x[k + 300:k + 500], cfg.y[k + 300:k + 500], cfg.z[k + 300:k + 500] = 1.0, 1.0, 1.0
    return cfg


def fieldset(fh, cfg, vel):
    f = fh.FieldSet(cfg.n)
    for nm, a in (("pos_x", cfg.x), ("pos_y", cfg.y), ("pos_z", cfg.z), ("vel_x", vel[0]),
                  ("vel_y", vel[1]), ("vel_z", vel[2])):
        f.f32_fields[nm] = dev(a)
    return f


def modules(fh, cfg):
    d = fh.SphDensityModule(cfg.h, cfg.cell_size, cfg.dims, cfg.mass)
    p = fh.SphPressureModule(cfg.gas_constant, cfg.rest_density, cfg.h, cfg.cell_size, cfg.dims,
                             cfg.mass)
    v = fh.SphViscosityModule(cfg.viscosity, cfg.h, cfg.cell_size, cfg.dims, cfg.mass)
    return d, p, v


@pytest.mark.parametrize("exact", [0, 1])
def test_density_module_leaves_the_hashgrid(fh, gpu_ctx, oracle, exact):
    """cell_start / sorted_indices written by the density module equal HashGrid::build's."""
    from forge_hip import workloads
    cfg = workloads.config0()
    f = fieldset(fh, cfg, state(cfg, 1))
    f.context(cfg.num_cells).set_option(fh.FH_OPT_SPH_EXACT, exact)
    d, _, _ = modules(fh, cfg)
    torch.cuda.synchronize()
    d.execute(f, cfg.dt)
    f.context().sync()
    f.context().set_option(fh.FH_OPT_SPH_EXACT, 0)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    assert np.array_equal(u32(f.u32_fields["cell_start"]), ocs)
    assert np.array_equal(u32(f.u32_fields["sorted_indices"]), osi)


@pytest.mark.parametrize("dims", [(16, 8, 2), (257, 1, 1), (16, 16, 256), (257, 256, 1),
                                  (128, 64, 128), (1025, 1024, 1)])
def test_density_module_grid_with_long_gaps(fh, gpu_ctx, oracle, dims):
    """Empty cells before, between and behind the runs, with runs at and beside the edges of the
    256-cell blocks that are filled apart from the slots."""
    nx, ny, nz = dims
    C = nx * ny * nz
    rng = np.random.default_rng(C)
    edges = np.array([0, 1, 255, 256, 257, 511, 512, 1023, 1024, 1025, 2047, 2048, C // 2, C - 1025,
                      C - 1024, C - 257, C - 256, C - 2, C - 1])
    edges = edges[(edges >= 0) & (edges < C)]
    f = fh.FieldSet(3000)
    for picks in ([0], [C - 1], [0, C - 1], edges, rng.choice(edges, 4), rng.integers(0, C, 2500)):
        cells = rng.choice(np.asarray(picks), 3000)
        cells[:len(picks)] = picks
        p = [(c + rng.uniform(0.1, 0.9, 3000)).astype(np.float32)
             for c in (cells % nx, cells // nx % ny, cells // (nx * ny))]
        for nm, a in zip(("pos_x", "pos_y", "pos_z"), p):
            f.f32_fields[nm] = dev(a)
        f.context(C)
        torch.cuda.synchronize()
        fh.SphDensityModule(1.0, 1.0, dims, 1.0).execute(f, 1e-4)
        f.context().sync()
        ocs, osi, _ = oracle.hashgrid_build(*p, 1.0, (0, 0, 0), dims)
        assert np.array_equal(u32(f.u32_fields["cell_start"]), ocs)
        assert np.array_equal(u32(f.u32_fields["sorted_indices"]), osi)


@pytest.mark.parametrize("which", ["pressure", "viscosity"])
@pytest.mark.parametrize("case", ["c0", "clumps"])
def test_unfused_pass_is_bit_exact(fh, gpu_ctx, oracle, which, case):
    """One pass from the oracle's own density and grid: identical velocities."""
    from forge_hip import workloads
    cfg = workloads.config0() if case == "c0" else clumps()
    print(f"unfused {which} on {case} ({cfg.n} particles)", flush=True)
    vel = state(cfg, 2)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    prm = oracle.sph_params(cfg.h, cfg.cell_size, cfg.dims, cfg.mass, cfg.gas_constant,
                            cfg.rest_density, cfg.viscosity)
    rho = oracle.sph_density(prm, cfg.x, cfg.y, cfg.z, ocs, osi)
    rho[::97] = 0.0  # particles below the 1e-6 density cut: skipped as i and as j
    f = fieldset(fh, cfg, vel)
    f.f32_fields["density"] = dev(rho)
    f.u32_fields["cell_start"] = fh.from_u32(ocs)
    f.u32_fields["sorted_indices"] = fh.from_u32(osi)
    _, p, v = modules(fh, cfg)
    m = p if which == "pressure" else v
    ref = (oracle.sph_pressure if which == "pressure" else oracle.sph_viscosity)(
        prm, cfg.x, cfg.y, cfg.z, *vel, rho, ocs, osi, cfg.dt)
    f.context(cfg.num_cells)
    torch.cuda.synchronize()
    m.execute(f, cfg.dt)
    f.context().sync()
    for c, nm in enumerate(("vel_x", "vel_y", "vel_z")):
        got = f.f32_fields[nm].cpu().numpy()
        assert np.array_equal(got, ref[c]), nm
    assert not np.array_equal(ref[0], vel[0])  # the pass did change the state


def test_unfused_pipeline_is_bit_exact(fh, gpu_ctx, oracle):
    """density -> pressure -> viscosity -> gravity -> integrate -> box, one Pipeline::step with
    the exact density pass: the viscosity pass sees the velocities the pressure pass wrote."""
    from forge_hip import workloads
    cfg = workloads.small_sph(n=20_000, cols=24)
    vel = state(cfg, 3)
    f = fieldset(fh, cfg, vel)
    f.context(cfg.num_cells).set_option(fh.FH_OPT_SPH_EXACT, 1)
    d, p, v = modules(fh, cfg)
    pipe = fh.Pipeline()
    for m in (d, p, v, fh.GravityModule(*cfg.gravity), fh.IntegrateModule(),
              fh.BoxColliderModule(*cfg.box_min, *cfg.box_max, cfg.restitution)):
        pipe.add(m)
    torch.cuda.synchronize()
    pipe.step(f, cfg.dt)
    f.context().set_option(fh.FH_OPT_SPH_EXACT, 0)
    prm = oracle.sph_params(cfg.h, cfg.cell_size, cfg.dims, cfg.mass, cfg.gas_constant,
                            cfg.rest_density, cfg.viscosity)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    rho = oracle.sph_density(prm, cfg.x, cfg.y, cfg.z, ocs, osi)
    v1 = oracle.sph_pressure(prm, cfg.x, cfg.y, cfg.z, *vel, rho, ocs, osi, cfg.dt)
    v2 = oracle.sph_viscosity(prm, cfg.x, cfg.y, cfg.z, *v1, rho, ocs, osi, cfg.dt)
    v3 = oracle.gravity(*v2, cfg.gravity, cfg.dt)
    s = oracle.integrate(cfg.x, cfg.y, cfg.z, *v3, cfg.dt)
    s = oracle.box_collider(*s, cfg.box_min, cfg.box_max, cfg.restitution)
    assert np.array_equal(f.f32_fields["density"].cpu().numpy(), rho)
    for nm, o in zip(("pos_x", "pos_y", "pos_z", "vel_x", "vel_y", "vel_z"), s):
        assert np.array_equal(f.f32_fields[nm].cpu().numpy(), o), nm


def shuffled_grid(kind, cfg, oracle, rng):
    """A grid the exact walks must not take for one of these positions, or that they walk in its
    edge cases: positions moved since the build, or a sparse row beside a dense one (streams far
    longer than the lanes' ranges)."""
    if kind == "sparse":
        k = cfg.n // 2
        cfg.x[:k] = rng.uniform(0.0, 1.0, k)
        cfg.y[:k], cfg.z[:k] = rng.uniform(0.1, 0.124, k), rng.uniform(0.2, 0.224, k)
        cfg.x[k:], cfg.y[k:] = rng.uniform(0.0, 1.0, cfg.n - k), 0.13
        cfg.z[k:] = 0.21 + 0.3 * (np.arange(cfg.n - k) % 97 > 0)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    if kind == "moved":
        for a in ("x", "y", "z"):
            v = getattr(cfg, a)
            v += rng.uniform(-0.04, 0.04, cfg.n).astype(np.float32)
    return ocs, osi


@pytest.mark.parametrize("which", ["pressure", "viscosity"])
@pytest.mark.parametrize("kind", ["moved", "sparse"])
@pytest.mark.parametrize("n", [65, 6000])
def test_unfused_pass_over_other_grids_is_bit_exact(fh, gpu_ctx, oracle, which, kind, n):
    from forge_hip import workloads
    cfg = workloads.small_sph(n=n, cols=16)
    rng = np.random.default_rng(n + len(kind))
    ocs, osi = shuffled_grid(kind, cfg, oracle, rng)
    vel = state(cfg, 4)
    prm = oracle.sph_params(cfg.h, cfg.cell_size, cfg.dims, cfg.mass, cfg.gas_constant,
                            cfg.rest_density, cfg.viscosity)
    rho = oracle.sph_density(prm, cfg.x, cfg.y, cfg.z, ocs, osi)
    f = fieldset(fh, cfg, vel)
    f.f32_fields["density"] = dev(rho)
    f.u32_fields["cell_start"] = fh.from_u32(ocs)
    f.u32_fields["sorted_indices"] = fh.from_u32(osi)
    ref = (oracle.sph_pressure if which == "pressure" else oracle.sph_viscosity)(
        prm, cfg.x, cfg.y, cfg.z, *vel, rho, ocs, osi, cfg.dt)
    _, p, v = modules(fh, cfg)
    f.context(cfg.num_cells)
    torch.cuda.synchronize()
    (p if which == "pressure" else v).execute(f, cfg.dt)
    f.context().sync()
    for c, nm in enumerate(("vel_x", "vel_y", "vel_z")):
        assert np.array_equal(f.f32_fields[nm].cpu().numpy(), ref[c]), nm


@pytest.mark.parametrize("which", ["pressure", "viscosity"])
def test_unfused_pass_over_a_malformed_grid(fh, gpu_ctx, oracle, which):
    """Ids beyond n are no neighbours, and a particle that the grid does not hold (its slot holds such
    an id) is walked from its own position: what the CPU restatement computes with the bad slots
    removed from the neighbour lists."""
    from forge_hip import workloads
    cfg = workloads.small_sph(n=5000, cols=16)
    vel = state(cfg, 5)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    prm = oracle.sph_params(cfg.h, cfg.cell_size, cfg.dims, cfg.mass, cfg.gas_constant,
                            cfg.rest_density, cfg.viscosity)
    rho = oracle.sph_density(prm, cfg.x, cfg.y, cfg.z, ocs, osi)
    bad = osi.copy()
    bad[100::500] = 0xFFFFFFF0
    gone = osi[100::500]
    # the restatement over the same lists: a particle far away in the place of the missing ids
    far = cfg.n
    x, y, z = (np.append(a, np.float32(9.0)) for a in (cfg.x, cfg.y, cfg.z))
    ids = np.where(bad < cfg.n, bad, far).astype(np.uint32)
    ov = [np.append(a, np.float32(0.0)) for a in vel]
    ref = (oracle.sph_pressure if which == "pressure" else oracle.sph_viscosity)(
        prm, x, y, z, *ov, np.append(rho, np.float32(1.0)), ocs, np.append(ids, np.uint32(far)),
        cfg.dt)
    f = fieldset(fh, cfg, vel)
    f.f32_fields["density"] = dev(rho)
    f.u32_fields["cell_start"] = fh.from_u32(ocs)
    f.u32_fields["sorted_indices"] = fh.from_u32(bad)
    _, p, v = modules(fh, cfg)
    f.context(cfg.num_cells)
    torch.cuda.synchronize()
    (p if which == "pressure" else v).execute(f, cfg.dt)
    f.context().sync()
    for c, nm in enumerate(("vel_x", "vel_y", "vel_z")):
        got = f.f32_fields[nm].cpu().numpy()
        assert np.array_equal(got, ref[c][:cfg.n]), nm
    assert not np.array_equal(ref[0][gone], vel[0][gone])  # the missing ones moved as well


@pytest.mark.parametrize("which", ["pressure", "viscosity"])
@pytest.mark.parametrize("shift", [1, 7, 2500])
def test_unfused_pass_over_a_grid_with_duplicates(fh, gpu_ctx, oracle, which, shift):
    """A particle that the grid holds twice (beside its own slot, in its neighbourhood or in a far
    cell) is a neighbour twice and is updated once; one whose slot the duplicate takes is walked
    from its own position: bit for bit the CPU restatement over the same lists."""
    from forge_hip import workloads
    cfg = workloads.small_sph(n=5000, cols=16)
    vel = state(cfg, 6)
    ocs, osi, _ = oracle.hashgrid_build(cfg.x, cfg.y, cfg.z, cfg.cell_size, (0, 0, 0), cfg.dims)
    prm = oracle.sph_params(cfg.h, cfg.cell_size, cfg.dims, cfg.mass, cfg.gas_constant,
                            cfg.rest_density, cfg.viscosity)
    rho = oracle.sph_density(prm, cfg.x, cfg.y, cfg.z, ocs, osi)
    ids = osi.copy()
    at = np.arange(50, cfg.n - shift, 97)
    ids[at] = osi[at + shift]
    twice, gone = osi[at + shift], osi[at]
    assert np.bincount(ids, minlength=cfg.n)[twice].min() >= 2
    ref = (oracle.sph_pressure if which == "pressure" else oracle.sph_viscosity)(
        prm, cfg.x, cfg.y, cfg.z, *vel, rho, ocs, ids, cfg.dt)
    f = fieldset(fh, cfg, vel)
    f.f32_fields["density"] = dev(rho)
    f.u32_fields["cell_start"] = fh.from_u32(ocs)
    f.u32_fields["sorted_indices"] = fh.from_u32(ids)
    _, p, v = modules(fh, cfg)
    f.context(cfg.num_cells)
    torch.cuda.synchronize()
    (p if which == "pressure" else v).execute(f, cfg.dt)
    f.context().sync()
    for c, nm in enumerate(("vel_x", "vel_y", "vel_z")):
        assert np.array_equal(f.f32_fields[nm].cpu().numpy(), ref[c]), nm
    for some in (twice, gone):
        assert not np.array_equal(ref[0][some], vel[0][some])
