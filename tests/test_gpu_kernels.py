"""Kernel forms at the sizes where they change, against the oracle: the
V-cycle bit for bit (both sides do the same arithmetic in the same order)."""
import ctypes as C

import numpy as np
import pytest

from fluidisim_amd import _lib
from fluidisim_amd import workloads as W
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def problem(wl):
    d = wl.domain
    return po.Problem(d.nx, d.ny, d.nz, d.dx, wl.eta, rho=wl.rho, g_eff=wl.g_eff, rest=wl.rest,
                      homogeneous_ghost=wl.homogeneous_ghost, closed_lid=wl.closed_lid, solid=wl.solid,
                      open_u=wl.open_u, open_v=wl.open_v, open_w=wl.open_w)


def oracle_options(wl, **kw):
    o = wl.options
    return po.options(multigrid=1, smoother=o["smoother"], max_levels=o["max_levels"], pre=o["pre_sweeps"],
                      post=o["post_sweeps"], coarse=o["coarse_sweeps"], coarse_op=o.get("coarse_operator", 0), **kw)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def assert_vcycle_is_the_oracles(wl, **overrides):
    wl.options.update(overrides)
    vol = W.build_volume(wl)
    prob = problem(wl)
    _, prec = po.assemble(prob, np.zeros(wl.domain.cells, np.float32), 1.0)
    r = np.random.default_rng(13).uniform(-1.0, 1.0, wl.domain.cells).astype(np.float32)
    r[prec == 0] = 0.0
    z = vol.precondition(torch.from_numpy(r).cuda()).cpu().numpy()
    z_ref = po.vcycle(prob, r, oracle_options(wl)).astype(np.float32)
    vol.close()
    assert np.abs(z_ref).max() > 0
    assert np.array_equal(bits(z), bits(z_ref)), f"max diff {np.abs(z - z_ref).max()}"


@pytest.mark.parametrize("size,levels,sweeps", [
    ((32, 32, 32), 1, (2, 2, 8)),   # coarsest 16^3: the tail's largest level, two cells of a colour per thread
    ((32, 32, 32), 1, (1, 2, 7)),   # an odd number of coarsest sweeps
    ((32, 32, 32), -1, (2, 1, 2)),  # 16^3 as the first of the tail's levels
    ((40, 32, 24), 1, (2, 2, 3)),   # 20 x 12 x 16: the last pairs of a colour partly missing
    ((28, 20, 20), 1, (2, 2, 2)),   # 14 x 10 x 10: one pair per thread at most
    ((20, 12, 12), 1, (2, 2, 1)),   # 10 x 6 x 6, one coarsest sweep
    ((36, 32, 32), 1, (2, 2, 2)),   # 18 x 16 x 16: one level too large for the tail
    ((52, 8, 24), 2, (2, 2, 3)),    # 26 x 12 x 4 over 13 x 6 x 2: odd rows
    ((16, 8, 16), -1, (2, 2, 4)),   # 8 x 8 x 4 over 4 x 4 x 2: the last level in one wavefront
    ((16, 16, 16), -1, (1, 3, 3)),  # 8^3 over 4^3 over 2^3: two levels in one wavefront
    ((16, 16, 16), -1, (2, 2, 0)),  # no coarsest sweep
    ((20, 12, 12), -1, (2, 1, 5)),  # 10 x 6 x 6 over 5 x 3 x 3
    ((8, 8, 8), 1, (2, 2, 2)),      # 4^3 alone
    ((12, 8, 8), -1, (2, 2, 3)),    # 6 x 4 x 4 over 3 x 2 x 2
    ((128, 8, 64), 1, (2, 2, 2)),   # 64 x 32 x 4 = 8192: above the tail
    ((128, 4, 64), 1, (2, 2, 3)),   # 64 x 32 x 2: the longest plane
])
def test_tail_levels_match_the_oracle(size, levels, sweeps):
    wl = W.tank(*size, seed=21)
    assert_vcycle_is_the_oracles(wl, max_levels=levels, pre_sweeps=sweeps[0], post_sweeps=sweeps[1],
                                 coarse_sweeps=sweeps[2])


@pytest.mark.parametrize("share", [0.0005, 0.05, 1.0], ids=["few", "index", "overflow"])
@pytest.mark.parametrize("smoother", [_lib.SMOOTH_JACOBI, _lib.SMOOTH_RBGS])
@pytest.mark.parametrize("size", [(32, 24, 28), (36, 18, 20), (34, 16, 16)])
def test_rows_with_fractional_apertures_match_the_oracle(share, smoother, size):
    """The ghost-row index: a share of the faces fractional (almost every wet
    row flagged at 1.0: more rows than the index holds, the general kernels),
    on quads and on rows that do not split into quads."""
    wl = W.tank(*size, seed=31)
    rng = np.random.default_rng(32)
    d = wl.domain
    solid = np.asarray(wl.solid).reshape(d.nz, d.ny, d.nx) != 0
    opens = []
    for axis, shape in ((2, (d.nz, d.ny, d.nx + 1)), (1, (d.nz, d.ny + 1, d.nx)), (0, (d.nz + 1, d.ny, d.nx))):
        a = np.where(rng.random(shape) < share, rng.uniform(0.05, 0.95, shape), 1.0).astype(np.float32)
        lo = [slice(None)] * 3
        hi = [slice(None)] * 3
        lo[axis], hi[axis] = slice(0, -1), slice(1, None)
        a[tuple(lo)][solid] = 0
        a[tuple(hi)][solid] = 0
        lo[axis], hi[axis] = 0, -1
        a[tuple(lo)] = 0
        if axis:
            a[tuple(hi)] = 0
        opens.append(a.ravel())
    wl.open_u, wl.open_v, wl.open_w = opens
    wl.closed_lid = False
    assert_vcycle_is_the_oracles(wl, smoother=smoother, coarse_operator=_lib.COARSE_REDISCRETISED)


@pytest.mark.parametrize("share", [0.1, 0.6])
def test_scattered_water_matches_the_f64_oracle(share):
    """A level set of scattered water cells: with 0.6 of the cells water almost
    every one has an air neighbour, more rows than the ghost-row index holds."""
    from fluidisim_amd.volume import Domain3, Volume3
    nx, ny, nz, dx, rho, dt = 32, 20, 24, 0.05, 1000.0, 0.004
    rng = np.random.default_rng(41)
    water = rng.random((nz, ny, nx)) < share
    phi = np.where(water, rng.uniform(-0.04, -0.005, water.shape), rng.uniform(0.005, 0.04, water.shape)).astype(np.float32)
    label = np.where(water, _lib.LABEL_WATER, _lib.LABEL_AIR).astype(np.uint8)
    u, v, w = (rng.uniform(-0.2, 0.2, s).astype(np.float32) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)))
    u[:, :, [0, nx]] = 0
    v[:, [0, ny]] = 0
    w[[0, nz]] = 0
    vol = Volume3.configure(Domain3(nx, ny, nz, dx), rho=rho, g_eff=9.81, preconditioner=_lib.PRECOND_MULTIGRID,
                            smoother=_lib.SMOOTH_RBGS, max_levels=-1, pre_sweeps=2, post_sweeps=2, coarse_sweeps=8,
                            coarse_operator=_lib.COARSE_GALERKIN)
    vol.set_level_set(label.ravel(), phi.ravel())
    vol.set_velocity(u.ravel(), v.ravel(), w.ravel())
    rep = vol.project_mobile3(-rho / dt, dt / rho, 2000, rel_tol=1e-8, warm=False)
    p = vol.pressure().cpu().numpy().astype(np.float64)
    vol.close()
    p64, *_ = po.apic_project(nx, ny, nz, dx, rho, dt, label.ravel(), phi.ravel(), u.ravel(), v.ravel(), w.ravel(),
                              precision=64)
    m = water.ravel()
    # the oracle stops at a relative residual of 1e-6 on a system whose smallest
    # theta (0.11) keeps its condition below 100
    assert np.linalg.norm(p[m] - p64[m]) <= 1e-4 * np.linalg.norm(p64[m])


@pytest.mark.parametrize("size,levels,sweeps", [
    ((48, 32, 32), -1, (2, 2, 8)),   # 24 x 16 x 16 above the tail
    ((48, 32, 32), -1, (3, 1, 5)),   # an odd number of sweeps: the other buffer
    ((48, 32, 32), -1, (1, 2, 1)),   # one pre-sweep: the fine level a thread per cell
    ((48, 32, 32), -1, (2, 0, 0)),   # no post-sweep, no coarsest sweep
    ((32, 32, 32), 1, (2, 2, 8)),    # 16^3: the tail's largest level
    ((52, 36, 40), 2, (2, 3, 2)),    # 26 x 20 x 18 over 13 x 10 x 9: odd rows
    ((34, 32, 32), -1, (2, 2, 3)),   # rows that do not split into quads
    ((36, 34, 38), 1, (4, 2, 3)),    # 18 x 19 x 17 as the coarsest level above the tail
], ids=str)
@pytest.mark.parametrize("smoother", [_lib.SMOOTH_JACOBI, _lib.SMOOTH_RBGS])
@pytest.mark.parametrize("coarse_operator", [_lib.COARSE_REDISCRETISED, _lib.COARSE_GALERKIN])
def test_levels_of_row_coefficients_match_the_oracle(size, levels, sweeps, smoother, coarse_operator):
    if smoother == _lib.SMOOTH_RBGS and 0 in sweeps:
        sweeps = (1, 1, 3)
    wl = W.tank(*size, seed=51)
    assert_vcycle_is_the_oracles(wl, max_levels=levels, pre_sweeps=sweeps[0], post_sweeps=sweeps[1],
                                 coarse_sweeps=sweeps[2], smoother=smoother, coarse_operator=coarse_operator)


@pytest.mark.parametrize("sweeps", [0, 1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("size", [
    (40, 36, 32),   # 20 x 18 x 16: tiles cut by the level's edge in x and y
    (48, 34, 42),   # 24 x 17 x 21: odd rows and planes
    (80, 16, 56),   # 40 x 8 x 28
], ids=str)
def test_a_coarsest_level_above_the_tail_matches_the_oracle(size, sweeps):
    """1 to 16 colour passes, up to five to a launch."""
    assert_vcycle_is_the_oracles(W.tank(size[0], size[2], size[1], seed=71), max_levels=1, coarse_sweeps=sweeps)


@pytest.mark.parametrize("options", [
    dict(smoother=_lib.SMOOTH_RBGS, coarse_operator=_lib.COARSE_GALERKIN),
    dict(smoother=_lib.SMOOTH_RBGS, coarse_operator=_lib.COARSE_GALERKIN, fine_sweeps=_lib.SWEEP_SINGLE),
    dict(smoother=_lib.SMOOTH_JACOBI, coarse_operator=_lib.COARSE_REDISCRETISED),
    dict(preconditioner=_lib.PRECOND_JACOBI),
], ids=["bricks", "single", "jacobi", "pcg"])
@pytest.mark.parametrize("size", [(64, 24, 40), (36, 20, 24), (128, 8, 16)], ids=str)
def test_blocks_that_fall_dry_and_wet_leave_no_trace(size, options):
    """Dry blocks are skipped: a solver whose surface falls and rises between
    projections gives the bits of a fresh one each time."""
    from fluidisim_amd.volume import Domain3, Volume3
    nx, ny, nz = size
    rng = np.random.default_rng(81)
    o = dict(preconditioner=_lib.PRECOND_MULTIGRID, max_levels=-1, pre_sweeps=2, post_sweeps=2, coarse_sweeps=4)
    o.update(options)
    faces = [(0.2 * rng.standard_normal(s)).astype(np.float32).ravel()
             for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]

    def volume():
        vol = Volume3.configure(Domain3(nx, ny, nz, 0.05), rho=1000.0, g_eff=9.81, **o)
        vol.set_surface_mode(False, False)
        return vol

    def project(vol, fill):
        # the lower part of the columns wet, a tenth of the columns dry
        eta = 0.05 * nz * fill * (rng_eta.random((ny, nx)) > 0.1) + 0.02
        vol.set_free_surface(eta.astype(np.float32).ravel(), 0.05 * nz * fill)
        vol.set_velocity(*faces)
        rep = vol.project_mobile3(-1e5, 1e-5, 500, rel_tol=1e-7, warm=False)
        return rep.iterations, [t.cpu().numpy().ravel() for t in (vol.pressure(), vol.velocity_u(), vol.velocity_v(),
                                                                  vol.velocity_w())]

    used = volume()
    for step, fill in enumerate((0.3, 0.9, 0.0, 0.2, 1.0, 0.5)):
        rng_eta = np.random.default_rng(step)
        it, got = project(used, fill)
        fresh = volume()
        rng_eta = np.random.default_rng(step)
        it_ref, ref = project(fresh, fill)
        fresh.close()
        assert it == it_ref
        for a, b in zip(got, ref):
            assert np.array_equal(bits(a), bits(b)), (step, fill)
    used.close()


@pytest.mark.parametrize("options", [
    dict(smoother=_lib.SMOOTH_RBGS, coarse_operator=_lib.COARSE_GALERKIN),
    dict(smoother=_lib.SMOOTH_RBGS, coarse_operator=_lib.COARSE_GALERKIN, fine_sweeps=_lib.SWEEP_SINGLE),
    dict(smoother=_lib.SMOOTH_JACOBI, coarse_operator=_lib.COARSE_REDISCRETISED),
], ids=["bricks", "single", "jacobi"])
@pytest.mark.parametrize("size", [(32, 24, 32), (128, 16, 32), (34, 24, 32)], ids=str)
@pytest.mark.parametrize("tuned", [False, True], ids=["tile", "tuned"])
def test_a_residual_on_air_is_restricted_with_the_rest(size, options, tuned):
    """The preconditioner's argument is any vector: on the dry layers just
    above the surface it reaches the second coarse level, whatever blocks the
    fine kernels are split into."""
    nx, ny, nz = size
    wl = W.tank(nx, nz, ny, seed=91)
    rng = np.random.default_rng(92)
    # layers 16 and below wet: 18 and 19 are dry beside wet ones in a cell of the second coarse level
    wl.eta = rng.uniform(17.1, 17.4, nx * ny).astype(np.float32)
    wl.options.update(options)
    vol = W.build_volume(wl)
    if tuned:
        vol.autotune()
    r = rng.uniform(-1.0, 1.0, wl.domain.cells).astype(np.float32)
    z = vol.precondition(torch.from_numpy(r).cuda()).cpu().numpy()
    vol.close()
    z_ref = po.vcycle(problem(wl), r, oracle_options(wl)).astype(np.float32)
    assert np.array_equal(bits(z), bits(z_ref)), f"max diff {np.abs(z - z_ref).max()}"


@pytest.mark.parametrize("form", ["bf16", "cut", "cut jacobi", "level set", "level set bf16", "learned v-cycle",
                                  "learned sweeps"])
def test_blocks_that_fall_dry_and_wet_leave_no_trace_in_any_form(form):
    """As above for the 16-bit vectors, the ghost-row index and flexible CG
    (which folds <A d, z> over dry cells too)."""
    from fluidisim_amd.volume import Domain3, Volume3
    nx, ny, nz, dx = 64, 24, 40, 0.05
    rng = np.random.default_rng(83)
    o = dict(preconditioner=_lib.PRECOND_MULTIGRID, smoother=_lib.SMOOTH_RBGS, max_levels=-1, pre_sweeps=2,
             post_sweeps=2, coarse_sweeps=4, coarse_operator=_lib.COARSE_GALERKIN)
    if "bf16" in form:
        o["vcycle_storage"] = _lib.STORE_BF16
    if "cut" in form:
        o["coarse_operator"] = _lib.COARSE_REDISCRETISED
    if "jacobi" in form:
        o["smoother"] = _lib.SMOOTH_JACOBI
    net = None
    if "learned" in form:
        from fluidisim_amd.learned import WEIGHTS, Network
        net = Network()
        net.load(WEIGHTS)
        o.update(preconditioner=_lib.PRECOND_LEARNED, learned_budget=8, learned_vcycle=int("v-cycle" in form))
    faces = [(0.2 * rng.standard_normal(s)).astype(np.float32)
             for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
    opens = []
    for axis, f in ((2, faces[0]), (1, faces[1]), (0, faces[2])):
        a = np.where(rng.random(f.shape) < 0.02, rng.uniform(0.3, 0.9, f.shape), 1.0).astype(np.float32)
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[axis], hi[axis] = 0, -1
        a[tuple(lo)] = 0
        f[tuple(lo)] = 0
        if axis:
            a[tuple(hi)] = 0
        f[tuple(hi)] = 0
        opens.append(a.ravel())
    faces = [f.ravel() for f in faces]

    def volume():
        vol = Volume3.configure(Domain3(nx, ny, nz, dx), rho=1000.0, g_eff=9.81, **o)
        vol.set_surface_mode(False, False)
        if net is not None:
            net.attach(vol)
        return vol

    def project(vol, step, fill):
        draw = np.random.default_rng(step)
        eta = (dx * (np.round(nz * fill) + draw.uniform(-0.4, 0.4, (ny, nx))) * (draw.random((ny, nx)) > 0.1) + 0.02)
        if "level set" in form:
            z = (np.arange(nz) + 0.5)[:, None, None] * dx
            phi = np.clip(z - eta[None], -2 * dx, 2 * dx).astype(np.float32)
            vol.set_level_set(np.where(phi < 0, _lib.LABEL_WATER, _lib.LABEL_AIR).astype(np.uint8).ravel(), phi.ravel())
        else:
            if "cut" in form:
                vol.set_solid(None, *opens)
            vol.set_free_surface(eta.astype(np.float32).ravel(), dx * nz * fill)
        vol.set_velocity(*faces)
        rep = vol.project_mobile3(-1e5, 1e-5, 300, rel_tol=1e-6, warm=False)
        return rep.iterations, [t.cpu().numpy().ravel() for t in (vol.pressure(), vol.velocity_u(), vol.velocity_v(),
                                                                  vol.velocity_w())]

    used = volume()
    for step, fill in enumerate((0.3, 0.9, 0.2, 0.7)):
        it, got = project(used, step, fill)
        fresh = volume()
        it_ref, ref = project(fresh, step, fill)
        fresh.close()
        assert it == it_ref and it > 0
        for a, b in zip(got, ref):
            assert np.array_equal(bits(a), bits(b)), (step, fill)
    used.close()


@pytest.mark.parametrize("size", [(34, 30, 28), (30, 30, 30)], ids=str)
@pytest.mark.parametrize("sweeps", [4, 7])
def test_an_odd_coarsest_level_over_64_kib_in_the_tail_matches_the_oracle(size, sweeps):
    """17 x 15 x 14 and 15^3 cells, 24 bytes of LDS each. (An aperture in the
    wall at +x keeps these widths out of the padded domain, whose levels have
    even rows.)"""
    nx, ny, nz = size
    wl = W.tank(nx, nz, ny, seed=101)
    d = wl.domain
    solid = np.asarray(wl.solid).reshape(nz, ny, nx) != 0
    opens = []
    for axis, shape in ((2, (nz, ny, nx + 1)), (1, (nz, ny + 1, nx)), (0, (nz + 1, ny, nx))):
        a = np.ones(shape, np.float32)
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[axis], hi[axis] = slice(0, -1), slice(1, None)
        a[tuple(lo)][solid] = 0
        a[tuple(hi)][solid] = 0
        lo[axis], hi[axis] = 0, -1
        a[tuple(lo)] = 0
        a[tuple(hi)] = 0
        opens.append(a)
    opens[0][:, :, nx] = ~solid[:, :, nx - 1]
    wl.open_u, wl.open_v, wl.open_w = [a.ravel() for a in opens]
    assert_vcycle_is_the_oracles(wl, max_levels=1, coarse_sweeps=sweeps)
    # in the tail: no pass over the level in a launch of its own
    vol = W.build_volume(wl)
    L = _lib.lib()
    assert L.fsp_profile_begin(vol._h, b"k_r6_gs", 64) == 0
    vol.precondition(torch.ones(d.cells, device="cuda"))
    n, total = C.c_uint32(), C.c_double()
    assert L.fsp_profile_end(vol._h, C.byref(n), C.byref(total), None, None, 0) == 0
    vol.close()
    assert n.value == 0
