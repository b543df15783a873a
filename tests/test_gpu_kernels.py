"""Kernel forms at the sizes where they change, against the oracle: the
V-cycle bit for bit (both sides do the same arithmetic in the same order)."""
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
])
def test_tail_levels_match_the_oracle(size, levels, sweeps):
    wl = W.tank(*size, seed=21)
    assert_vcycle_is_the_oracles(wl, max_levels=levels, pre_sweeps=sweeps[0], post_sweeps=sweeps[1],
                                 coarse_sweeps=sweeps[2])
