"""The three forms of the means in the FP64 flux_ranocha lines: a series where the line's
densities and temperatures differ by at most a factor (23/17)^2 = 1.83, a longer one up to a factor 4,
logarithms beyond. Each line takes its own form; the wavefront's path serves all its lines."""
import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build, oracle_for

pytestmark = pytest.mark.gpu

# 1 + 1e-9: differences far below the sums; 1.2: the short series; 3: both series; 6: all three
# forms; 50: a strong shock in almost every pair
FACTORS = [1 + 1e-9, 1.2, 3.0, 6.0, 50.0]


@pytest.mark.parametrize("factor", FACTORS)
@pytest.mark.parametrize("volume", ["fd", "hg"])
@pytest.mark.parametrize("ndims,polydeg,level", [(2, 2, 3), (2, 3, 3), (2, 4, 2), (3, 2, 1), (3, 3, 1), (3, 4, 1)])
def test_fp64_volume_flux_means(ndims, polydeg, level, volume, factor):
    """Node values of density and temperature drawn between 1 and `factor`; for factor 50 in the last
    element of the mesh only, 1.1 elsewhere, so that one tile mixes the forms (2D levels 2 and 3
    end in partial tiles for polydeg 2 and 4). Criterion of the FP64 RHS parity tests: 1e-12 of
    max|du| against the oracle."""
    spec = dict(ndims=ndims, polydeg=polydeg, level=level, cmin=(-1,) * ndims, cmax=(1,) * ndims, ic="constant",
                volume_integral=volume, surface_flux="llf")
    o = oracle_for(spec)
    semi, _ = build(spec, "fp64")
    rng = np.random.default_rng(23)
    E, NN = semi.nelements(), semi.nnodes() ** ndims
    spread = np.full((E, 1), factor)
    if factor == 50.0:
        spread[:-1] = 1.1
    rho = 1 + (spread - 1) * rng.uniform(size=(E, NN))
    T = 1 + (spread - 1) * rng.uniform(size=(E, NN))
    v = 0.3 * rng.uniform(-1, 1, (E, NN, ndims))
    prim = np.concatenate([rho[..., None], v, (rho * T)[..., None]], axis=-1)
    u = np.ascontiguousarray(semi.equations.prim2cons(prim)).reshape(-1)
    du = np.empty_like(u)
    th.rhs_hyperbolic_(du, u, semi, 0.0)
    ref = o.rhs(u, 0.0)
    err = float(np.max(np.abs(du - ref)) / np.max(np.abs(ref)))
    print(f"{ndims}D p{polydeg} {volume} factor {factor:g}: relative error {err:.3e}", flush=True)
    assert err < 1e-12
    semi.close()
