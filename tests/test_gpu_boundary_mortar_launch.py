"""Dirichlet boundaries that depend on time, on meshes with mortars: their states come from the
mortars' launch, again at every call."""
import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build, oracle_for

pytestmark = pytest.mark.gpu


# one mortar workgroup and several, boundary nodes below and above one workgroup, ends of both
@pytest.mark.parametrize("ndims,polydeg,level", [(2, 2, 2), (2, 3, 5), (2, 4, 3), (3, 2, 2), (3, 3, 2), (3, 4, 3)])
def test_states_follow_time(ndims, polydeg, level):
    """Criterion of the FP64 RHS parity tests: 1e-12 of max|du| against the oracle, on a state with
    1 % noise (du of the smooth one is a small difference of fluxes, whose rounding is not the subject)."""
    spec = dict(ndims=ndims, polydeg=polydeg, level=level, cmin=(0,) * ndims, cmax=(2,) * ndims,
                ic="convergence_test", source="convergence_test", periodicity=False,
                refinement_patches=[((0.5,) * ndims, (1.5,) * ndims)])
    o = oracle_for(spec)
    semi, _ = build(spec, "fp64")
    u = semi.compute_coefficients(0.1)
    u = u * (1 + 0.01 * np.random.default_rng(3).standard_normal(u.shape))
    du = np.empty_like(u)
    for t in (0.1, 0.7):
        th.rhs_hyperbolic_(du, u, semi, t)
        ref = o.rhs(u, t)
        err = float(np.max(np.abs(du - ref)) / np.max(np.abs(ref)))
        print(f"{ndims}D p{polydeg} t = {t}: relative error {err:.3e}", flush=True)
        assert err < 1e-12
    semi.close()
