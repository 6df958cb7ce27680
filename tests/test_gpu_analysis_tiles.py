"""Error norms and integrals at the edges of their launches: partial tiles, one tile, several tiles
to a workgroup, both compilations of the exact solution, NaN in the state."""
import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build, oracle_for

pytestmark = pytest.mark.gpu

# elements for each workgroup of the error norms: 3D 10, 5, 3 and 2D 51, 36, 28 for polydeg 2, 3, 4
MESHES = [(2, 2, 2), (2, 3, 3), (2, 4, 1), (3, 2, 1), (3, 3, 1), (3, 4, 2), (2, 3, 8)]


def _analyze(spec, t, nan=False):
    o = oracle_for(spec)
    o.set_initial_condition(spec["ic"], spec.get("ic_params", ()))
    semi, _ = build(spec, "fp64")
    u = semi.compute_coefficients(0.0)
    u = u * (1 + 0.01 * np.random.default_rng(5).standard_normal(u.shape))
    if nan:
        u[semi.nvariables() - 1] = np.nan  # the energy of the first node
    semi._lib.trixi_hip_upload_u(semi.ctx, u.ctypes.data)
    rec = th.AnalysisCallback(semi).analyze(t, 0)
    semi.close()
    return rec, o.error_norms(u, t), o.integrals(u)


# the bounds of the solver tests' norms: sums to 1e-11, maxima and integrals to 1e-12
@pytest.mark.parametrize("ndims,polydeg,level", MESHES)
@pytest.mark.parametrize("ic", ["convergence_test", "density_pulse", "weak_blast_wave"])
def test_norms_and_integrals_match_oracle(ndims, polydeg, level, ic):
    spec = dict(ndims=ndims, polydeg=polydeg, level=level, cmin=(-2,) * ndims, cmax=(2,) * ndims, ic=ic)
    rec, (l2, linf), (cons, ent) = _analyze(spec, 0.25)
    np.testing.assert_allclose(rec["l2"], l2, rtol=1e-11)
    np.testing.assert_allclose(rec["linf"], linf, rtol=1e-12)
    # integrals of the velocities' momenta can cancel: to 1e-12 of the largest
    np.testing.assert_allclose(rec["integrals"], cons, rtol=1e-12, atol=1e-12 * np.max(np.abs(cons)))
    assert rec["entropy"] == pytest.approx(ent, rel=1e-12)


@pytest.mark.parametrize("ndims", [2, 3])
def test_nan_stays_in_its_variable(ndims):
    spec = dict(ndims=ndims, polydeg=3, level=2, cmin=(0,) * ndims, cmax=(2,) * ndims, ic="convergence_test")
    rec, (l2, linf), _ = _analyze(spec, 0.25, nan=True)
    assert np.isnan(rec["l2"][-1]) and np.isnan(rec["linf"][-1]) and np.isnan(rec["entropy"])
    np.testing.assert_allclose(rec["l2"][:-1], l2[:-1], rtol=1e-11)
    np.testing.assert_allclose(rec["linf"][:-1], linf[:-1], rtol=1e-12)
