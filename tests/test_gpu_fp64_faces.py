"""Both elements of an interface use one surface flux, so that what leaves one element enters the
other: FP64 flux_ranocha lines, whose own face states come from their node records."""
import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("surface", ["llf", "llf_naive"])
@pytest.mark.parametrize("volume", ["fd", "hg"])
@pytest.mark.parametrize("ndims,polydeg,level", [(2, 2, 3), (2, 3, 3), (2, 4, 3), (3, 2, 2), (3, 3, 2), (3, 4, 2)])
def test_interface_fluxes_cancel(ndims, polydeg, level, volume, surface):
    """Gas at rest, constant in each element: the volume terms of density and energy are zero, and
    at a node inside one face du is that face's dissipation alone, lambda (u_left - u_right) / 2
    times the same factor on both sides. With one lambda the two elements' values add up to zero
    exactly; with one that differs in the last place they do not."""
    spec = dict(ndims=ndims, polydeg=polydeg, level=level, cmin=(-1,) * ndims, cmax=(1,) * ndims, ic="constant",
                volume_integral=volume, surface_flux=surface)
    semi, _ = build(spec, "fp64")
    n, E, V = polydeg + 1, semi.nelements(), ndims + 2
    rng = np.random.default_rng(5)
    rho, p = rng.uniform(0.5, 2.0, (2, E))
    u = np.zeros((E, n ** ndims, V))
    u[:, :, 0] = rho[:, None]
    u[:, :, -1] = (p / (semi.equations.gamma - 1))[:, None]
    du = np.empty(u.size)
    th.rhs_hyperbolic_(du, np.ascontiguousarray(u).reshape(-1), semi, 0.0)
    du = du.reshape((E,) + (n,) * ndims + (V,))  # [e][k][j][i][v]
    inner = (slice(1, n - 1),) * (ndims - 1)
    left, right = semi.mesh.neighbor_ids.T
    for d in range(ndims):
        pick = semi.mesh.orientations == d
        a = np.moveaxis(du, ndims - d, 1)[left[pick], n - 1]  # last nodes of the left element
        b = np.moveaxis(du, ndims - d, 1)[right[pick], 0]
        for v in (0, V - 1):
            la, lb = a[(slice(None),) + inner + (v,)], b[(slice(None),) + inner + (v,)]
            assert np.all(np.abs(la) > 0)
            off = int(np.sum(la + lb != 0))
            print(f"{ndims}D p{polydeg} {volume} {surface} direction {d} value {v}: {off} of {la.size} do not cancel",
                  flush=True)
            assert off == 0
    semi.close()
