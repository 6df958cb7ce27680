"""rhs_hyperbolic_ in FP32 mode rounds its FP64 input on load and widens its result on store, inside the
element kernel and the kernels before it: the same bits as the RHS of the rounded array widened
afterwards, on every mesh kind, with partial tiles, and for arrays that overlap."""
import ctypes

import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build

pytestmark = pytest.mark.gpu

BOX2, BOX3 = ((-0.4, -0.4), (0.4, 0.4)), ((-0.5,) * 3, (0.5,) * 3)
CASES = {
    "2d_p2_partial_tile": dict(ndims=2, polydeg=2, level=3),
    "2d_p3_hg": dict(ndims=2, polydeg=3, level=3, volume_integral="hg"),
    "2d_p4_hg_mortars": dict(ndims=2, polydeg=4, level=3, volume_integral="hg", refinement_patches=(BOX2,)),
    "2d_p3_slip_mortars": dict(ndims=2, polydeg=3, level=2, periodicity=False, boundary_condition="slip_wall",
                               refinement_patches=(BOX2,)),
    "3d_p2_weak": dict(ndims=3, polydeg=2, level=1, volume_integral="weak"),
    "3d_p3_dirichlet_mortars": dict(ndims=3, polydeg=3, level=2, periodicity=False, refinement_patches=(BOX3,)),
    "3d_p4_hg": dict(ndims=3, polydeg=4, level=1, volume_integral="hg"),
}


@pytest.mark.parametrize("name", CASES)
def test_fp32_rhs_between_fp64_arrays_is_the_native_rhs(name):
    import torch
    d = CASES[name]["ndims"]
    spec = dict(cmin=(-1,) * d, cmax=(1,) * d, ic="convergence_test") | CASES[name]
    semi, _ = build(spec, "fp32")
    u0 = semi.compute_coefficients(0.1)
    rng = np.random.default_rng(5)
    u = torch.from_numpy(u0 * (1 + 0.05 * rng.uniform(-1, 1, u0.size))).cuda()
    u32 = u.float()
    du32 = torch.empty_like(u32)
    torch.cuda.synchronize()
    th._lib.check(semi._lib.trixi_hip_set_stream(semi.ctx, None), semi.ctx, "set_stream")
    th._lib.check(semi._lib.trixi_hip_rhs_native(semi.ctx, ctypes.c_void_p(du32.data_ptr()),
                                                 ctypes.c_void_p(u32.data_ptr()), 0.3), semi.ctx, "rhs_native")
    th._lib.check(semi._lib.trixi_hip_synchronize(semi.ctx), semi.ctx, "synchronize")
    want = du32.double()
    du = torch.full_like(u, float("nan"))
    th.rhs_hyperbolic_(du, u, semi, 0.3)
    assert torch.equal(du, want)
    th.rhs_hyperbolic_(u, u, semi, 0.3)  # in place
    assert torch.equal(u, want)
    semi.close()
