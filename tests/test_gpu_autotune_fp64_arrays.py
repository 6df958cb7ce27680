"""After autotuning, an FP32 context's RHS between FP64 arrays runs on the chosen tile, as the native RHS does."""
import ctypes

import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [dict(ndims=3, polydeg=3, level=2), dict(ndims=2, polydeg=3, level=4, volume_integral="hg"),
                                  dict(ndims=2, polydeg=2, level=3, periodicity=False)])
def test_rhs_between_fp64_arrays_after_autotuning(spec):
    import torch
    d = spec["ndims"]
    semi, _ = build(dict(cmin=(-1,) * d, cmax=(1,) * d, ic="convergence_test") | spec, "fp32")
    u0 = semi.compute_coefficients(0.0)
    before, after = np.empty_like(u0), np.empty_like(u0)
    th.rhs_hyperbolic_(before, u0, semi, 0.2)
    n = ctypes.c_int(0)
    th._lib.check(semi._lib.trixi_hip_autotune(semi.ctx, 2, None, 0, ctypes.byref(n)), semi.ctx, "autotune")
    assert n.value >= 1
    th.rhs_hyperbolic_(after, u0, semi, 0.2)
    assert np.array_equal(after, before)
    u = torch.from_numpy(u0).cuda()
    du = torch.full_like(u, float("nan"))
    th.rhs_hyperbolic_(du, u, semi, 0.2)
    assert np.array_equal(du.cpu().numpy(), before)
    semi.close()
