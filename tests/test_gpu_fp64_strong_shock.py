"""FP64 flux_ranocha lines whose nodes differ much (logarithms) beside lines whose nodes do not (series).

A wavefront holds lines of several elements, and takes the path that serves them all. What a pair
of nodes gives must not depend on that path, so each element is judged by its own size."""
import numpy as np
import pytest

import trixi_hip as th
from gpu_helpers import build, oracle_for

pytestmark = pytest.mark.gpu

MESHES = [(2, 2, 3), (2, 3, 3), (2, 4, 2), (3, 2, 2), (3, 3, 2), (3, 4, 2)]
EPS = np.finfo(np.float64).eps


def set_up(ndims, polydeg, level, volume):
    spec = dict(ndims=ndims, polydeg=polydeg, level=level, cmin=(-1,) * ndims, cmax=(1,) * ndims, ic="constant",
                volume_integral=volume, surface_flux="llf")
    semi, _ = build(spec, "fp64")
    return spec, semi


def draw(semi, spread, scale_rho=1.0, scale_T=1.0, seed=29):
    """Conservative state [E, NN, V]; density and temperature of element e between 1 and spread[e]."""
    D, E = semi.mesh.ndims, semi.nelements()
    NN = semi.nnodes() ** D
    rng = np.random.default_rng(seed)
    s = np.broadcast_to(np.asarray(spread, dtype=np.float64), (E,))[:, None]
    rho = scale_rho * s ** rng.uniform(size=(E, NN))
    T = scale_T * s ** rng.uniform(size=(E, NN))
    v = 0.3 * np.sqrt(scale_T) * rng.uniform(-1, 1, (E, NN, D))
    prim = np.concatenate([rho[..., None], v, (rho * T)[..., None]], axis=-1)
    return np.ascontiguousarray(semi.equations.prim2cons(prim))


def rhs(semi, u):
    du = np.empty(u.size)
    th.rhs_hyperbolic_(du, np.ascontiguousarray(u).reshape(-1), semi, 0.0)
    return du.reshape(u.shape)


def term_size(semi, u):
    """Per element and variable: the largest term of du, J^-1 max|flux|, over the element and its
    face neighbours (whose states its surface fluxes hold, with their wave speeds)."""
    w = semi.equations.cons2prim(u.reshape(-1, u.shape[-1])).reshape(u.shape)
    v, p = np.abs(w[..., 1:-1]).max(axis=-1), w[..., -1]
    speed = v + np.sqrt(semi.equations.gamma * p / w[..., 0])
    f = speed[..., None] * np.abs(u) + p[..., None] * np.concatenate(
        [np.zeros_like(v)[..., None], np.ones_like(u[..., 1:-1]), v[..., None]], axis=-1)
    # a momentum may vanish where its flux does not: its density times the speed
    f[..., 1:-1] = np.maximum(f[..., 1:-1], (speed ** 2 * u[..., 0])[..., None])
    f = f.max(axis=1)
    return semi.inverse_jacobian[:, None] * np.maximum(f, f[semi.mesh.element_neighbors].max(axis=1))


# Round-off of one du value in units of term_size: per direction the volume terms, sum_j |Dsplit_ij|
# |f_ij|, at most 36 (polydeg 4, end node) with few roundings each, and 1/w = 10 for the face; three
# directions, GPU and oracle each. 200, as the free-stream tests use.
BOUND = 200 * EPS


@pytest.mark.parametrize("volume", ["fd", "hg"])
@pytest.mark.parametrize("ndims,polydeg,level", MESHES)
def test_strong_element_among_ordinary_ones(ndims, polydeg, level, volume):
    """One element with a factor 50 between its nodes, 1.1 elsewhere. Every element against the oracle at
    its own size (not with shock capturing, whose blending factor's own conditioning adds to the terms'
    round-off); the elements that share no face with the strong one bit for bit as without it."""
    spec, semi = set_up(ndims, polydeg, level, volume)
    E = semi.nelements()
    strong = E - 2
    spread = np.full(E, 1.1)
    plain = draw(semi, spread)
    spread[strong] = 50.0
    u = plain.copy()
    u[strong] = draw(semi, spread)[strong]
    du, du_plain = rhs(semi, u), rhs(semi, plain)
    if volume == "fd":
        ref = oracle_for(spec).rhs(u.reshape(-1), 0.0).reshape(u.shape)
        err = np.abs(du - ref).max(axis=1) / term_size(semi, u)
        print(f"{ndims}D p{polydeg}: largest error {err.max() / EPS:.1f} eps of the terms", flush=True)
        assert err.max() < BOUND
    apart = np.ones(E, dtype=bool)
    apart[strong] = False
    apart[semi.mesh.element_neighbors[strong]] = False
    assert np.array_equal(du[apart], du_plain[apart])
    assert not np.array_equal(du[strong], du_plain[strong])
    semi.close()


@pytest.mark.parametrize("scales", [(1.0, 1.0), (1e-6, 1e5)])
@pytest.mark.parametrize("factor", [1.69, 1.71, 2.5, 1e3, 1e8])
@pytest.mark.parametrize("ndims,polydeg,level", MESHES)
def test_every_pair_apart(ndims, polydeg, level, factor, scales):
    """Node values between 1 and `factor` in every element, around the ranges of the series and far
    beyond, also in units in which the values are far from 1."""
    spec, semi = set_up(ndims, polydeg, level, "fd")
    u = draw(semi, factor, *scales)
    ref = oracle_for(spec).rhs(u.reshape(-1), 0.0).reshape(u.shape)
    err = np.abs(rhs(semi, u) - ref).max(axis=1) / term_size(semi, u)
    print(f"{ndims}D p{polydeg} factor {factor:g} scales {scales}: {err.max() / EPS:.1f} eps", flush=True)
    assert err.max() < BOUND
    semi.close()


@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("what", ["density", "pressure", "both", "nan"])
@pytest.mark.parametrize("ndims,polydeg,level", MESHES)
def test_negative_values_give_nan(ndims, polydeg, level, what, whole):
    """A negative density or pressure, or NaN, at one node or in a whole element: NaN in the energy at that node
    (or all of them), nothing in the elements that share no face with it."""
    _, semi = set_up(ndims, polydeg, level, "fd")
    E, NN = semi.nelements(), semi.nnodes() ** ndims
    u = draw(semi, 1.1)
    plain = rhs(semi, u)
    bad, node = E - 2, NN // 2
    at = slice(None) if whole else node
    u[bad, at, 1:-1] = 0
    if what in ("density", "both"):
        u[bad, at, 0] *= -1
    if what in ("pressure", "both"):
        u[bad, at, -1] *= -1
    if what == "nan":
        u[bad, at, -1] = np.nan
    du = rhs(semi, u)
    assert np.all(np.isnan(du[bad, at, -1]))
    apart = np.ones(E, dtype=bool)
    apart[bad] = False
    apart[semi.mesh.element_neighbors[bad]] = False
    assert np.array_equal(du[apart], plain[apart])
    semi.close()
