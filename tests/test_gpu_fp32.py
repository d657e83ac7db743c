"""Errors that single precision must not have: shifts that grow with the length of a
sequence or with the size of the coordinates.  The references are the FP64 passes
(compared with the oracle elsewhere) or the FP64 oracle, on the same FP32-rounded
inputs.
"""
import numpy as np
import pytest
import torch

from oracle import psm_oracle as O

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

import parsmooth  # noqa: E402
from parsmooth import FunctionalModel, MVNSqrt  # noqa: E402
from parsmooth import models as M  # noqa: E402
from parsmooth.batch import IteratedSmoother  # noqa: E402
from parsmooth.data import bearings_data_batch, cv_model, lgssm_data  # noqa: E402
from parsmooth.linearization import cubature, extended, unscented  # noqa: E402

DEV = torch.device("cuda", 0)
DT = float(np.float32(0.01))
S1, S2 = (-1.5, 0.5), (1.0, 1.0)
npy = lambda x: x.detach().double().cpu().numpy()
r32 = lambda a: np.asarray(a, np.float32).astype(np.float64)


def turn_models(dtype, s1=S1, s2=S2):
    Q, R, obs_f, trans_f = M.make_parameters(0.01, 0.1, 0.5, DT, s1, s2)
    t = lambda a: torch.as_tensor(r32(a), device=DEV).to(dtype)
    return (FunctionalModel(trans_f, MVNSqrt(t(np.zeros(5)), t(np.linalg.cholesky(Q)))),
            FunctionalModel(obs_f, MVNSqrt(t(np.zeros(2)), t(np.linalg.cholesky(R)))))


@pytest.mark.parametrize("method", [cubature, unscented], ids=["cubature", "unscented"])
def test_loglikelihood_of_long_sequences(method):
    """The log-likelihood's error per step, one way for every sequence, is at most one
    FP32 rounding (2^-24): a step's term is a sum of values of about 1 whose roundings
    go both ways, and what does not average out is a factor of the model that is off
    the same way at every step."""
    T, B = 1000, 200
    rng = np.random.RandomState(0)
    x0 = np.array([3.0, 2.0, 1.0, 0.0]) + 0.3 * rng.randn(B, 4)
    states, obs = bearings_data_batch([T] * B, x0, DT, 0.5, S1, S2, q=3.16, seed=1)
    ys, m0 = np.concatenate(obs), np.stack([s[0] for s in states]) + 0.1 * rng.randn(B, 5)
    L0 = np.repeat(0.3 * np.eye(5)[None], B, 0)
    nom, ell = None, {}
    for dtype in (torch.float64, torch.float32):
        t = lambda a: torch.as_tensor(r32(a), device=DEV).to(dtype)
        run = IteratedSmoother([T] * B, *turn_models(dtype), method, dtype=dtype)
        run.set_data(t(ys), t(m0), t(L0))
        if nom is None:   # a nominal near the posterior, the same for both types
            mean, fac = run.run(2, (t(np.concatenate(states)), t(np.repeat(0.1 * np.eye(5)[None], B * (T + 1), 0))))
            nom = r32(npy(mean)), r32(npy(fac))
        ell[dtype] = npy(run.run(1, tuple(map(t, nom)), return_loglikelihood=True)[2])
    shift = np.median(ell[torch.float32] - ell[torch.float64]) / T
    assert abs(shift) <= 2.0 ** -24, shift


# the points' bearings on both sides of the negative x axis, where a bearing jumps by
# 2 pi, and far from the sensors
@pytest.mark.parametrize("mean", [(-6.0, 0.55), (-6.0, 0.4), (-6.0, 0.5), (-40.0, 1.02), (3.0, 2.0), (150.0, 90.0)])
def test_bearing_regression(mean):
    """F, the noise factor and b of one cubature regression.  F is the points' increments
    over their distances: FP32 leaves it 1e-5 of its size (the increments are sums of ten
    terms with errors of a few 2^-24 each, over factors whose condition is below 10)."""
    m = r32(np.array([*mean, 1.0, -0.5, 0.3]))
    L = r32(np.tril(0.1 + 0.05 * np.arange(25).reshape(5, 5) / 25) + 0.4 * np.eye(5))
    out = {}
    for dtype in (torch.float64, torch.float32):
        t = lambda a: torch.as_tensor(a, device=DEV).to(dtype)
        out[dtype] = [npy(a) for a in cubature(turn_models(dtype)[1], MVNSqrt(t(m), t(L)))]
    F = out[torch.float64][0]
    for a, b, size in zip(out[torch.float32], out[torch.float64], (0.0, 0.0, np.abs(F).max() * np.abs(m).max())):
        assert np.abs(a - b).max() <= 1e-5 * max(np.abs(b).max(), size), (a, b)


@pytest.mark.parametrize("method", [cubature, unscented], ids=["cubature", "unscented"])
def test_regressions_far_from_the_origin(method):
    """A filter pass on a track and its sensors moved by 4096 units: the coordinated
    turn and the bearings see no difference, and the nominal is on the grid of FP32
    numbers of that size, so that the move is exact.  The moved means have the rounding
    to that grid (half a spacing of 2^-11) on top of the passes' own 2e-5, the
    log-likelihood a few roundings of values of about 1 a step."""
    T, move, grid = 400, 4096.0, 2.0 ** -11
    states, obs = bearings_data_batch([T], [[3.0, 2.0, 1.0, 0.0]], DT, 0.5, S1, S2, q=3.16, seed=4)
    rng = np.random.RandomState(2)
    nm = states[0].astype(np.float64) + 0.03 * rng.randn(T + 1, 5)
    nm[:, :2] = np.round(nm[:, :2] / grid) * grid
    nL = np.repeat((0.3 * np.eye(5) + 0.02 * np.tril(np.ones((5, 5))))[None], T + 1, 0)
    t = lambda a: torch.as_tensor(r32(a), device=DEV).to(torch.float32)
    out = {}
    for at in (0.0, move):
        by = np.array([at, at, 0.0, 0.0, 0.0])
        models = turn_models(torch.float32, *(tuple(at + v for v in s) for s in (S1, S2)))
        nom = t(nm + by), t(nL)
        assert np.array_equal(npy(nom[0]), r32(nm) + by)
        filt, ell = parsmooth.filtering(t(obs[0]), MVNSqrt(t(nm[0] + by), t(0.3 * np.eye(5))), *models, method, MVNSqrt(*nom),
                                        return_loglikelihood=True)
        out[at] = npy(filt.mean) - by, npy(filt.chol), float(ell)
    (m0, f0, e0), (m1, f1, e1) = out[0.0], out[move]
    np.testing.assert_allclose(m1, m0, rtol=0, atol=0.5 * grid + 2e-5)
    np.testing.assert_allclose(f1, f0, rtol=0, atol=1e-5)
    assert abs(e1 - e0) <= T * 4 * 2.0 ** -24, (e1, e0)


NOMINALS = {"near": lambda x: x, "far": lambda x: x + 1e4, "farther": lambda x: -1e6 + 0 * x,
            "nan": lambda x: np.where(np.arange(len(x))[:, None] % 7 == 3, np.nan, x),
            "infinite": lambda x: np.where(np.arange(len(x))[:, None] % 2 == 0, np.inf, -np.inf) + 0 * x}


@pytest.mark.parametrize("nominal", NOMINALS)
def test_linear_models_do_not_use_the_nominal(nominal):
    """A linear model under the extended rule does not depend on the nominal: neither a
    far one nor one that is not finite may cost its result anything.  Bounds: FP32
    means and factors are held to 2^-24 of their size, and a pass adds a few tens of
    such errors: 2e-6."""
    T = 700
    F, Q, H, R = (r32(a) for a in cv_model())
    cQ, cR = r32(np.linalg.cholesky(Q)), r32(np.linalg.cholesky(R))
    m0, L0 = r32([30.0, -20.0, 1.0, 2.0]), r32(np.eye(4))
    x, ys = (r32(a) for a in lgssm_data(m0, F, H, cR @ cR.T, cQ @ cQ.T, np.zeros(4), np.zeros(2), T, random_state=3))
    to, oo = O.FunctionalModel(O.Linear(F), O.MVNSqrt(np.zeros(4), cQ)), O.FunctionalModel(O.Linear(H), O.MVNSqrt(np.zeros(2), cR))
    f, ell = O.filtering(ys, O.MVNSqrt(m0, L0), to, oo, O.extended, None, True, return_loglikelihood=True)
    ref = O.smoothing(to, f, O.extended, None, True)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=DEV)
    td = FunctionalModel(M.LinearFunction(t(F)), MVNSqrt(t(np.zeros(4)), t(cQ)))
    od = FunctionalModel(M.LinearFunction(t(H)), MVNSqrt(t(np.zeros(2)), t(cR)))
    x0, nom = MVNSqrt(t(m0), t(L0)), MVNSqrt(t(NOMINALS[nominal](x)), t(np.tile(np.eye(4), (T + 1, 1, 1))))

    def near(got, want, what):
        got, want = npy(got), np.asarray(want)
        assert np.abs(got - want).max() <= 2e-6 * np.abs(want).max(), (nominal, what, np.abs(got - want).max())

    fd, ell_d = parsmooth.filtering(t(ys), x0, td, od, extended, nom, return_loglikelihood=True)
    near(fd.mean, f[0], "filtered mean")
    near(ell_d, ell, "log-likelihood")
    exact = MVNSqrt(t(f[0]), t(f[1]))
    near(parsmooth.smoothing(td, exact, extended, nom).mean, O.smoothing(to, O.MVNSqrt(r32(f[0]), r32(f[1])), O.extended, None, True)[0],
         "smoothed mean")
    post = parsmooth.filter_smoother(t(ys), x0, td, od, extended, nom)
    near(post.mean, ref[0], "mean of the joint pass")
    for k in (2, 3):
        post = parsmooth.iterated_smoothing(t(ys), x0, td, od, extended, nom, criterion=parsmooth.FixedIterations(k))
        near(post.mean, ref[0], f"{k} iterations")
    eps = np.random.RandomState(1).randn(T + 1, 3, 4)
    near(parsmooth.sampling(t(eps), 3, td, exact, extended, nom),
         O.sampling(r32(eps), to, O.MVNSqrt(r32(f[0]), r32(f[1])), O.extended, O.MVNSqrt(f[0], f[1])), "samples")


def test_unused_nominal_components():
    """The coordinated turn with positions observed linearly uses the nominal's
    velocity and turn rate only: its positions may be anything."""
    T = 300
    states, _ = bearings_data_batch([T], [[3.0, 2.0, 1.0, 0.0]], DT, 0.5, S1, S2, q=3.16, seed=5)
    x = states[0].astype(np.float64)
    t = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=DEV)
    ys = t(x[1:, :2] + 0.1 * np.random.RandomState(0).randn(T, 2))
    od = FunctionalModel(M.LinearFunction(t(np.eye(2, 5))), MVNSqrt(t(np.zeros(2)), t(0.1 * np.eye(2))))
    x0, L = MVNSqrt(t(x[0]), t(0.3 * np.eye(5))), t(np.tile(0.1 * np.eye(5), (T + 1, 1, 1)))
    out = []
    for fill in (0.0, np.nan):
        nm = x.copy()
        nm[:, :2] = fill
        out.append(parsmooth.filter_smoother(ys, x0, turn_models(torch.float32)[0], od, extended, MVNSqrt(t(nm), L)))
    assert torch.equal(out[0].mean, out[1].mean) and torch.equal(out[0].chol, out[1].chol)
