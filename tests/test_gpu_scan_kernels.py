"""The scan kernels at the sizes where their levels, chunks and groups end: every
number of lanes per combination, both forms, FP64 and FP32, against the FP64
oracle; the sampler's and the adjoint's chunk edges; the log-likelihood sum.

Tolerances: as in the other parity tests, FP64 1e-9 relative to max(1,
|reference|) (one pass over at most 4,100 states of a contracting system: about
4,100 x 2^-53 x a condition number below 1e3), FP32 1e-4 for means and 1e-3 for
covariances against the oracle on the same FP32-rounded inputs.
"""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import psm_oracle as O

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a HIP device", allow_module_level=True)

import parsmooth  # noqa: E402
from parsmooth import FunctionalModel, MVNSqrt, MVNStandard  # noqa: E402
from parsmooth import models as M  # noqa: E402
from parsmooth import _native as N  # noqa: E402
from parsmooth.batch import IteratedSmoother  # noqa: E402
from parsmooth.linearization import cubature, extended, gauss_hermite, unscented  # noqa: E402

DEV = torch.device("cuda", 0)
ROW, QUAD = N.SCAN_TEAM | N.SCAN_ROW, N.SCAN_TEAM | N.SCAN_QUAD
npy = lambda x: x.detach().double().cpu().numpy()


def gram(L):
    return L @ np.swapaxes(L, -1, -2)


def close(a, b, tol, what):
    err = float(np.abs(a - b).max()) / max(1.0, float(np.abs(b).max()))
    assert err <= tol, f"{what}: rel err {err:.3e} > {tol:.1e}"


def problem(nx, ny, lengths, seed, dtype):
    """A ragged batch of one contracting linear model; prior factors are square
    roots without a triangle of zeros."""
    rng = np.random.RandomState(seed)
    rd = (lambda a: np.asarray(a, np.float32).astype(np.float64)) if dtype == torch.float32 else np.asarray
    F = rd(0.95 * np.linalg.qr(rng.randn(nx, nx))[0])
    H = rd(rng.randn(ny, nx) / np.sqrt(nx))
    cQ = rd(0.3 * np.eye(nx) + 0.1 * np.tril(rng.rand(nx, nx)))
    cR = rd(0.4 * np.eye(ny) + 0.1 * np.tril(rng.rand(ny, ny)))
    b, c = rd(0.1 * rng.randn(nx)), rd(0.1 * rng.randn(ny))
    S = len(lengths)
    m0 = rd(rng.randn(S, nx))
    L0 = rd(np.eye(nx)[None] + 0.2 * rng.randn(S, nx, nx))
    obs = [rd(O.lgssm_data(m0[s], F, H, gram(cR), gram(cQ), b, c, T, random_state=seed + s)[1])
           for s, T in enumerate(lengths)]
    return F, cQ, b, H, cR, c, m0, L0, obs


def check_pass(nx, ny, lengths, sqrt, dtype, schedules, seed=0, sequential=False, method=extended):
    F, cQ, b, H, cR, c, m0, L0, obs = problem(nx, ny, lengths, seed, dtype)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=DEV).to(dtype)
    cov = (lambda L: L) if sqrt else gram
    cls_o, cls = (O.MVNSqrt, MVNSqrt) if sqrt else (O.MVNStandard, MVNStandard)
    to = O.FunctionalModel(O.Linear(F), cls_o(b, cov(cQ)))
    oo = O.FunctionalModel(O.Linear(H), cls_o(c, cov(cR)))
    td = FunctionalModel(M.LinearFunction(t(F)), cls(t(b), t(cov(cQ))))
    od = FunctionalModel(M.LinearFunction(t(H)), cls(t(c), t(cov(cR))))
    refs, ells = [], []
    for s, y in enumerate(obs):
        f, ell = O.filtering(y, cls_o(m0[s], cov(L0[s])), to, oo, O.extended, None, True, return_loglikelihood=True)
        refs.append(O.smoothing(to, f, O.extended, None, True))
        ells.append(ell)
    tm, tc, te = (1e-9, 1e-9, 1e-9) if dtype == torch.float64 else (1e-4, 1e-3, 1e-3)
    n = sum(T + 1 for T in lengths)
    counts = []
    for sch in schedules:
        r = IteratedSmoother(list(lengths), td, od, method, sqrt=sqrt, dtype=dtype, sequential=sequential)
        if sch is not None:
            r.prob.set_schedule(*sch)
        r.set_data(t(np.concatenate(obs)), t(m0), t(cov(L0)))
        nom = (t(np.zeros((n, nx))), t(np.tile(np.eye(nx), (n, 1, 1))))
        mean, fac, ell = r.run(1, nom, use_graph=False, return_loglikelihood=True)
        gm, gL = r.split(mean), r.split(fac)
        for s, ref in enumerate(refs):
            what = f"nx {nx} ny {ny} {'sqrt' if sqrt else 'cov'} {lengths} {sch} seq {s}"
            close(npy(gm[s]), ref[0], tm, what + " mean")
            close(gram(npy(gL[s])) if sqrt else npy(gL[s]), gram(ref[1]) if sqrt else ref[1], tc, what + " cov")
            close(npy(ell)[s], np.asarray(ells[s]), te, what + " log-likelihood")
        counts.append(r.fallback_count())
    return counts


# chunk 1, so that the level edges (1, 16, 256, 4096 items of one, two, three and
# four levels, and one item more) are numbers of states
@pytest.mark.parametrize("states", [2, 15, 16, 17, 255, 256, 257, 4096, 4097])
@pytest.mark.parametrize("sqrt", [True, False])
def test_level_edges(states, sqrt):
    check_pass(2, 1, [states - 1], sqrt, torch.float64, [None, (1, 1 | ROW), (1, 2 | ROW), (3, 4 | ROW)])


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 2), (3, 1), (4, 2), (5, 2), (6, 3), (7, 4), (8, 4)])
@pytest.mark.parametrize("sqrt", [True, False])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["fp64", "fp32"])
def test_state_dimensions(nx, ny, sqrt, dtype):
    """Ragged sequences, with a sequence inside a chunk, through every kernel: the
    default, 16 lanes, four lanes, one lane."""
    check_pass(nx, ny, [200, 1, 2, 77], sqrt, dtype,
               [None, (1, 1 | ROW), (2, 2 | ROW), (4, 2 | QUAD), (4, 2 | QUAD | N.SCAN_HALF), (4, 2)], seed=nx)


@pytest.mark.parametrize("lengths", [[127] * 3, [128] * 3, [129, 1, 300], [2047], [2049, 2049]], ids=str)
def test_loglikelihood_blocks(lengths):
    """The log-likelihood sum at the mean lengths where its block size changes."""
    check_pass(1, 1, lengths, True, torch.float64, [None])


# 2 nx and 2 nx + 1 points are staged, 3 ** nx are not (nx > 1); the exact
# regression of a linear model is the model, so the oracle's Taylor form is the
# reference; the spread of the unit nominal covariance is that of the noise
@pytest.mark.parametrize("method", [cubature, unscented, gauss_hermite], ids=["cubature", "unscented", "gauss_hermite"])
@pytest.mark.parametrize("nx,ny", [(1, 2), (2, 1), (3, 3), (5, 2)])
def test_fp32_regression(method, nx, ny):
    check_pass(nx, ny, [40, 3], True, torch.float32, [None], seed=3, method=method)


# 64 sequences per workgroup, up to three steps a round: lengths off whole rounds,
# workgroups off whole ones, and the dimensions at which one, two and three steps fit
@pytest.mark.parametrize("nseq,nx,ny", [(1, 2, 1), (63, 2, 1), (64, 1, 1), (65, 3, 2), (130, 2, 1), (3, 5, 2),
                                        (3, 6, 3), (3, 7, 4), (3, 8, 4)])
@pytest.mark.parametrize("sqrt", [True, False])
def test_sequential_ahead(nseq, nx, ny, sqrt):
    """The sequential passes at a nominal trajectory, whose linearizations run
    ahead of the recursion."""
    lengths = [1 + (5 * s + 2) % 11 for s in range(nseq)]
    check_pass(nx, ny, lengths, sqrt, torch.float64, [None], seed=nseq, sequential=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n_states", [1, 4096, 4097, 8192, 8193, 12288, 12289, 24576, 24577, 1 << 21, 1 << 22])
def test_states_per_chunk(n_states, dtype):
    """The chunk rule at its lines: chunks as it says, for a problem as it is made and
    after set_schedule(0, 0), and a pass of the shorter ones agrees with the oracle
    (test_level_edges does the short ones)."""
    from parsmooth._engine import Problem, states_per_chunk
    want = {1: 1, 4096: 1, 4097: 2, 8192: 2, 8193: 3, 12288: 3, 12289: 2, 24576: 3, 24577: 0, 1 << 21: 24, 1 << 22: 40}
    assert states_per_chunk(n_states) == want[n_states]
    if n_states > 1:
        p = Problem(2, 1, [n_states - 1], dtype, True, DEV)
        small = dtype == torch.float32 and n_states >= 1 << 21   # two FP32 words a state: the library's choice
        assert p.struct.chunk == (0 if small else want[n_states])
        assert p.state_offsets.tolist() == [0, n_states]
        p.set_schedule(5, 2)
        assert (p.struct.chunk, p.struct.scan_k) == (5, 2)
        p.set_schedule(0, 0)
        assert (p.struct.chunk, p.struct.scan_k) == (0 if small else want[n_states], 0)
    if n_states in (8193, 12289):
        check_pass(2, 1, [n_states - 1], True, dtype, [None])


# chunks of 16, 24 and 32 states; 255 / 257 and 4095 / 4097 are one item off whole
# groups and off the next chunk size
@pytest.mark.parametrize("states", [2, 16, 17, 255, 256, 257, 4095, 4096, 4097])
@pytest.mark.parametrize("sqrt,samples", [(True, 1), (True, 67), (False, 3)])
def test_sampling_chunks(states, sqrt, samples):
    nx, T = 3, states - 1
    F, cQ, b, H, cR, c, m0, L0, obs = problem(nx, 2, [T], 3, torch.float64)
    cov = (lambda L: L) if sqrt else gram
    cls_o, cls = (O.MVNSqrt, MVNSqrt) if sqrt else (O.MVNStandard, MVNStandard)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=DEV)
    to = O.FunctionalModel(O.Linear(F), cls_o(b, cov(cQ)))
    oo = O.FunctionalModel(O.Linear(H), cls_o(c, cov(cR)))
    filt = O.filtering(obs[0], cls_o(m0[0], cov(L0[0])), to, oo, O.extended, None, True)
    eps = np.random.RandomState(1).randn(states, samples, nx)
    ref = O.sampling(eps, to, filt, O.extended, filt)
    td = FunctionalModel(M.LinearFunction(t(F)), cls(t(b), t(cov(cQ))))
    got = parsmooth.sampling(t(eps), samples, td, cls(t(filt[0]), t(filt[1])), extended, cls(t(filt[0]), t(filt[1])))
    # the recursion uses the noise factors themselves; a filtered factor of the
    # oracle is lower triangular with a positive diagonal, as the kernels' are
    close(npy(got), ref, 1e-9, f"{states} states, {samples} samples")


@pytest.mark.parametrize("states", [2, 17, 257])
def test_sampling_of_any_factors(states):
    """Filtered factors that are square roots without a triangle of zeros: the last
    state's draw is its mean and that factor times the normals, as it stands."""
    nx, T, samples = 3, states - 1, 5
    F, cQ, b, H, cR, c, m0, L0, obs = problem(nx, 2, [T], 5, torch.float64)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=DEV)
    to = O.FunctionalModel(O.Linear(F), O.MVNSqrt(b, cQ))
    oo = O.FunctionalModel(O.Linear(H), O.MVNSqrt(c, cR))
    filt = O.filtering(obs[0], O.MVNSqrt(m0[0], L0[0]), to, oo, O.extended, None, True)
    turned = filt[1] @ np.linalg.qr(np.random.RandomState(2).randn(states, nx, nx))[0]
    filt = O.MVNSqrt(filt[0], turned)
    eps = np.random.RandomState(1).randn(states, samples, nx)
    ref = O.sampling(eps, to, filt, O.extended, filt)
    traj = MVNSqrt(t(filt[0]), t(turned))
    got = parsmooth.sampling(t(eps), samples, FunctionalModel(M.LinearFunction(t(F)), MVNSqrt(t(b), t(cQ))), traj, extended, traj)
    close(npy(got), ref, 1e-9, f"{states} states")


GUARDED = """
import sys
sys.path[:0] = {path!r}
import torch
from tests.test_gpu_scan_kernels import N, ROW, QUAD, check_pass, extended, cubature
from parsmooth import set_fp32_fallback
set_fp32_fallback(1.0)
for method in (extended, cubature):
    count = check_pass(5, 2, [1500, 1, 700], True, torch.float32,
                       [None, (1, 1 | ROW), (2, 2 | QUAD), (2, 2 | QUAD | N.SCAN_HALF), (2, 2), (4, 2)], seed=8, method=method)
    print(method.__name__, "recomputed", count, flush=True)
    assert all(n > 0 for n in count)
print("guarded launches agree")
"""


def test_guarded_recomputation():
    """Every kernel of an FP32 pass as the pair of launches that large problems take
    (PSM_FB_SINGLE_WAVES=0, read once per process), with the threshold at which every
    check raises its flag: the second launches run, on 1, 4 and 16 lanes a
    combination, find their inputs as the first had them, and count."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = GUARDED.format(path=[root, os.path.join(root, "sqrt-parallel-smoothers_amd")])
    out = subprocess.run([sys.executable, "-c", code], env={**os.environ, "PSM_FB_SINGLE_WAVES": "0"}, cwd=root,
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and "guarded launches agree" in out.stdout, out.stdout + out.stderr


def _build(theta, nx=2):
    q, r, a = torch.exp(theta[0]), torch.exp(theta[1]), theta[2]
    eye = torch.eye(nx, dtype=theta.dtype)
    return {"trans_params": (0.9 * eye + a * torch.diag(torch.ones(nx - 1, dtype=theta.dtype), 1)).reshape(-1),
            "trans_q_mean": torch.zeros(nx, dtype=theta.dtype), "trans_q_chol": torch.sqrt(q) * eye,
            "obs_params": eye[:1].reshape(-1), "obs_q_mean": torch.zeros(1, dtype=theta.dtype),
            "obs_q_chol": torch.sqrt(r).reshape(1, 1), "m0": torch.zeros(1, nx, dtype=theta.dtype), "L0": eye[None]}


# one, two and three levels of chunks of 8 states, and one state more and less
@pytest.mark.parametrize("states", [2, 7, 8, 9, 64, 65, 513])
def test_adjoint_chunks(states):
    """Reverse-mode gradient of the log-likelihood against central differences of
    the oracle (step 1e-5: an error of about 1e-10 / 1e-5 x |ell| / |g|, 1e-6)."""
    from parsmooth.gradient import IteratedLoglikelihood
    nx, T = 2, states - 1
    theta = np.array([np.log(0.05), np.log(0.3), 0.1])

    def model(th):
        v = {k: x.numpy() for k, x in _build(torch.as_tensor(th)).items()}
        tm = O.FunctionalModel(O.Linear(v["trans_params"].reshape(nx, nx)), O.MVNSqrt(v["trans_q_mean"], v["trans_q_chol"]))
        om = O.FunctionalModel(O.Linear(v["obs_params"].reshape(1, nx)), O.MVNSqrt(v["obs_q_mean"], v["obs_q_chol"]))
        return v, tm, om

    v, tm, om = model(theta)
    ys = np.asarray(O.lgssm_data(np.zeros(nx), v["trans_params"].reshape(nx, nx), v["obs_params"].reshape(1, nx),
                                 gram(v["obs_q_chol"]), gram(v["trans_q_chol"]), np.zeros(nx), np.zeros(1), T,
                                 random_state=np.random.RandomState(0))[1], np.float64)

    def ell(th):
        _, tm, om = model(th)
        return O.filtering(ys, O.MVNSqrt(np.zeros(nx), np.eye(nx)), tm, om, O.extended, None, True,
                           return_loglikelihood=True)[1]

    obj = IteratedLoglikelihood(_build, N.MODEL_LINEAR, N.MODEL_LINEAR, nx, 1, [T], ys, extended, 2,
                                (np.zeros((T + 1, nx)), np.tile(np.eye(nx), (T + 1, 1, 1))))
    got, grad = obj.value_and_grad(torch.as_tensor(theta))
    assert float(got[0]) == pytest.approx(ell(theta), rel=1e-10)
    h = 1e-5
    fd = np.array([(ell(theta + h * e) - ell(theta - h * e)) / (2 * h) for e in np.eye(3)])
    np.testing.assert_allclose(grad[0].cpu().numpy(), fd, rtol=1e-6, atol=1e-6)
