"""Whole-pass driver over a ragged batch of sequences: shapes and dtypes are
checked here, buffers are torch tensors on the HIP device, and every pass is
one call into libparsmooth_hip.so."""
from __future__ import annotations

import ctypes
import os
from typing import Optional, Sequence

import numpy as np
import torch

from . import _native as N
from .models import TorchFunction
from ._base import MVNSqrt, MVNStandard
from .linearization._methods import Method, model_struct


# Default threshold of min|diag| / max|diag| below which an FP32 square-root
# step is recomputed in FP64 (see include/psm.h, psm_problem.fallback_ratio).
FP32_FALLBACK_RATIO = 1e-4


def set_fp32_fallback(ratio: float):
    """Set the FP64 re-triangularisation threshold for FP32 square-root runs
    created afterwards (0 disables the fallback)."""
    global FP32_FALLBACK_RATIO
    FP32_FALLBACK_RATIO = float(ratio)


def to_dev(x, dtype, dev):
    if isinstance(x, torch.Tensor):
        return x.to(device=dev, dtype=dtype).contiguous()
    return torch.as_tensor(np.asarray(x, dtype=np.float64)).to(device=dev, dtype=dtype).contiguous()


def compute_dtype(x0) -> torch.dtype:
    m = x0[0]
    if isinstance(m, torch.Tensor) and m.dtype in (torch.float32, torch.float64):
        return m.dtype
    if isinstance(m, np.ndarray) and m.dtype == np.float32:
        return torch.float32
    return torch.float64


def states_per_chunk(n_states: int, nx: int = 5, dtype: torch.dtype = torch.float64) -> int:
    """States per chunk, 0 for the library's choice (4 to 16: 32,768 chunks).

    A lane's chain through a state of its chunk is longer than one through a level
    of the scan, and up to 4096 chunks the 16-lane scan has three levels of 16 groups,
    however many chunks there are: up to 3 * 4096 states the chunk is as short as
    that allows (six iterations, FP64, nx = 5, against 4: T = 200 568 us at 1, 758;
    3,000 757 at 1, 927; 4,500 813 at 2, 951; 11,000 953 at 3, 1025).  With more
    chunks the fan-in of 2 keeps three levels up to 32,768 of them, and what a chunk
    costs and saves crosses slowly: the lines at 8192 chunks and 24,576 states are
    measured (15,000 1022 at 2, 1074 at 3; 24,000 1119 at 3, 1202 at 4; 26,000 1199
    at 3, 1202 at 4, 1147 at 2; 60,000 1360 at 4, 1470 at 2).  FP32, the covariance
    form and nx = 2 and 6 cross at the same sizes: from 200 to 24,000 states the rule is
    1 to 33 % faster than a chunk of 4 in all of them.

    Where the chip is full many times over, the scan's share is what counts, and
    shrinks with the chunk (one iteration, against 16: FP64, nx = 5, 2.2 million states
    2.47 ms at 24, 2.61; 4.2 million 4.32 at 40, 4.72; 8.5 million 8.62 at 40, 9.00; FP32
    1.46, 1.58; 2.59, 2.80; 5.03, 5.21; the covariance form, nx 4 to 8, and nx 2 in FP64
    gain up to 11 % and lose at most 3).  FP32 items of one or two dimensions are too small for
    it (nx = 2, 4.2 million states: 784 us at 16, 889 at 40)."""
    if n_states <= 3 * 4096:
        return -(-n_states // 4096)
    if n_states <= 3 * 8192:
        return -(-n_states // 8192)
    if n_states >= 1 << 21 and nx * dtype.itemsize >= 16:
        return 40 if n_states >= 1 << 22 else 24
    return 0


class Problem:
    """Dims, dtype, form and the sequence layout of one batch.

    ``lengths[s]`` is the number of observations of sequence s; it owns
    ``lengths[s] + 1`` states (its prior state first).

    A kept problem may be used on any stream: its offsets are in place when the
    constructor returns.  ``one_call``: the problem serves only calls on the current
    stream, and its offsets may be filled in on it (a copy from host memory would
    wait for what the stream still has to do)."""

    def __init__(self, nx: int, ny: int, lengths: Sequence[int], dtype: torch.dtype, sqrt: bool,
                 dev, chunk: int = 0, tangent_code: Optional[int] = None, one_call: bool = False):
        lengths = np.asarray(lengths, dtype=np.int64).reshape(-1)
        if lengths.size == 0 or np.any(lengths < 1):
            raise ValueError("every sequence needs at least one observation")
        self.nx, self.ny = int(nx), int(ny)
        self.lengths = lengths
        self.n_seq = int(lengths.size)
        offs = np.zeros(self.n_seq + 1, dtype=np.int64)
        offs[1:] = np.cumsum(lengths + 1)
        self.state_offsets_host = offs
        self.n_states = int(offs[-1])
        self.n_obs = int(lengths.sum())
        self.dtype = dtype
        self.sqrt = sqrt
        self.dev = dev
        # FP64 re-triangularisation fallback of the FP32 square-root path
        self.fallback_counter = torch.zeros(1, dtype=torch.int64, device=dev)
        self.state_offsets = torch.arange(0, 2 * self.n_states, self.n_states, device=dev) \
            if one_call and self.n_seq == 1 else torch.as_tensor(offs).to(dev)
        code = N.dtype_code(dtype) if tangent_code is None else int(tangent_code)
        if not N.lib().psm_supported(code, N.FORM_SQRT if sqrt else N.FORM_STD, self.nx, self.ny):
            raise NotImplementedError(f"no compiled kernels for nx={nx}, ny={ny}, dtype code {code}")
        ratio = FP32_FALLBACK_RATIO if (code in (N.PSM_F32, N.PSM_F32_TANGENT) and sqrt) else 0.0
        self.tangent = tangent_code is not None
        self.struct = N.PsmProblem(code, N.FORM_SQRT if sqrt else N.FORM_STD,
                                   self.nx, self.ny, self.n_seq, int(chunk) or self.default_chunk(), self.n_states,
                                   self.state_offsets.data_ptr(), float(ratio), 0,
                                   self.fallback_counter.data_ptr())
        self.ws_bytes = int(N.lib().psm_workspace_bytes(ctypes.byref(self.struct)))
        if self.ws_bytes == 0:
            N.check(-1, "psm_workspace_bytes")
        self._ws = None

    # candidate schedules of the library's autotuner: chunk, and scan fan-in
    # with or without the 16-lane upper scan levels (N.SCAN_TEAM), the half-wave
    # level 0 (N.SCAN_HALF) and the four-lane level 0 (N.SCAN_QUAD), and the
    # 16-lane level 0 (N.SCAN_ROW), both with 16-lane upper levels
    TUNE_CHUNKS = (2, 4, 8, 16, 32)   # and 1 up to 8192 states
    TUNE_SCAN_K = tuple(k | f for f in (0, N.SCAN_TEAM, N.SCAN_HALF, N.SCAN_TEAM | N.SCAN_HALF,
                                        N.SCAN_TEAM | N.SCAN_QUAD,
                                        N.SCAN_TEAM | N.SCAN_QUAD | N.SCAN_HALF)
                        for k in (2, 4, 8)) + tuple(k | N.SCAN_TEAM | N.SCAN_ROW for k in (1, 2))

    def default_chunk(self) -> int:
        """The chunk of a problem for which none is asked (0: the library's choice)."""
        if "PSM_CHUNK" in os.environ:
            return 0
        if self.tangent:
            # tangent types scan with one lane per combination: the library's choice,
            # longer where the chip is full (FP64, a million states: 349 ms at 40, 392)
            return 40 if self.n_states >= 1 << 20 else 0
        return states_per_chunk(self.n_states, self.nx, self.dtype)

    def set_schedule(self, chunk: int, scan_k: int):
        """Fix the launch schedule and resize the workspace.  (0, 0) is a new problem's
        schedule; with a scan_k of its own, chunk 0 is the library's choice."""
        self.struct.chunk = int(chunk) if chunk or scan_k else self.default_chunk()
        self.struct.scan_k = int(scan_k)
        nbytes = int(N.lib().psm_workspace_bytes(ctypes.byref(self.struct)))
        if nbytes == 0:
            N.check(-1, "psm_workspace_bytes")
        if self._ws is not None and self._ws.numel() < nbytes:
            self._ws = None
        self.ws_bytes = nbytes

    def autotune(self, mods, ys, m0, L0, nom_m, nom_L, filt, out):
        """Time every candidate schedule of one filter-smoother pass at the given
        nominal and keep the fastest; returns (chunk, scan_k, ms per pass)."""
        saved = (self.struct.chunk, self.struct.scan_k)
        need = 0
        for c in range(1, 65):  # the refinement stage may pick any chunk up to 64
            for k in self.TUNE_SCAN_K:
                self.struct.chunk, self.struct.scan_k = c, k
                need = max(need, int(N.lib().psm_workspace_bytes(ctypes.byref(self.struct))))
        self.struct.chunk, self.struct.scan_k = saved
        ws = torch.empty(need, dtype=torch.uint8, device=self.dev)
        bc, bk, ms = ctypes.c_int32(0), ctypes.c_int32(0), ctypes.c_float(0.0)
        rc = N.lib().psm_autotune(ctypes.byref(self.struct), ctypes.byref(mods.trans), ctypes.byref(mods.obs),
                                  mods.sigma_ref(), N.ptr(ys), N.ptr(m0), N.ptr(L0), N.ptr(nom_m), N.ptr(nom_L),
                                  N.ptr(filt[0]), N.ptr(filt[1]), N.ptr(out[0]), N.ptr(out[1]), N.ptr(ws),
                                  need, N.stream_ptr(), ctypes.byref(bc), ctypes.byref(bk), ctypes.byref(ms))
        N.check(rc, "psm_autotune")
        del ws
        self.set_schedule(bc.value, bk.value)
        return bc.value, bk.value, ms.value

    @property
    def workspace(self) -> torch.Tensor:
        if self._ws is None:
            self._ws = torch.empty(self.ws_bytes, dtype=torch.uint8, device=self.dev)
        return self._ws

    def new_traj(self):
        m = torch.empty((self.n_states, self.nx), dtype=self.dtype, device=self.dev)
        L = torch.empty((self.n_states, self.nx, self.nx), dtype=self.dtype, device=self.dev)
        return m, L

    def default_nominal(self):
        """Zero mean and identity chol/cov at every state
        (parsmooth/parallel/_filtering.py:25-28, _smoothing.py:21-28)."""
        m = torch.zeros((self.n_states, self.nx), dtype=self.dtype, device=self.dev)
        L = torch.eye(self.nx, dtype=self.dtype, device=self.dev).expand(self.n_states, self.nx, self.nx).contiguous()
        return m, L


class Models:
    """ctypes views of the transition / observation models and the sigma table."""

    def __init__(self, prob: Problem, trans, obs, method: Method):
        self.prob = prob
        self.trans, keep_t = model_struct(trans, prob.dtype, prob.dev, prob.sqrt, nin=prob.nx)
        self.trans_fn = keep_t[3]
        self.obs, self.obs_fn = None, None
        keep_o = ()
        if obs is not None:
            self.obs, keep_o = model_struct(obs, prob.dtype, prob.dev, prob.sqrt, nin=prob.nx)
            self.obs_fn = keep_o[3]
            if self.obs_fn.nin != prob.nx or self.obs_fn.nout != prob.ny:
                raise ValueError("observation function dims do not match the problem")
        if self.trans_fn.nin != prob.nx or self.trans_fn.nout != prob.nx:
            raise ValueError("transition function dims do not match the state dimension")
        self.sigma, keep_s = method.sigma(prob.nx, prob.dtype, prob.dev)
        self._keep = (keep_t, keep_o, keep_s)
        self._tables = {}

    @property
    def tabulated(self) -> bool:
        return isinstance(self.trans_fn, TorchFunction) or isinstance(self.obs_fn, TorchFunction)

    def prepare(self, nom_m, nom_L, obs: bool = True):
        """Evaluate torch-callable models at the linearization points of this
        nominal trajectory (row i = state i) into persistent tables."""
        if not self.tabulated:
            return
        xi = self._keep[2][0] if self.sigma is not None else None
        L = nom_L
        if xi is not None and not self.prob.sqrt:
            L = torch.linalg.cholesky(nom_L)   # the kernels factor the covariance the same way
        for name, fn, struct in (("trans", self.trans_fn, self.trans),
                                 ("obs", self.obs_fn, self.obs if obs else None)):
            if struct is None or not isinstance(fn, TorchFunction):
                continue
            width = fn.row_width(xi.shape[0] if xi is not None else 0)
            buf = self._tables.get(name)
            if buf is None or buf.shape != (self.prob.n_states, width):
                buf = torch.empty((self.prob.n_states, width), dtype=self.prob.dtype, device=self.prob.dev)
                self._tables[name] = buf
            fn.tabulate(nom_m.reshape(-1, fn.nin), L.reshape(-1, fn.nin, fn.nin), xi, out=buf)
            struct.params = buf.data_ptr()

    def sigma_ref(self):
        return ctypes.byref(self.sigma) if self.sigma is not None else None


def filter_pass(prob: Problem, mods: Models, ys, m0, L0, nom_m, nom_L, want_ell: bool,
                out=None):
    out_m, out_L = out if out is not None else prob.new_traj()
    ell = torch.empty(prob.n_seq, dtype=torch.float64, device=prob.dev) if want_ell else None
    mods.prepare(nom_m, nom_L)
    rc = N.lib().psm_filter(ctypes.byref(prob.struct), ctypes.byref(mods.trans), ctypes.byref(mods.obs),
                            mods.sigma_ref(), N.ptr(ys), N.ptr(m0), N.ptr(L0), N.ptr(nom_m),
                            N.ptr(nom_L), N.ptr(out_m), N.ptr(out_L), N.ptr(ell),
                            N.ptr(prob.workspace), prob.ws_bytes, N.stream_ptr())
    N.check(rc, "psm_filter")
    return out_m, out_L, ell


def smoother_pass(prob: Problem, mods: Models, fm, fL, nom_m, nom_L, out=None):
    out_m, out_L = out if out is not None else prob.new_traj()
    mods.prepare(nom_m, nom_L, obs=False)
    rc = N.lib().psm_smoother(ctypes.byref(prob.struct), ctypes.byref(mods.trans), mods.sigma_ref(),
                              N.ptr(fm), N.ptr(fL), N.ptr(nom_m), N.ptr(nom_L), N.ptr(out_m),
                              N.ptr(out_L), N.ptr(prob.workspace), prob.ws_bytes, N.stream_ptr())
    N.check(rc, "psm_smoother")
    return out_m, out_L


def filter_smoother_pass(prob: Problem, mods: Models, ys, m0, L0, nom_m, nom_L, filt, out,
                         use_graph: bool = False):
    fm, fL = filt
    om, oL = out
    mods.prepare(nom_m, nom_L)
    rc = N.lib().psm_filter_smoother(ctypes.byref(prob.struct), ctypes.byref(mods.trans),
                                     ctypes.byref(mods.obs), mods.sigma_ref(), N.ptr(ys), N.ptr(m0),
                                     N.ptr(L0), N.ptr(nom_m), N.ptr(nom_L), N.ptr(fm), N.ptr(fL),
                                     N.ptr(om), N.ptr(oL), N.ptr(prob.workspace), prob.ws_bytes,
                                     int(bool(use_graph)), N.stream_ptr())
    N.check(rc, "psm_filter_smoother")
    return om, oL


def _seq_models_ready(mods: Models, nom_m, nom_L, obs: bool = True):
    if nom_m is None:
        if mods.tabulated:
            raise NotImplementedError(
                "parallel=False without a nominal trajectory linearizes at the running estimate, "
                "which a torch-callable or conditional-moments model cannot be evaluated at ahead "
                "of the recursion; pass a nominal trajectory or use a parsmooth.models function")
    else:
        mods.prepare(nom_m, nom_L, obs=obs)


def seq_filter_pass(prob: Problem, mods: Models, ys, m0, L0, nom_m, nom_L, want_ell: bool,
                    out=None):
    """Sequential filter, one lane per sequence (parallel=False).  nom_m None:
    the transition is linearized at the filtered and the observation at the
    predicted state."""
    out_m, out_L = out if out is not None else prob.new_traj()
    ell = torch.empty(prob.n_seq, dtype=torch.float64, device=prob.dev) if want_ell else None
    _seq_models_ready(mods, nom_m, nom_L)
    rc = N.lib().psm_seq_filter(ctypes.byref(prob.struct), ctypes.byref(mods.trans),
                                ctypes.byref(mods.obs), mods.sigma_ref(), N.ptr(ys), N.ptr(m0),
                                N.ptr(L0), N.ptr(nom_m), N.ptr(nom_L), N.ptr(out_m), N.ptr(out_L),
                                N.ptr(ell), N.stream_ptr())
    N.check(rc, "psm_seq_filter")
    return out_m, out_L, ell


def seq_smoother_pass(prob: Problem, mods: Models, fm, fL, nom_m, nom_L, out=None):
    """Sequential (Rauch-Tung-Striebel) smoother, one lane per sequence.
    nom_m None: the transition out of state k is linearized at the smoothed
    state k+1."""
    out_m, out_L = out if out is not None else prob.new_traj()
    _seq_models_ready(mods, nom_m, nom_L, obs=False)
    rc = N.lib().psm_seq_smoother(ctypes.byref(prob.struct), ctypes.byref(mods.trans), mods.sigma_ref(),
                                  N.ptr(fm), N.ptr(fL), N.ptr(nom_m), N.ptr(nom_L), N.ptr(out_m),
                                  N.ptr(out_L), N.stream_ptr())
    N.check(rc, "psm_seq_smoother")
    return out_m, out_L


def mean_sq_diff(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """mean((a - b)^2) on the device, accumulated in FP64 (one-element tensor)."""
    out = torch.empty(1, dtype=torch.float64, device=a.device)
    a = a.contiguous()
    b = b.to(a.dtype).contiguous()
    if a.shape != b.shape:
        raise ValueError("mean_sq_diff needs equal shapes")
    rc = N.lib().psm_mean_sq_diff(N.dtype_code(a.dtype), a.numel(), N.ptr(a), N.ptr(b), N.ptr(out),
                                  N.stream_ptr())
    N.check(rc, "psm_mean_sq_diff")
    return out
