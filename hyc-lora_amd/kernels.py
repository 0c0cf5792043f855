"""Host-side launchers: torch tensors in, torch tensors out, every computation done by the HIP library.

torch is used for device memory and the current stream only.  Nothing here computes on the CPU and
nothing falls back to torch ops for the hot path: inputs that are not CUDA tensors raise.
"""
import ctypes
import functools
from dataclasses import dataclass
from typing import Optional

import torch

from . import _abi, _host
from ._abi import HycDesc, check

BF16 = torch.bfloat16


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream():
    """handle of torch's current stream on the current device (the kernels are launched on it)"""
    if _raw_stream is not None:                    # no Stream object is built: 0.5 us instead of 5 per launch
        return _raw_stream(torch.cuda.current_device())
    return torch.cuda.current_stream().cuda_stream


def _p(t):
    """device address for a pointer argument of the library (the prototypes turn the number into a pointer)"""
    return None if t is None else t.data_ptr()


def _need(t, dtype, name):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError("%s must be a CUDA (ROCm) tensor: the hot path runs on the GPU only" % name)
    if t.dtype != dtype:
        raise ValueError("%s must be %s, got %s" % (name, dtype, t.dtype))
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % name)
    return t


def _need_vec(t, dtype, n, name):
    """a contiguous device vector of exactly n elements (the kernels index it without further checks)"""
    _need(t, dtype, name)
    if t.numel() != n:
        raise ValueError("%s must hold %d elements, got %d" % (name, n, t.numel()))
    return t


def _need_weight(w, H):
    if not isinstance(w, torch.Tensor) or not w.is_cuda or not w.is_contiguous() or w.numel() != H:
        raise ValueError("weight must be a contiguous CUDA tensor of %d elements" % H)
    return w


def threshold_value(t):
    """Python float of a threshold.  A device tensor costs one host round trip the first time; the float is then kept
    on the tensor object together with the tensor's version counter, so the frozen threshold of a calibrated module
    (the same 0-d tensor call after call) is read back once, not at every step, and an in-place update of the tensor
    (`copy_`, `mul_`, a restored state) is seen.  The read-back is a synchronisation: the calibration calls of a module
    must run outside a stream capture."""
    if not isinstance(t, torch.Tensor):
        return float(t)
    cached = getattr(t, "_hyc_float", None)
    version = t._version
    if cached is None or cached[0] != version:
        cached = (version, float(t))
        try:
            t._hyc_float = cached
        except AttributeError:
            pass
    return cached[1]


class KeptBudget:
    """Room for the sparse side data (kept softmax probabilities, element outliers) of one calibrated site, so that its
    steady-state calls never wait for the GPU.

    The reference reads the number of kept entries back on every call (`to_sparse()`, compress_function.py:153, :269)
    before it can allocate them.  Here a call that has a budget allocates `capacity(rows)` entries - 1.25 x the largest
    kept fraction seen so far, plus a little - cuts the row offsets off at that capacity on the device (hyc_csr_offsets)
    and leaves the true total in a device word.  Entries past the capacity are dropped, which must not go unnoticed: the
    total travels to pinned host memory behind the kernels, and the next call of the site that finds it arrived checks
    it (`poll`), raises if entries were dropped and grows the budget.  `sync_check()` does the same at once.
    """
    MARGIN = 1.25

    def __init__(self):
        self.per_row = -1.0        # largest kept entries per row seen (negative: nothing seen yet)
        self._pending = []         # (event, pinned int64 scalar, capacity, rows) of calls not checked yet
        self._spare = []           # pinned scalars to use again

    @property
    def ready(self):
        return self.per_row >= 0.0

    def observe(self, nnz, rows):
        self.per_row = max(self.per_row, nnz / max(rows, 1))

    def capacity(self, rows):
        return int(self.per_row * self.MARGIN * rows) + rows // 8 + 1024

    def watch(self, total, capacity, rows):
        """keep an eye on `total` (int64 device scalar of a call that was given `capacity`)"""
        if torch.cuda.is_current_stream_capturing():
            return                                  # a captured call is checked by whoever replays it (SparseRows.total)
        host = self._spare.pop() if self._spare else torch.empty((), dtype=torch.int64, pin_memory=True)
        host.copy_(total, non_blocking=True)
        done = torch.cuda.Event()
        done.record()
        self._pending.append((done, host, capacity, rows))

    def _check(self, host, capacity, rows):
        n = int(host)
        self._spare.append(host)
        self.observe(n, rows)
        if n > capacity:
            raise RuntimeError("a compressed activation kept %d sparse entries but its buffers were sized for %d "
                               "(1.25 x the largest share seen before): the entries beyond were dropped and the "
                               "gradients computed from that call are not exact.  The budget has been raised; "
                               "repeat the step." % (n, capacity))

    def poll(self):
        """check the calls whose totals have arrived; never waits (and asks nothing of the runtime during a capture)"""
        if torch.cuda.is_current_stream_capturing():
            return
        while self._pending and self._pending[0][0].query():
            _, host, capacity, rows = self._pending.pop(0)
            self._check(host, capacity, rows)

    def sync_check(self):
        """wait for every watched call and check it"""
        while self._pending:
            done, host, capacity, rows = self._pending.pop(0)
            done.synchronize()
            self._check(host, capacity, rows)


def kept_budget(threshold):
    """The KeptBudget that travels with a threshold tensor (created on first use; None for a plain number).  A site that
    is still calibrating measures a fresh threshold tensor on every call, so each of its calls finds a new budget and
    sizes its buffers exactly; the frozen threshold of a calibrated site is the same tensor call after call, so its
    first steady-state call reads the total back once and the later ones do not."""
    if not isinstance(threshold, torch.Tensor):
        return None
    budget = getattr(threshold, "_hyc_budget", None)
    if budget is None:
        budget = KeptBudget()
        try:
            threshold._hyc_budget = budget
        except AttributeError:
            return None
    return budget


def _csr_offsets(lib, counts, rows, budget):
    """(row_ptr, nnz to allocate, total) from per-row counts.  Without a budget, or with one that has seen nothing yet,
    the total is read back (one host round trip) and the buffers are exact; otherwise nothing waits."""
    dev = counts.device
    row_ptr = torch.empty(rows + 1, dtype=torch.int32, device=dev)
    total = torch.empty((), dtype=torch.int64, device=dev)
    if budget is not None and budget.ready:
        budget.poll()
        cap = budget.capacity(rows)
        check(lib.hyc_csr_offsets(_p(counts), rows, cap, _p(row_ptr), _p(total), _stream()))
        budget.watch(total, cap, rows)
        return row_ptr, cap, total
    check(lib.hyc_csr_offsets(_p(counts), rows, -1, _p(row_ptr), _p(total), _stream()))
    nnz = int(total.item())
    if budget is not None:
        budget.observe(nnz, rows)
    return row_ptr, nnz, total


def num_outlier_channels(H, ratio):
    """k = floor(ratio*H + 1/2)"""
    import math
    return int(math.floor(ratio * H + 0.5))


# ----------------------------------------------------------------------------------------------------
# channel mode
# ----------------------------------------------------------------------------------------------------
SCALE_RULES = {"range": _abi.SCALE_RANGE, "absmax": _abi.SCALE_ABSMAX}
DEFAULT_SCALE_RULE = "absmax"


@dataclass
class ChannelPlan:
    """the static part of one activation site: its outlier-channel set and the rule its group scales follow
    ("absmax": 2 max|x| / (2^bits - 1), the reference's formula over the interval made symmetric about zero, so that no
    element ends up more than half a step away; "range": the reference's (max - min) / (2^bits - 1) as it stands,
    which has no zero point and clips groups that are not centred on 0)"""
    H: int
    k: int
    idx: torch.Tensor    # int32 [k], ascending
    plan: torch.Tensor   # int32 [H/8] (bit pattern of the uint32 lookup words)
    scale_rule: str = DEFAULT_SCALE_RULE


def kth_value(x, k):
    """the k-th smallest (1-based) of all elements of x (bf16 or fp32) as a 0-d fp32 tensor; the value
    `torch.kthvalue(x.flatten().float(), k).values` gives, without a sort and without a host round trip"""
    if x.dtype not in (BF16, torch.float32):
        raise ValueError("x must be bfloat16 or float32, got %s" % x.dtype)
    if not x.is_cuda:
        raise ValueError("x must live on the GPU")
    x = x.contiguous()
    lib = _abi.load()
    out = torch.empty((), dtype=torch.float32, device=x.device)
    ws = torch.empty(lib.hyc_kth_value_workspace_bytes() // 4, dtype=torch.int32, device=x.device)
    code = _abi.DTYPE_BF16 if x.dtype == BF16 else _abi.DTYPE_F32
    check(lib.hyc_kth_value(_p(x), code, x.numel(), int(k), _p(out), _p(ws), _stream()))
    return out


def channel_absmax(x2d, amax=None):
    """running per-channel max |x| (fp32 [H]); pass the previous result to accumulate"""
    if isinstance(x2d, torch.Tensor) and x2d.is_cuda and not x2d.is_contiguous():
        x2d = x2d.contiguous()                     # calibration only (twice per site): a copy is acceptable
    _need(x2d, BF16, "x")
    M, H = x2d.shape
    if amax is None:
        amax = torch.zeros(H, dtype=torch.float32, device=x2d.device)
    _need_vec(amax, torch.float32, H, "amax")
    check(_abi.load().hyc_channel_absmax(_p(x2d), M, H, _p(amax), _stream()))
    return amax


def select_channels(amax, k, scale_rule=DEFAULT_SCALE_RULE):
    if scale_rule not in SCALE_RULES:
        raise ValueError("scale_rule must be 'absmax' or 'range', got %r" % (scale_rule,))
    _need(amax, torch.float32, "amax")
    H = amax.numel()
    if H % 8 or not 0 <= k <= H:
        raise ValueError("select_channels: H=%d must be a multiple of 8 and 0 <= k=%d <= H" % (H, k))
    idx = torch.empty(max(k, 1), dtype=torch.int32, device=amax.device)[:k]
    plan = torch.empty(H // 8, dtype=torch.int32, device=amax.device)
    check(_abi.load().hyc_select_channels(_p(amax), H, k, _p(idx), _p(plan), _stream()))
    return ChannelPlan(H, k, idx, plan, scale_rule)


def _check_plan(plan, device=None):
    """the kernels index plan.plan [H/8] and plan.idx [k] without further checks, so they must be int32 device
    tensors of exactly those sizes, on the device of the activation they are used with"""
    for name, t, n in (("plan.plan", plan.plan, plan.H // 8), ("plan.idx", plan.idx, plan.k)):
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise ValueError("%s must be a CUDA (ROCm) tensor; after loading a checkpoint on the host, move the "
                             "calibration state to the GPU (load_calibration_state does)" % name)
        if t.dtype != torch.int32 or not t.is_contiguous() or t.numel() != n:
            raise ValueError("%s must be a contiguous int32 tensor of %d elements" % (name, n))
        if device is not None and t.device != device:      # (a device without an index means the current one)
            want = torch.device(device)
            index = want.index if want.index is not None else torch.cuda.current_device()
            if t.device.type != want.type or t.device.index != index:
                raise ValueError("%s lives on %s, the activation on %s" % (name, t.device, device))
    if plan.scale_rule not in SCALE_RULES:
        raise ValueError("scale_rule must be 'absmax' or 'range', got %r" % (plan.scale_rule,))


def channel_desc(plan: ChannelPlan, bits, group, device=None):
    _check_plan(plan, device)
    return _checked_desc(plan, bits, group)


def _checked_desc(plan, bits, group):
    """channel_desc of a plan that _check_plan has just passed"""
    d = HycDesc()
    d.mode, d.bits, d.group, d.k = _abi.MODE_CHANNEL, bits, group, plan.k
    d.chan_plan = plan.plan.data_ptr()
    d.chan_idx = plan.idx.data_ptr() if plan.k else None
    d.scale_rule = SCALE_RULES[plan.scale_rule]
    return d


def dense_desc(bits=4):
    d = HycDesc()
    d.mode, d.bits = _abi.MODE_DENSE, bits
    return d


@dataclass
class ChannelCompressed:
    """a [M,H] bf16 activation held as codes + outlier channels + group scales"""
    stored: torch.Tensor   # uint8 [M, H*bits/8] (int8 [M,H] for 8 bits)
    vals: torch.Tensor     # bf16 [M, k]
    scales: torch.Tensor   # bf16 [M, H/group]
    plan: ChannelPlan
    bits: int
    group: int
    M: int
    H: int

    def desc(self):
        return channel_desc(self.plan, self.bits, self.group, self.stored.device)

    def nbytes(self):
        return self.stored.numel() * self.stored.element_size() + 2 * self.vals.numel() + 2 * self.scales.numel()


class _Native:
    """the functions of csrc/host/host.cpp, loaded with the first one asked for (a package whose libraries are not built can be
    imported).  Each returns None for what it does not cover, and the caller goes on with the form written out here."""

    def __getattr__(self, name):
        if name.startswith("_"):
            raise AttributeError(name)
        module = _host.load(torch.nn.Parameter, ChannelCompressed, ChannelPlan, ThresholdCompressed, SparseRows)
        if module is None:
            self.__dict__[name] = lambda *args: None
        else:
            self.__dict__.update((n, f) for n, f in vars(module).items() if not n.startswith("_"))
        return self.__dict__[name]


native = _Native()


def node(name):
    """the function `name` of csrc/host/host.cpp that also records the operator's backward natively, without a torch.autograd.Function
    around it (None, or a None from it: the Function serves).  Whoever puts something else in the place of `native`, to count the calls
    or to have the interpreted forms alone, sees every one of them: nothing is recorded past it."""
    return getattr(native, name) if type(native) is _Native else None


def alloc_channel(M, H, plan, bits, group, device):
    if plan.H != H:
        raise ValueError("the outlier-channel plan was made for %d channels, the activation has %d" % (plan.H, H))
    _check_plan(plan, torch.device(device) if not isinstance(device, torch.device) else device)
    stored = torch.empty((M, H * bits // 8), dtype=torch.int8 if bits == 8 else torch.uint8, device=device)
    vals = torch.empty((M, plan.k), dtype=BF16, device=device)
    scales = torch.empty((M, H // group), dtype=BF16, device=device)
    return ChannelCompressed(stored, vals, scales, plan, bits, group, M, H)


def _need_rows(t, name):
    """a bf16 [M, H] matrix whose rows are contiguous; the rows themselves may be further apart (a column slice)"""
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError("%s must be a CUDA (ROCm) tensor: the hot path runs on the GPU only" % name)
    if t.dtype != BF16 or t.dim() != 2 or (t.shape[1] > 1 and t.stride(1) != 1):
        raise ValueError("%s must be a bfloat16 matrix with contiguous rows" % name)
    return t


def compress_channel(x2d, plan, bits, group):
    out = native.compress(x2d, plan, bits, group)
    if out is not None:
        return out
    _need_rows(x2d, "x")
    M, H = x2d.shape
    lib = _abi.load()
    check(lib.hyc_check_shape(H, bits, group, _abi.MODE_CHANNEL))
    out = alloc_channel(M, H, plan, bits, group, x2d.device)
    d = _checked_desc(plan, bits, group)
    pitch = x2d.stride(0) if M > 1 else H
    check(lib.hyc_compress_rows(_p(x2d), pitch, M, H, ctypes.byref(d), _p(out.stored), _p(out.vals), _p(out.scales), None,
                                _stream()))
    return out


def decompress_channel(c: ChannelCompressed):
    xhat = native.decompress(c)
    if xhat is not None:
        return xhat
    xhat = torch.empty((c.M, c.H), dtype=BF16, device=c.stored.device)
    d = c.desc()
    check(_abi.load().hyc_decompress(_p(c.stored), _p(c.vals), _p(c.scales), c.M, c.H, ctypes.byref(d), _p(xhat), _stream()))
    return xhat


# ----------------------------------------------------------------------------------------------------
# threshold mode (the scheme of the reference snapshot)
# ----------------------------------------------------------------------------------------------------
def scale_strides(scale, S, H):
    """(stride_token, stride_channel) of a per-tensor [] / per-channel [1,H] / per-token [S,1] scale"""
    n = scale.numel()
    if n == 1:
        return 0, 0
    if scale.dim() >= 2 and scale.shape[-1] == H and n == H:
        return 0, 1
    if scale.dim() >= 2 and scale.shape[-1] == 1 and n == S:
        return 1, 0
    raise ValueError("scale of shape %s is neither per-tensor, per-channel [1,%d] nor per-token [%d,1]"
                     % (tuple(scale.shape), H, S))


@dataclass
class ThresholdCompressed:
    stored: torch.Tensor               # uint8 [M, H*bits/8] / int8 [M,H]
    row_ptr: torch.Tensor              # int32 [M+1]
    cols: torch.Tensor                 # int32 [nnz]
    vals: torch.Tensor                 # bf16 [nnz]
    threshold: float
    scale: torch.Tensor
    L: Optional[torch.Tensor]
    R: Optional[torch.Tensor]
    bits: int
    M: int
    H: int
    S: int

    def desc(self):
        return threshold_desc(self.threshold, self.scale, self.bits, self.S, self.H, self.L, self.R,
                              self.row_ptr, self.cols, self.vals)


def threshold_desc(threshold, scale, bits, S, H, L=None, R=None, row_ptr=None, cols=None, vals=None):
    d = HycDesc()
    d.mode, d.bits = _abi.MODE_THRESHOLD, bits
    d.threshold = float(threshold)
    d.scale = scale.data_ptr()
    d.scale_stride_token, d.scale_stride_channel = scale_strides(scale, S, H)
    d.S = S
    rank = 0 if L is None else L.shape[-1]
    d.rank = rank
    if rank:
        d.L, d.R = L.data_ptr(), R.data_ptr()
    if row_ptr is not None:
        d.csr_row_ptr = row_ptr.data_ptr()
        d.csr_cols = cols.data_ptr() if cols.numel() else None
        d.csr_vals = vals.data_ptr() if vals.numel() else None
    return d


def fit_rows(L, S):
    """pad with zero rows / cut L [S', r] to S rows (the reference's pad_cut_L); L is tiny"""
    have = L.shape[0]
    if have == S:
        return L.contiguous()
    if have > S:
        return L[:S].contiguous()
    out = torch.zeros((S, L.shape[1]), dtype=L.dtype, device=L.device)
    out[:have] = L
    return out


def threshold_native(x, norm, w, bias, eps, S, threshold, scale, bits, L, R, budget):
    """(y, mean, rstd, ThresholdCompressed) of x [..., H] in native code (norm: 0 compress only, 1 rms norm, 2 layer norm), or None:
    a budget that has seen nothing yet, or what the native form does not cover"""
    if budget is None or not budget.ready or not isinstance(x, torch.Tensor) or not x.numel():
        return None
    H = x.shape[-1]
    M = x.numel() // H
    budget.poll()
    cap = budget.capacity(M)
    done = native.threshold_fwd(x, norm, w, bias, eps, S, threshold, scale, bits, L, R, cap, _slab_entries(budget, H, 16384))
    if done is None:
        return None
    y, mean, rstd, stored, row_ptr, cols, vals, total = done
    budget.watch(total, cap, M)
    return y, mean, rstd, ThresholdCompressed(stored, row_ptr, cols, vals, float(threshold), scale, L, R, bits, M, H, S)


def threshold_norm(x, norm, w, bias, eps, static_value, bits, rank, quirk, interpreted, label):
    """y of a calibrated norm of the reference's scheme with its backward recorded natively, or None: the Function serves"""
    outlier, L, scale, R = static_value
    possible = node("recordable")
    if possible is None or not possible(x, w, bias):
        return None
    done = threshold_native(x, norm, w, bias, eps, x.shape[-2] if x.dim() >= 2 else 1, threshold_value(outlier), scale, bits,
                            L if rank > 0 else None, R if rank > 0 else None, kept_budget(outlier))
    if done is None:
        return None
    y, mean, rstd, c = done
    return native.norm_record(y, x, w, bias, c, mean, rstd, quirk, interpreted, label)


def compress_threshold(x2d, S, threshold, scale, bits, L=None, R=None, budget=None):
    """codes + CSR outliers of x [M,H] (row m is sequence position m mod S).  One host read-back
    (the outlier total) sizes the CSR arrays, as `.to_sparse()` does in the reference; with a KeptBudget that has seen
    a call they are sized ahead of time and nothing waits."""
    done = threshold_native(x2d, 0, None, None, 0.0, S, threshold, scale, bits, L, R, budget) if x2d.dim() == 2 else None
    if done is not None:
        return done[3]
    _need(x2d, BF16, "x")
    _need(scale, BF16, "scale")
    M, H = x2d.shape
    lib = _abi.load()
    check(lib.hyc_check_shape(H, bits, 0, _abi.MODE_THRESHOLD))
    dev = x2d.device
    if L is not None:
        L = fit_rows(_need(L, BF16, "L"), S)
        _need(R, BF16, "R")
    stored = torch.empty((M, H * bits // 8), dtype=torch.int8 if bits == 8 else torch.uint8, device=dev)
    counts = torch.empty(M, dtype=torch.int32, device=dev)
    d = threshold_desc(threshold, scale, bits, S, H, L, R)
    check(lib.hyc_compress(_p(x2d), M, H, ctypes.byref(d), _p(stored), None, None, _p(counts), _stream()))
    row_ptr, nnz, _ = _csr_offsets(lib, counts, M, budget)
    cols = torch.empty(nnz, dtype=torch.int32, device=dev)
    vals = torch.empty(nnz, dtype=BF16, device=dev)
    check(lib.hyc_ref_outlier_fill(_p(x2d), M, H, ctypes.byref(d), _p(row_ptr), _p(cols) if nnz else None,
                                   _p(vals) if nnz else None, _stream()))
    return ThresholdCompressed(stored, row_ptr, cols, vals, float(threshold), scale, L, R, bits, M, H, S)


def outlier_counts(x2d, S, threshold, bits=8, L=None, R=None):
    _need(x2d, BF16, "x")
    M, H = x2d.shape
    counts = torch.empty(M, dtype=torch.int32, device=x2d.device)
    one = torch.ones(1, dtype=BF16, device=x2d.device)
    if L is not None:
        L = fit_rows(L, S)
    d = threshold_desc(threshold, one, bits, S, H, L, R)
    check(_abi.load().hyc_ref_outlier_count(_p(x2d), M, H, ctypes.byref(d), _p(counts), _stream()))
    return counts


def decompress_threshold(c: ThresholdCompressed):
    xhat = native.decompress(c)
    if xhat is not None:
        return xhat
    xhat = torch.empty((c.M, c.H), dtype=BF16, device=c.stored.device)
    d = c.desc()
    check(_abi.load().hyc_decompress(_p(c.stored), None, None, c.M, c.H, ctypes.byref(d), _p(xhat), _stream()))
    return xhat


# ----------------------------------------------------------------------------------------------------
# fused operators
# ----------------------------------------------------------------------------------------------------
ACT_CODES = {"silu": _abi.ACT_SILU, "gelu": _abi.ACT_GELU_TANH}


def _wdtype(w):
    if w.dtype == torch.float32:
        return _abi.DTYPE_F32
    if w.dtype == BF16:
        return _abi.DTYPE_BF16
    raise ValueError("RMSNorm weight must be bf16 or fp32, got %s" % w.dtype)


def rmsnorm_fwd_compress_channel(x2d, w, eps, plan, bits, group):
    """-> (y bf16 [M,H], rstd fp32 [M], ChannelCompressed of x)"""
    _need(x2d, BF16, "x")
    M, H = x2d.shape
    _need_weight(w, H)
    lib = _abi.load()
    check(lib.hyc_check_shape(H, bits, group, _abi.MODE_CHANNEL))
    y = torch.empty_like(x2d)
    rstd = torch.empty(M, dtype=torch.float32, device=x2d.device)
    c = alloc_channel(M, H, plan, bits, group, x2d.device)
    d = _checked_desc(plan, bits, group)
    check(lib.hyc_rmsnorm_fwd_compress(_p(x2d), _p(w), _wdtype(w), float(eps), M, H, ctypes.byref(d), _p(y), _p(rstd),
                                       _p(c.stored), _p(c.vals), _p(c.scales), None, _stream()))
    return y, rstd, c


def rmsnorm_fwd_compress_threshold(x2d, w, eps, S, threshold, scale, bits, L=None, R=None, budget=None):
    """-> (y, rstd, ThresholdCompressed of x)"""
    _need(x2d, BF16, "x")
    _need(scale, BF16, "scale")
    M, H = x2d.shape
    _need_weight(w, H)
    lib = _abi.load()
    dev = x2d.device
    if L is not None:
        L = fit_rows(_need(L, BF16, "L"), S)
        _need(R, BF16, "R")
    y = torch.empty_like(x2d)
    rstd = torch.empty(M, dtype=torch.float32, device=dev)
    stored = torch.empty((M, H * bits // 8), dtype=torch.int8 if bits == 8 else torch.uint8, device=dev)
    counts = torch.empty(M, dtype=torch.int32, device=dev)
    d = threshold_desc(threshold, scale, bits, S, H, L, R)
    check(lib.hyc_rmsnorm_fwd_compress(_p(x2d), _p(w), _wdtype(w), float(eps), M, H, ctypes.byref(d), _p(y), _p(rstd),
                                       _p(stored), None, None, _p(counts), _stream()))
    row_ptr, nnz, _ = _csr_offsets(lib, counts, M, budget)
    cols = torch.empty(nnz, dtype=torch.int32, device=dev)
    vals = torch.empty(nnz, dtype=BF16, device=dev)
    check(lib.hyc_ref_outlier_fill(_p(x2d), M, H, ctypes.byref(d), _p(row_ptr), _p(cols) if nnz else None,
                                   _p(vals) if nnz else None, _stream()))
    return y, rstd, ThresholdCompressed(stored, row_ptr, cols, vals, float(threshold), scale, L, R, bits, M, H, S)


def layernorm_fwd_supported(H, bits):
    """rows the one-pass LayerNorm forward covers"""
    return bits in (1, 2, 4, 8) and H % (64 // bits) == 0 and H * bits // 64 <= 1024


def _need_bias(bias, w, H):
    if bias is None:
        return None
    if not bias.is_cuda or not bias.is_contiguous() or bias.numel() != H or bias.dtype != w.dtype:
        raise ValueError("bias must be a contiguous CUDA tensor of %d elements in the weight's dtype" % H)
    return bias


def layernorm_fwd_compress_channel(x2d, w, bias, eps, plan, bits, group):
    """-> (y bf16 [M,H], mean fp32 [M], rstd fp32 [M], ChannelCompressed of x), one pass over x"""
    _need(x2d, BF16, "x")
    M, H = x2d.shape
    _need_weight(w, H)
    _need_bias(bias, w, H)
    lib = _abi.load()
    check(lib.hyc_check_shape(H, bits, group, _abi.MODE_CHANNEL))
    y = torch.empty_like(x2d)
    mean = torch.empty(M, dtype=torch.float32, device=x2d.device)
    rstd = torch.empty(M, dtype=torch.float32, device=x2d.device)
    c = alloc_channel(M, H, plan, bits, group, x2d.device)
    d = _checked_desc(plan, bits, group)
    check(lib.hyc_layernorm_fwd_compress(_p(x2d), _p(w), _p(bias), _wdtype(w), float(eps), M, H, ctypes.byref(d), _p(y),
                                         _p(mean), _p(rstd), _p(c.stored), _p(c.vals), _p(c.scales), None, _stream()))
    return y, mean, rstd, c


def layernorm_fwd_compress_threshold(x2d, w, bias, eps, S, threshold, scale, bits, L=None, R=None, budget=None):
    """-> (y, mean, rstd, ThresholdCompressed of x)"""
    _need(x2d, BF16, "x")
    _need(scale, BF16, "scale")
    M, H = x2d.shape
    _need_weight(w, H)
    _need_bias(bias, w, H)
    lib = _abi.load()
    dev = x2d.device
    if L is not None:
        L = fit_rows(_need(L, BF16, "L"), S)
        _need(R, BF16, "R")
    y = torch.empty_like(x2d)
    mean = torch.empty(M, dtype=torch.float32, device=dev)
    rstd = torch.empty(M, dtype=torch.float32, device=dev)
    stored = torch.empty((M, H * bits // 8), dtype=torch.int8 if bits == 8 else torch.uint8, device=dev)
    counts = torch.empty(M, dtype=torch.int32, device=dev)
    d = threshold_desc(threshold, scale, bits, S, H, L, R)
    check(lib.hyc_layernorm_fwd_compress(_p(x2d), _p(w), _p(bias), _wdtype(w), float(eps), M, H, ctypes.byref(d), _p(y),
                                         _p(mean), _p(rstd), _p(stored), None, None, _p(counts), _stream()))
    row_ptr, nnz, _ = _csr_offsets(lib, counts, M, budget)
    cols = torch.empty(nnz, dtype=torch.int32, device=dev)
    vals = torch.empty(nnz, dtype=BF16, device=dev)
    check(lib.hyc_ref_outlier_fill(_p(x2d), M, H, ctypes.byref(d), _p(row_ptr), _p(cols) if nnz else None,
                                   _p(vals) if nnz else None, _stream()))
    return y, mean, rstd, ThresholdCompressed(stored, row_ptr, cols, vals, float(threshold), scale, L, R, bits, M, H, S)


def _source(c, M, H):
    """(stored, vals, scales, desc) of a ChannelCompressed, or of a dense bf16 x_hat, that holds an [M, H] activation"""
    if isinstance(c, (ChannelCompressed, ThresholdCompressed)) and (c.M, c.H) != (M, H):
        raise ValueError("the saved activation is [%d, %d], the gradient is [%d, %d]" % (c.M, c.H, M, H))
    if isinstance(c, ChannelCompressed):
        return c.stored, c.vals, c.scales, c.desc()
    if isinstance(c, ThresholdCompressed):
        c = decompress_threshold(c)
    _need(c, BF16, "x_hat")
    if c.numel() != M * H or c.shape[-1] != H:
        raise ValueError("the saved activation is %s, the gradient is [%d, %d]" % (tuple(c.shape), M, H))
    return c, None, None, dense_desc()


def rmsnorm_bwd(dy2d, src, w, rstd, c2_quirk=True):
    """-> (dx bf16 [M,H], dw in w's dtype [H]); src is a ChannelCompressed, ThresholdCompressed or dense x_hat"""
    _need(dy2d, BF16, "dy")
    M, H = dy2d.shape
    _need_weight(w, H)
    _need_vec(rstd, torch.float32, M, "rstd")
    lib = _abi.load()
    stored, vals, scales, d = _source(src, M, H)
    P = lib.hyc_rmsnorm_bwd_partials(M, H)
    partials = torch.empty((max(P, 1), H), dtype=torch.float32, device=dy2d.device)
    dx = torch.empty_like(dy2d)
    dw = torch.empty(H, dtype=w.dtype, device=dy2d.device)
    check(lib.hyc_rmsnorm_bwd(_p(dy2d), _p(stored), _p(vals), _p(scales), _p(w), _wdtype(w), _p(rstd), M, H,
                              ctypes.byref(d), 1 if c2_quirk else 0, _p(dx), _p(partials), _p(dw), _stream()))
    return dx, dw


def layernorm_bwd(dy2d, src, w, mean, rstd):
    """-> (dx bf16 [M,H], dw in w's dtype [H]) with xn = (x_hat - mean) * rstd; db = dy.sum(0) is the caller's"""
    _need(dy2d, BF16, "dy")
    M, H = dy2d.shape
    _need_weight(w, H)
    _need_vec(mean, torch.float32, M, "mean")
    _need_vec(rstd, torch.float32, M, "rstd")
    lib = _abi.load()
    stored, vals, scales, d = _source(src, M, H)
    P = lib.hyc_rmsnorm_bwd_partials(M, H)
    partials = torch.empty((max(P, 1), H), dtype=torch.float32, device=dy2d.device)
    dx = torch.empty_like(dy2d)
    dw = torch.empty(H, dtype=w.dtype, device=dy2d.device)
    check(lib.hyc_layernorm_bwd(_p(dy2d), _p(stored), _p(vals), _p(scales), _p(w), _wdtype(w), _p(mean), _p(rstd), M, H,
                                ctypes.byref(d), _p(dx), _p(partials), _p(dw), _stream()))
    return dx, dw


def bias_grad(dy2d, dtype):
    """the sum of dy bf16 [M, H] over its rows, accumulated in fp32, as a vector of `dtype` (bf16 or fp32)"""
    _need(dy2d, BF16, "dy")
    M, H = dy2d.shape
    lib = _abi.load()
    partials = torch.empty((max(lib.hyc_bias_grad_partials(M, H), 1), H), dtype=torch.float32, device=dy2d.device)
    db = torch.empty(H, dtype=dtype, device=dy2d.device)
    check(lib.hyc_bias_grad(_p(dy2d), M, H, _p(partials), _p(db), _wdtype(db), _stream()))
    return db


def rmsnorm_bwd_partial(dy2d, src, w, rstd, c2_quirk=True):
    """-> (dx bf16 [M,H], fp32 partial rows [P,H] whose column sum is dw); the caller does the last reduction"""
    _need(dy2d, BF16, "dy")
    M, H = dy2d.shape
    _need_weight(w, H)
    _need_vec(rstd, torch.float32, M, "rstd")
    lib = _abi.load()
    stored, vals, scales, d = _source(src, M, H)
    P = lib.hyc_rmsnorm_bwd_partials(M, H)
    partials = torch.empty((max(P, 1), H), dtype=torch.float32, device=dy2d.device)
    dx = torch.empty_like(dy2d)
    check(lib.hyc_rmsnorm_bwd(_p(dy2d), _p(stored), _p(vals), _p(scales), _p(w), _wdtype(w), _p(rstd), M, H,
                              ctypes.byref(d), 1 if c2_quirk else 0, _p(dx), _p(partials), None, _stream()))
    return dx, partials[:lib.hyc_rmsnorm_bwd_partial_rows(M, H, ctypes.byref(d))]


def act_bwd(act, g2d, src):
    """act in {'silu', 'gelu'} -> dx bf16 [M,H]"""
    _need(g2d, BF16, "grad_output")
    M, H = g2d.shape
    stored, vals, scales, d = _source(src, M, H)
    dx = torch.empty_like(g2d)
    code = ACT_CODES[act]
    check(_abi.load().hyc_act_bwd(code, _p(g2d), _p(stored), _p(vals), _p(scales), M, H, ctypes.byref(d), _p(dx), _stream()))
    return dx


def hadamard_bwd(g2d, src1, src2):
    """-> (g * x2_hat, x1_hat * g)"""
    _need(g2d, BF16, "grad_output")
    M, H = g2d.shape
    s1, v1, c1, d1 = _source(src1, M, H)
    s2, v2, c2, d2 = _source(src2, M, H)
    dx1, dx2 = torch.empty_like(g2d), torch.empty_like(g2d)
    check(_abi.load().hyc_hadamard_bwd(_p(g2d), _p(s1), _p(v1), _p(c1), ctypes.byref(d1), _p(s2), _p(v2), _p(c2),
                                       ctypes.byref(d2), M, H, _p(dx1), _p(dx2), _stream()))
    return dx1, dx2


def gated_act_bwd(act, g2d, src_act, src_up, src_gate, room=None):
    """backward of act(gate) * up in one pass -> (d_gate, d_up); the three sources are ChannelCompressed.  With `room` (a
    number of columns, 0 included) the two are the halves of one [M, 2 H + room] matrix, returned as a third value."""
    _need(g2d, BF16, "grad_output")
    M, H = g2d.shape
    sa, va, ca, da = _source(src_act, M, H)
    su, vu, cu, du = _source(src_up, M, H)
    sg, vg, cg, dg = _source(src_gate, M, H)
    both = None
    if room is None:
        d_gate, d_up, pitch = torch.empty_like(g2d), torch.empty_like(g2d), H
    else:
        both = torch.empty((M, 2 * H + room), dtype=BF16, device=g2d.device)
        d_gate, d_up, pitch = both[:, :H], both[:, H:2 * H], 2 * H + room
    code = ACT_CODES[act]
    check(_abi.load().hyc_gated_act_bwd_rows(code, _p(g2d), _p(sa), _p(va), _p(ca), ctypes.byref(da), _p(su), _p(vu), _p(cu),
                                             ctypes.byref(du), _p(sg), _p(vg), _p(cg), ctypes.byref(dg), M, H, _p(d_gate), pitch,
                                             _p(d_up), pitch, _stream()))
    return (d_gate, d_up) if room is None else (d_gate, d_up, both)


def _row_kernel_fits(H, bits, group, widths):
    return bits in widths and group in (64, 128) and H % (64 // bits) == 0 and H * bits // 64 <= 1024


def act_fwd_compress_supported(H, bits, group):
    """shapes the one-pass activation forward covers"""
    return _row_kernel_fits(H, bits, group, (2, 4, 8))


def hadamard_fwd_compress_supported(H, bits1, group1, bits2, group2):
    """shapes the one-pass product forward covers (two operands of 2-bit codes: at most 512 chunks per segment)"""
    return (bits1 == bits2 and group1 == group2 and _row_kernel_fits(H, bits1, group1, (2, 4, 8)) and
            (bits1 != 2 or H * bits1 // 64 <= 512))


def act_fwd_compress(act, x2d, plan, bits, group):
    """y = act(x) (F.silu / F.gelu values) and the compressed x from one read of x -> (y, ChannelCompressed)"""
    _need_rows(x2d, "x")
    M, H = x2d.shape
    c = alloc_channel(M, H, plan, bits, group, x2d.device)
    d = _checked_desc(plan, bits, group)
    y = torch.empty((M, H), dtype=BF16, device=x2d.device)
    code = ACT_CODES[act]
    check(_abi.load().hyc_act_fwd_compress(code, _p(x2d), x2d.stride(0) if M > 1 else H, M, H, ctypes.byref(d), _p(y),
                                           _p(c.stored), _p(c.vals), _p(c.scales), _stream()))
    return y, c


def hadamard_fwd_compress(a2d, b2d, plan_a, plan_b, bits, group):
    """y = a * b and both operands compressed, each read once -> (y, c_a, c_b)"""
    _need_rows(a2d, "x1")
    _need_rows(b2d, "x2")
    if a2d.shape != b2d.shape:
        raise ValueError("x1 %s and x2 %s differ in shape" % (tuple(a2d.shape), tuple(b2d.shape)))
    M, H = a2d.shape
    ca = alloc_channel(M, H, plan_a, bits, group, a2d.device)
    cb = alloc_channel(M, H, plan_b, bits, group, a2d.device)
    da, db = _checked_desc(plan_a, bits, group), _checked_desc(plan_b, bits, group)
    y = torch.empty((M, H), dtype=BF16, device=a2d.device)
    check(_abi.load().hyc_hadamard_fwd_compress(_p(a2d), a2d.stride(0) if M > 1 else H, _p(b2d), b2d.stride(0) if M > 1 else H,
                                                M, H, ctypes.byref(da), ctypes.byref(db), _p(y), _p(ca.stored), _p(ca.vals),
                                                _p(ca.scales), _p(cb.stored), _p(cb.vals), _p(cb.scales), _stream()))
    return y, ca, cb


def gated_act_fwd_supported(H, bits, group):
    """shapes the one-pass forward covers (the rest takes the activation, three compress calls and a product)"""
    if bits not in (2, 4, 8) or group not in (64, 128) or H % (64 // bits) != 0:
        return False
    chunks, most, lpg = H * bits // 64, 512 if bits == 2 else 768, group // 8
    # one workgroup per row, or 2 to 4 workgroups (whole scale groups each) for rows of up to 1024 chunks
    return chunks <= most or (chunks <= 1024 and any(chunks % n == 0 and (chunks // n) % lpg == 0 and
                                                     -(-(chunks // n) // 64) * 64 <= most for n in (2, 3, 4)))


def gated_act_fwd(act, gate2d, up2d, plan_act, plan_up, plan_gate, bits, group):
    """h = act(gate) * up and the compressed act(gate), up, gate in one pass -> (h, c_act, c_up, c_gate).
    gate and up are bf16 [M, H] matrices with contiguous rows (column slices of one projection output are fine);
    the plans are the outlier-channel sets of the three sites."""
    _need_rows(gate2d, "gate")
    _need_rows(up2d, "up")
    if gate2d.shape != up2d.shape:
        raise ValueError("gate %s and up %s differ in shape" % (tuple(gate2d.shape), tuple(up2d.shape)))
    M, H = gate2d.shape
    dev = gate2d.device
    outs = [alloc_channel(M, H, p, bits, group, dev) for p in (plan_act, plan_up, plan_gate)]
    descs = [_checked_desc(p, bits, group) for p in (plan_act, plan_up, plan_gate)]
    h = torch.empty((M, H), dtype=BF16, device=dev)
    code = ACT_CODES[act]
    flat = []
    for o in outs:
        flat += [_p(o.stored), _p(o.vals), _p(o.scales)]
    check(_abi.load().hyc_gated_act_fwd(code, _p(gate2d), gate2d.stride(0) if M > 1 else H, _p(up2d),
                                        up2d.stride(0) if M > 1 else H, M, H, ctypes.byref(descs[0]), ctypes.byref(descs[1]),
                                        ctypes.byref(descs[2]), _p(h), *flat, _stream()))
    return (h,) + tuple(outs)


# ----------------------------------------------------------------------------------------------------
# weight gradient
# ----------------------------------------------------------------------------------------------------
STAGED_GRADW_MIN_TILES = 96


def gradw_staged_by_default(N_out, H):
    """whether dW [N_out, H] from a channel-compressed activation restores x_hat first.  Every 256 output features
    decode the same activation tile again (about a fifth on top of the dense product's time), against one pass that
    writes x_hat and its second read.  Measured at 4096 and 16 384 tokens, H = 4096 and 11008, N_out = 256 ... 4096:
    the staged route wins from 96 output tiles of 256 x 256 on (N_out >= 1536 at H = 4096, >= 768 at H = 11008)."""
    return -(-N_out // 256) * (H // 256) >= STAGED_GRADW_MIN_TILES


def gradw_gemm(dy2d, src, out_dtype=BF16, alpha=1.0, out=None, beta=0.0, staged=None):
    """dW [N_out, H] = alpha * dy^T @ x_hat (+ beta * out); src as for rmsnorm_bwd.

    A compressed src is decoded inside the GEMM, or (`staged`; None = by `gradw_staged_by_default`, never for the
    few output features LoRA training has) restored once into a transient matrix for the same kernel's dense form."""
    _need_rows(dy2d, "grad_output")                # rows may be a column slice of a wider matrix (pitch = stride(0))
    M, N_out = dy2d.shape
    H = src.H if isinstance(src, (ChannelCompressed, ThresholdCompressed)) else src.shape[-1]
    if staged is None:
        staged = gradw_staged_by_default(N_out, H)
    if staged and isinstance(src, ChannelCompressed):
        src = decompress_channel(src)
    stored, vals, scales, d = _source(src, M, H)
    lib = _abi.load()
    if out is None:
        out = torch.empty((N_out, H), dtype=out_dtype, device=dy2d.device)
    elif (not out.is_cuda or not out.is_contiguous() or tuple(out.shape) != (N_out, H)
          or out.dtype not in (BF16, torch.float32)):
        raise ValueError("out must be a contiguous bf16 or fp32 [%d, %d] CUDA tensor" % (N_out, H))
    ws_bytes = lib.hyc_gradw_workspace_bytes(M, N_out, H)
    ws = torch.empty(ws_bytes // 4, dtype=torch.float32, device=dy2d.device) if ws_bytes else None
    code = _abi.DTYPE_F32 if out.dtype == torch.float32 else _abi.DTYPE_BF16
    check(lib.hyc_gradw_gemm(_p(dy2d), dy2d.stride(0) if M > 1 else N_out, _p(stored), _p(vals), _p(scales), M, N_out, H, ctypes.byref(d),
                             float(alpha), float(beta), _p(out), code, _p(ws), _stream()))
    return out


def gradw_rows_per_call(M, N_out, unit, src):
    """how many of N_out rows of dW, whole groups of `unit`, gradw_gemm takes at a time without another order of its sums (src as there)"""
    H = src.H if isinstance(src, ChannelCompressed) else src.shape[-1]
    d = _source(src, M, H)[3]
    return int(_abi.load().hyc_gradw_rows_per_call(M, N_out, unit, H, ctypes.byref(d)))


# ----------------------------------------------------------------------------------------------------
# softmax
# ----------------------------------------------------------------------------------------------------
@dataclass
class SparseRows:
    """probabilities above the threshold, CSR over the flattened leading dims"""
    row_ptr: torch.Tensor   # int32 [rows+1]
    cols: torch.Tensor      # int32 [nnz] (or the capacity a KeptBudget provided: row_ptr says what is in use)
    vals: torch.Tensor      # bf16 [nnz]
    shape: tuple
    total: Optional[torch.Tensor] = None   # int64 0-d on the device: the entries above the threshold (> cols.numel(): some were dropped)

    @property
    def rows(self):
        return self.row_ptr.numel() - 1


def slab_room(per_row, N):
    """entries per row of the forward's slab of kept probabilities where `per_row` are expected, or 0 to read y a second time
    instead.  A slab entry is written and read (8 bytes) where the second read of y costs 2 N bytes a row: worth it while twice the
    expected share fits an eighth of the row (N / 2 bytes of traffic for the average row)."""
    cap = max(32, (int(2 * per_row) + 31) // 32 * 32)
    return cap if cap <= max(32, N // 8) and cap <= N else 0


def _slab_entries(budget, N, longest=4096):
    """slab_room for what a budget has seen, 0 while it has seen nothing"""
    return 0 if budget is None or not budget.ready or N > longest else slab_room(budget.per_row, N)


def _csr_from_counts(lib, y2d, threshold, counts, budget=None, slab=None):
    rows, N = y2d.shape
    dev = y2d.device
    row_ptr, nnz, total = _csr_offsets(lib, counts, rows, budget)
    cols = torch.empty(nnz, dtype=torch.int32, device=dev)
    vals = torch.empty(nnz, dtype=BF16, device=dev)
    if slab is not None and nnz:
        check(lib.hyc_softmax_fill_slab(_p(y2d), rows, N, float(threshold), _p(counts), _p(slab), slab.shape[1], _p(row_ptr),
                                        _p(cols), _p(vals), _stream()))
        return row_ptr, cols, vals, total
    check(lib.hyc_softmax_fill(_p(y2d), rows, N, float(threshold), _p(row_ptr), _p(cols) if nnz else None,
                               _p(vals) if nnz else None, _stream()))
    return row_ptr, cols, vals, total


def softmax_fwd(x, threshold=None, causal_period=None, inplace=False, budget=None):
    """y = softmax(x, -1) bf16; with a threshold also the kept entries (y > bf16(threshold)) as SparseRows.
    budget: the site's KeptBudget (see there): once it has seen a call, the kept entries are sized ahead of time and the
    call returns without waiting for the GPU.
    causal_period = S applies the causal mask of S query positions inside the kernel (row r is position r % S).
    inplace: y overwrites x (rows of at most 4096 entries: a row is held in registers before anything is written)."""
    if threshold is not None and causal_period is None and not inplace and budget is not None and budget.ready:
        N, cap = x.shape[-1], _slab_entries(budget, x.shape[-1])
        if cap and x.numel():
            budget.poll()
            room = budget.capacity(x.numel() // N)
            done = native.softmax_fwd(x, float(threshold), cap, room)
            if done is not None:
                budget.watch(done[4], room, x.numel() // N)
                return done[0], SparseRows(done[1], done[2], done[3], tuple(x.shape), done[4])
    _need(x, BF16, "x")
    N = x.shape[-1]
    x2 = x.reshape(-1, N)
    rows = x2.shape[0]
    lib = _abi.load()
    if inplace and N > 4096:
        raise ValueError("in-place softmax needs rows of at most 4096 entries")
    y = x2 if inplace else torch.empty_like(x2)
    counts = None if threshold is None else torch.empty(rows, dtype=torch.int32, device=x.device)
    thr = 0.0 if threshold is None else float(threshold)
    slab, cap = None, 0 if threshold is None or rows == 0 else _slab_entries(budget, N)
    if cap and (causal_period is None or 0 < int(causal_period) <= N):
        slab = torch.empty((rows, cap), dtype=torch.int32, device=x.device)
        check(lib.hyc_softmax_fwd_slab(_p(x2), rows, N, int(causal_period or 0), thr, _p(y), _p(counts), _p(slab), cap, _stream()))
    elif causal_period is None:
        check(lib.hyc_softmax_fwd(_p(x2), rows, N, thr, _p(y), _p(counts), _stream()))
    else:
        check(lib.hyc_softmax_causal_fwd(_p(x2), rows, N, int(causal_period), thr, _p(y), _p(counts), _stream()))
    if threshold is None:
        return y.reshape(x.shape), None
    row_ptr, cols, vals, total = _csr_from_counts(lib, y, threshold, counts, budget, slab)
    return y.reshape(x.shape), SparseRows(row_ptr, cols, vals, tuple(x.shape), total)


def softmax_sparsify(y, threshold, budget=None):
    """kept entries of already computed probabilities (budget: as for softmax_fwd)"""
    _need(y, BF16, "y")
    N = y.shape[-1]
    y2 = y.reshape(-1, N)
    lib = _abi.load()
    counts = torch.empty(y2.shape[0], dtype=torch.int32, device=y.device)
    check(lib.hyc_softmax_fwd(None, y2.shape[0], N, float(threshold), _p(y2), _p(counts), _stream()))
    row_ptr, cols, vals, total = _csr_from_counts(lib, y2, threshold, counts, budget)
    return SparseRows(row_ptr, cols, vals, tuple(y.shape), total)


def softmax_bwd(g, sp: SparseRows, inplace=False):
    """dx = (g - sum(g * p_hat)) * p_hat; with inplace, dx overwrites g"""
    if not inplace and g.dim() and sp.shape[-1] == g.shape[-1]:
        dx = native.softmax_bwd(g, sp)
        if dx is not None:
            return dx
    _need(g, BF16, "grad_output")
    N = g.shape[-1]
    g2 = g.reshape(-1, N)
    if sp.rows != g2.shape[0] or sp.shape[-1] != N:
        raise ValueError("the kept probabilities are %s, the gradient is %s" % (tuple(sp.shape), tuple(g.shape)))
    dx = g2 if inplace else torch.empty_like(g2)
    check(_abi.load().hyc_softmax_bwd(_p(g2), g2.shape[0], N, _p(sp.row_ptr), _p(sp.cols) if sp.cols.numel() else None,
                                      _p(sp.vals) if sp.vals.numel() else None, _p(dx), _stream()))
    return dx.reshape(g.shape)


def softmax_dense(sp: SparseRows):
    N = sp.shape[-1]
    out = torch.empty((sp.rows, N), dtype=BF16, device=sp.row_ptr.device)
    check(_abi.load().hyc_softmax_dense(sp.rows, N, _p(sp.row_ptr), _p(sp.cols) if sp.cols.numel() else None,
                                        _p(sp.vals) if sp.vals.numel() else None, _p(out), _stream()))
    return out.reshape(sp.shape)


def sparse_rows_to_coo(sp: SparseRows):
    """the sparse COO tensor `.to_sparse()` gives for the pruned probabilities (int64 indices, row-major)"""
    counts = (sp.row_ptr[1:] - sp.row_ptr[:-1]).long()
    rows = torch.repeat_interleave(torch.arange(sp.rows, device=counts.device), counts)
    lead = []
    for dim in reversed(sp.shape[:-1]):
        lead.append(rows % dim)
        rows = rows // dim
    idx = torch.stack(list(reversed(lead)) + [sp.cols.long()])
    return torch.sparse_coo_tensor(idx, sp.vals, sp.shape, is_coalesced=True)


def coo_to_sparse_rows(coo):
    coo = coo.coalesce()
    shape = tuple(coo.shape)
    idx = coo.indices()
    rows = torch.zeros_like(idx[0])
    for i, dim in enumerate(shape[:-1]):
        rows = rows * dim + idx[i]
    n_rows = 1
    for dim in shape[:-1]:
        n_rows *= dim
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int32, device=idx.device)
    if rows.numel():
        torch.cumsum(torch.bincount(rows, minlength=n_rows), 0, out=row_ptr[1:])
    return SparseRows(row_ptr, idx[-1].to(torch.int32).contiguous(), coo.values().to(BF16).contiguous(), shape)


def softmax_sparse_coo(y, threshold):
    return sparse_rows_to_coo(softmax_sparsify(y, threshold))


def sparse_coo_to_dense(coo):
    return softmax_dense(coo_to_sparse_rows(coo))


def softmax_prune(y, threshold):
    """y * (y > threshold) as a dense tensor (the reference's prune_softmax; not used by the softmax operator)"""
    return softmax_dense(softmax_sparsify(y, threshold))


# ----------------------------------------------------------------------------------------------------
# low-rank base
# ----------------------------------------------------------------------------------------------------
def low_rank_update(l, r, x, subtract, out=None):
    """out = bf16(x -/+ l @ r), x [B,S,H] (or [S,H]); in place when out is x"""
    _need(x, BF16, "x")
    _need(l, BF16, "l")
    _need(r, BF16, "r")
    S, H = x.shape[-2], x.shape[-1]
    M = x.numel() // H
    if l.shape[0] != S or r.shape[0] != l.shape[1] or r.shape[1] != H:
        raise ValueError("Incompatible dimensions")
    if out is None:
        out = torch.empty_like(x)
    elif _need(out, BF16, "out").shape != x.shape:
        raise ValueError("out must have x's shape")
    check(_abi.load().hyc_low_rank_update(_p(l), _p(r), _p(x), _p(out), M, S, H, l.shape[1], 1 if subtract else 0, _stream()))
    return out


# ----------------------------------------------------------------------------------------------------
# NF4 frozen base weights
# ----------------------------------------------------------------------------------------------------
@dataclass
class NF4Weight:
    """a frozen [out, in] bf16 weight held as 4-bit level indices + one fp32 abs-max per 64 consecutive weights"""
    packed: torch.Tensor   # uint8 [out*in/2]
    absmax: torch.Tensor   # fp32 [out*in/64]
    shape: tuple

    def nbytes(self):
        return self.packed.numel() + 4 * self.absmax.numel()


def nf4_quantize(w):
    _need(w, BF16, "w")
    n = w.numel()
    if n % 64:
        raise ValueError("NF4 blocks hold 64 weights: %d is not a multiple of 64" % n)
    packed = torch.empty(n // 2, dtype=torch.uint8, device=w.device)
    absmax = torch.empty(n // 64, dtype=torch.float32, device=w.device)
    check(_abi.load().hyc_nf4_quantize(_p(w), n, _p(packed), _p(absmax), _stream()))
    return NF4Weight(packed, absmax, tuple(w.shape))


def nf4_dequantize(q: NF4Weight, out=None):
    n = q.packed.numel() * 2
    if out is None:
        out = torch.empty(q.shape, dtype=BF16, device=q.packed.device)
    elif _need(out, BF16, "out").numel() != n:
        raise ValueError("out must hold %d weights" % n)
    check(_abi.load().hyc_nf4_dequantize(_p(q.packed), _p(q.absmax), n, _p(out), _stream()))
    return out


# ----------------------------------------------------------------------------------------------------
# LoRA beside a frozen NF4 base
# ----------------------------------------------------------------------------------------------------
def lora_room(n, r):
    """columns appended to the reduction of a group's input gradient for its n * r rank columns: whole steps of 64"""
    return -(-n * r // 64) * 64


def _lora_factors(factors, shapes, device, name):
    """every factor of a group is a bf16 matrix of its shape on `device` (the kernels index them by those shapes alone), else
    ValueError; True if all of them also lie as the kernels read them: contiguous, at multiples of 16 bytes"""
    if len(factors) != len(shapes):
        raise ValueError("%d factors %s for %d projections" % (len(factors), name, len(shapes)))
    as_read = True
    for f, shape in zip(factors, shapes):
        if not isinstance(f, torch.Tensor) or f.dtype is not BF16 or f.device != device or f.shape != shape:
            what = "%s %s on %s" % (f.dtype, tuple(f.shape), f.device) if isinstance(f, torch.Tensor) else type(f).__name__
            raise ValueError("%s must be bfloat16 %s on %s, got %s" % (name, tuple(shape), device, what))
        if f.data_ptr() % 16 or not f.is_contiguous():
            as_read = False
    return as_read


@functools.lru_cache(maxsize=256)
def _lora_kernels_cover(M, n, r, K, outs):
    """what the hyc_lora_* entries take: up to 4 factors of rank 8 to 32, and no more tokens and features than their launches count"""
    return (n <= 4 and r in (8, 16, 24, 32) and n * r <= 96 and K % 64 == 0 and K <= 1 << 24 and M <= 65535 * 128
            and sum(outs) <= 65535 * 128 - 4096 and all(o % 8 == 0 and o for o in outs))


def _lora_range_fits(M, pitch):
    """a token range of hyc_lora_up_bwd (at most 32768 tokens; rounded up to 64, twice its tile: a margin) stays below 2 GiB of rows
    `pitch` apart, however many ranges there are"""
    return (min(M, 32768) + 63) // 64 * 64 * pitch < 1 << 30


def _ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _i64s(vs):
    return (ctypes.c_int64 * len(vs))(*vs)


def lora_down(x2d, A):
    """h [M, n r] = x A_i^T side by side"""
    _need_rows(x2d, "x")
    M, Kf = x2d.shape
    n, r = len(A), A[0].shape[0]
    as_read = _lora_factors(A, [(r, Kf)] * n, x2d.device, "A")
    if not as_read or not _lora_kernels_cover(M, n, r, Kf, ()):
        return x2d @ torch.cat(list(A), dim=0).t()
    h = torch.empty((M, n * r), dtype=BF16, device=x2d.device)
    check(_abi.load().hyc_lora_down(_p(x2d), x2d.stride(0) if M > 1 else Kf, M, Kf, _ptrs(A), n, r, _p(h), _stream()))
    return h


def _thin(rows, w, input_grad):
    """whether `rows` (x or dY of a linear layer with weight w) and w are what the kernels for few output features take and read as they lie"""
    plain = (torch.Tensor, torch.nn.Parameter)
    return (type(rows) in plain and type(w) in plain and torch._C._has_storage(rows) and torch._C._has_storage(w)     # (no functorch wrapper)
            and rows.dtype is BF16 and w.dtype is BF16 and rows.is_cuda and rows.device == w.device and rows.numel() and rows.dim() >= 2 and w.dim() == 2 and not torch.is_grad_enabled() and rows.shape[-1] == w.shape[0 if input_grad else 1]
            and rows.is_contiguous() and w.is_contiguous() and rows.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and rows.device.index == torch.cuda.current_device()
            and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") is BF16)     # (else the product's result has its type)
            and bool(_abi.load().hyc_thin_covers(rows.numel() // rows.shape[-1], w.shape[1], w.shape[0], input_grad)))


def linear_fwd(x, w):
    """x w^T"""
    if not _thin(x, w, False):
        return x @ w.transpose(0, 1)
    y = torch.empty((*x.shape[:-1], w.shape[0]), dtype=BF16, device=x.device)
    M, Kf = x.numel() // w.shape[1], w.shape[1]
    check(_abi.load().hyc_lora_down(_p(x), Kf, M, Kf, _ptrs([w]), 1, w.shape[0], _p(y), _stream()))
    return y


def linear_dx(g, w):
    """g w"""
    if not _thin(g, w, True):
        return g @ w
    dx = torch.empty((*g.shape[:-1], w.shape[1]), dtype=BF16, device=g.device)
    check(_abi.load().hyc_thin_dx(_p(g), w.shape[0], g.numel() // w.shape[0], _p(w), w.shape[0], w.shape[1], _p(dx), _stream()))
    return dx


def _need_h(h, M, width):
    _need(h, BF16, "h")
    if h.shape != (M, width):
        raise ValueError("h must be [%d, %d], got %s" % (M, width, tuple(h.shape)))
    return h


def lora_up(h, B, scale, outs=None):
    """y [M, sum(out_i)] = scale * h_i B_i^T side by side.  outs: the widths out_i the factors must have (None: as they come)"""
    n, r = len(B), B[0].shape[-1]
    outs = [b.shape[0] for b in B] if outs is None else list(outs)
    M = h.shape[0]
    _need_h(h, M, n * r)
    as_read = _lora_factors(B, [(o, r) for o in outs], h.device, "B")
    y = torch.empty((M, sum(outs)), dtype=BF16, device=h.device)
    if as_read and _lora_kernels_cover(M, n, r, 64, tuple(outs)):
        check(_abi.load().hyc_lora_up(_p(h), M, _ptrs(B), _i64s(outs), n, r, float(scale), _p(y), _stream()))
        return y
    zero, col = h.new_zeros(1), 0
    for i, (b, o) in enumerate(zip(B, outs)):
        torch.addmm(zero, h[:, i * r:(i + 1) * r], b.t(), beta=0.0, alpha=scale, out=y[:, col:col + o])
        col += o
    return y


def few_rows_base(x2, base, h, B, scale, outs):
    """y [M, sum(outs)] = scale * h_i B_i^T + x W^T in one launch from the codes of W, or None where the products take other forms
    (hyc_few_rows_covers, and what the launch reads)"""
    (M, H), n, total = x2.shape, len(outs), sum(outs)
    r, pitch = h.shape[-1] // n, x2.stride(0) if M > 1 else H
    if not M or any(o % 16 for o in outs) or not _lora_kernels_cover(M, n, r, H, tuple(outs)) or h.shape != (M, n * r):
        return None
    if (x2.dtype != BF16 or not x2.is_cuda or x2.data_ptr() % 16 or x2.stride(1) != 1 or pitch < H or pitch % 8 or M * pitch >= 1 << 30
            or any(t.dtype != dt or t.numel() * per != total * H or t.device != x2.device or not t.is_contiguous() or t.data_ptr() % 16
                   for t, dt, per in ((base.packed, torch.uint8, 2), (base.absmax, torch.float32, 64)))):
        return None
    lib = _abi.load()
    if not lib.hyc_few_rows_covers(M, H, total, 0) or not _lora_factors(B, [(o, r) for o in outs], x2.device, "B"):
        return None
    _need(h, BF16, "h")
    y = torch.empty((M, total), dtype=BF16, device=x2.device)
    check(lib.hyc_few_rows_nf4(_p(x2), pitch, M, H, _p(base.packed), _p(base.absmax), _p(h), _ptrs(B), _i64s(outs), n, r, float(scale), _p(y), _stream()))
    return y


def few_rows(out, a, b):
    """out [M, N] = a @ b^T in one launch where that is better than a library product (hyc_few_rows_covers); whether it was"""
    (M, H), N = a.shape, b.shape[0]
    if any(t.dtype != BF16 or not t.is_cuda or not t.is_contiguous() or t.data_ptr() % 16 for t in (out, a, b)):
        return False
    lib = _abi.load()
    if not lib.hyc_few_rows_covers(M, H, N, 1):
        return False
    check(lib.hyc_few_rows(_p(a), H, M, H, _p(b), N, _p(out), _stream()))
    return True


def lora_up_bwd(gs, B, h, scale, room, ext=None):
    """(ext, dh, [dB_i]) from the gradients gs[i] [M, out_i] of a group: dB_i = scale * gs[i]^T h_i, dh = scale * gs[i] B_i
    side by side [M, n r] and, with zeros behind them, as the columns [sum(outs), + room) of ext.  ext: the buffer the gs
    already are the first columns of, side by side; None: they are copied into a new one."""
    M, n, r = gs[0].shape[0], len(gs), B[0].shape[-1]
    for g in gs:
        _need_rows(g, "grad_output")
        if g.shape[0] != M or g.device != h.device:
            raise ValueError("the gradients of a group must have the same rows, on the device of h")
    outs = [g.shape[1] for g in gs]
    total = sum(outs)
    as_read = _lora_factors(B, [(o, r) for o in outs], h.device, "B")
    _need_h(h, M, n * r)
    if room < n * r:
        raise ValueError("room for %d columns, the group has %d" % (room, n * r))
    copy = ext is None
    if copy:
        ext = torch.empty((M, total + room), dtype=BF16, device=h.device)
    else:
        _need(ext, BF16, "ext")
        if ext.shape != (M, total + room) or ext.device != h.device:
            raise ValueError("ext must be [%d, %d] on %s, got %s on %s" % (M, total + room, h.device, tuple(ext.shape), ext.device))
    if M and as_read and _lora_kernels_cover(M, n, r, 64, tuple(outs)) and _lora_range_fits(M, max(max(g.stride(0), o) for g, o in zip(gs, outs))):
        lib = _abi.load()
        dh = torch.empty((M, n * r), dtype=BF16, device=h.device)
        dB = [torch.empty_like(b) for b in B]
        outs_c = _i64s(outs)
        ws = torch.empty(lib.hyc_lora_up_bwd_workspace_bytes(M, outs_c, n, r) // 4, dtype=torch.float32, device=h.device)
        pitches = _i64s([g.stride(0) if M > 1 else o for g, o in zip(gs, outs)])
        check(lib.hyc_lora_up_bwd(_ptrs(gs), pitches, M, outs_c, _ptrs(B), _p(h), n, r, float(scale), _p(dh), _p(ext), total + room, room,
                                  1 if copy else 0, _ptrs(dB), _p(ws), _stream()))
        return ext, dh, dB
    zero = h.new_zeros(1)
    dh = torch.cat([torch.addmm(zero, g, b, beta=0.0, alpha=scale) for g, b in zip(gs, B)], dim=1)
    dB = [torch.addmm(zero, g.t(), h[:, i * r:(i + 1) * r], beta=0.0, alpha=scale) for i, g in enumerate(gs)]
    if copy:
        col = 0
        for g, o in zip(gs, outs):
            ext[:, col:col + o] = g
            col += o
    ext[:, total:] = 0
    ext[:, total:total + n * r] = dh
    return ext, dh, dB


def lora_weight_t(q: NF4Weight, A, outs, room):
    """[K, sum(outs) + room] = [W^T | A_i^T side by side | zeros]: the transposed weight of the group's input gradient"""
    total, Kf = q.shape
    n, r = len(A), A[0].shape[0]
    if sum(outs) != total or len(outs) != n:
        raise ValueError("%d projections of %s features in a weight of %s with %d factors" % (len(outs), list(outs), tuple(q.shape), n))
    _need_vec(q.packed, torch.uint8, total * Kf // 2, "packed")
    _need_vec(q.absmax, torch.float32, total * Kf // 64, "absmax")
    as_read = _lora_factors(A, [(r, Kf)] * n, q.packed.device, "A")
    if room < n * r:
        raise ValueError("room for %d columns, the group has %d" % (room, n * r))
    out = torch.empty((Kf, total + room), dtype=BF16, device=q.packed.device)
    if as_read and _lora_kernels_cover(0, n, r, Kf, tuple(outs)):
        check(_abi.load().hyc_lora_weight_t(_p(q.packed), _p(q.absmax), Kf, _ptrs(A), _i64s(outs), n, r, room, _p(out), _stream()))
        return out
    out[:, :total], out[:, total:] = nf4_dequantize(q).t(), 0
    out[:, total:total + n * r] = torch.cat(list(A), dim=0).t()
    return out


# ----------------------------------------------------------------------------------------------------
# rotary embedding + attention layout
# ----------------------------------------------------------------------------------------------------
def _need_tables(cos, sin, S, hd):
    if (cos is None) != (sin is None):
        raise ValueError("cos and sin go together")
    if cos is not None:
        _need_vec(cos, BF16, S * hd, "cos")
        _need_vec(sin, BF16, S * hd, "sin")


def rope_to_heads(x, heads, cos=None, sin=None, want_rows=False):
    """x bf16 [B, S, heads*hd] -> rotated [B, heads, S, hd] contiguous (and, with want_rows, also [B, S, heads*hd]);
    cos / sin bf16 [S, hd]; without them only the layout changes.  x may be a column slice of a wider [B, S, *]
    tensor (tokens a fixed pitch apart)."""
    if not isinstance(x, torch.Tensor) or not x.is_cuda or x.dtype != BF16 or x.dim() != 3:
        raise ValueError("x must be a bfloat16 [B, S, H] tensor on the GPU")
    B, S, H = x.shape
    pitch = x.stride(1) if S > 1 else H
    if x.stride(2) != 1 or (B > 1 and x.stride(0) != S * pitch):
        raise ValueError("x must have contiguous channels and evenly spaced tokens")
    if heads <= 0 or H % heads:
        raise ValueError("%d channels do not split into %d heads" % (H, heads))
    hd = H // heads
    _need_tables(cos, sin, S, hd)
    out_heads = torch.empty((B, heads, S, hd), dtype=BF16, device=x.device)
    out_rows = torch.empty((B, S, H), dtype=BF16, device=x.device) if want_rows else None
    check(_abi.load().hyc_rope_to_heads(_p(x), pitch, _p(cos), _p(sin), B, S, heads, hd, _p(out_heads), _p(out_rows),
                                        _stream()))
    return (out_heads, out_rows) if want_rows else out_heads


def _need_tokens(x, name):
    """(B, S, H, pitch) of a bf16 [B, S, H] tensor with contiguous channels and evenly spaced tokens"""
    if not isinstance(x, torch.Tensor) or not x.is_cuda or x.dtype != BF16 or x.dim() != 3:
        raise ValueError("%s must be a bfloat16 [B, S, H] tensor on the GPU" % name)
    B, S, H = x.shape
    pitch = x.stride(1) if S > 1 else (x.stride(0) if B > 1 else H)
    if x.stride(2) != 1 or (B > 1 and x.stride(0) != S * pitch):
        raise ValueError("%s must have contiguous channels and evenly spaced tokens" % name)
    return B, S, H, pitch


def rope_rows(x, heads, cos, sin):
    """x bf16 [B, S, heads*hd], possibly a column slice of a wider matrix -> the rotated rows, contiguous"""
    B, S, H, pitch = _need_tokens(x, "x")
    if heads <= 0 or H % heads:
        raise ValueError("%d channels do not split into %d heads" % (H, heads))
    hd = H // heads
    _need_tables(cos, sin, S, hd)
    out = torch.empty((B, S, H), dtype=BF16, device=x.device)
    check(_abi.load().hyc_rope_to_heads(_p(x), pitch, _p(cos), _p(sin), B, S, heads, hd, None, _p(out), _stream()))
    return out


def rope_from_heads(g, cos=None, sin=None):
    """gradient bf16 [B, heads, S, hd] -> [B, S, heads*hd] through the transposed rotation"""
    _need(g, BF16, "g")
    B, heads, S, hd = g.shape
    _need_tables(cos, sin, S, hd)
    out = torch.empty((B, S, heads * hd), dtype=BF16, device=g.device)
    check(_abi.load().hyc_rope_from_heads(_p(g), _p(cos), _p(sin), B, S, heads, hd, _p(out), _stream()))
    return out


# ----------------------------------------------------------------------------------------------------
# fused causal attention
# ----------------------------------------------------------------------------------------------------
def attn_supported(head_dim, S, widest_pitch, matrices=1):
    """shapes hyc_attn_fwd / hyc_attn_bwd cover (the library's fused attention serves the others); matrices: B * heads"""
    return head_dim in (64, 128) and S * widest_pitch < 1 << 30 and matrices * -(-S // 128) < 1 << 24


def attn_fwd(q, k, v, heads, scale, round_scores=False):
    """causal softmax(scale q k^T) v on [B, S, heads*hd] rows -> (out [B, S, heads*hd], lse fp32 [B, heads, S]); round_scores: from
    scores rounded to bf16, as attn_kept takes them, and with probabilities rounded once they are normalised, as it keeps them"""
    B, S, H, pq = _need_tokens(q, "q")
    pk, pv = _need_tokens(k, "k")[3], _need_tokens(v, "v")[3]
    if tuple(k.shape) != (B, S, H) or tuple(v.shape) != (B, S, H) or H % heads:
        raise ValueError("q, k, v must be [B, S, heads*hd] alike, got %s, %s, %s" % (tuple(q.shape), tuple(k.shape), tuple(v.shape)))
    out = torch.empty((B, S, H), dtype=BF16, device=q.device)
    lse = torch.empty((B, heads, S), dtype=torch.float32, device=q.device)
    lib = _abi.load()
    entry = lib.hyc_attn_kept_fwd if round_scores else lib.hyc_attn_fwd
    check(entry(_p(q), pq, _p(k), pk, _p(v), pv, B, S, heads, H // heads, float(scale), _p(out), H, _p(lse), _stream()))
    return out, lse


def _grad_rows(g, room):
    """((dq, dk, dv), pitch): empty gradients like g, or with `room` side by side in a matrix that comes as a fourth"""
    B, S, H = g.shape
    if room is None:
        return tuple(torch.empty((B, S, H), dtype=BF16, device=g.device) for _ in range(3)), H
    both = torch.empty((B * S, 3 * H + room), dtype=BF16, device=g.device)
    return tuple(both[:, i * H:(i + 1) * H].unflatten(0, (B, S)) for i in range(3)) + (both,), 3 * H + room


def attn_bwd(g, q, k, v, out, lse, heads, scale, cos=None, sin=None, room=None):
    """(dq, dk, dv) of attn_fwd at the given q, k, v, out and lse; with cos / sin the gradients of q and k before their
    rotation.  With `room` (a number of columns, 0 included) the three lie side by side in one [B*S, 3 H + room] matrix,
    returned as a fourth value."""
    B, S, H, pg = _need_tokens(g, "g")
    ptrs = []
    for name, t in (("q", q), ("k", k), ("v", v), ("out", out)):
        if tuple(t.shape) != (B, S, H):
            raise ValueError("%s is %s, the gradient is %s" % (name, tuple(t.shape), tuple(g.shape)))
        ptrs += [_p(t), _need_tokens(t, name)[3]]
    _need_vec(lse, torch.float32, B * heads * S, "lse")
    _need_tables(cos, sin, S, H // heads)
    grads, pitch = _grad_rows(g, room)
    ws = torch.empty(2 * B * heads * S, dtype=torch.float32, device=g.device)
    check(_abi.load().hyc_attn_bwd(_p(g), pg, *ptrs, _p(lse), _p(cos), _p(sin), B, S, heads, H // heads, float(scale),
                                   _p(grads[0]), pitch, _p(grads[1]), pitch, _p(grads[2]), pitch, _p(ws), _stream()))
    return grads


def _attn_kept_shape(threshold, S, head_dim):
    # (the kernels compare with the threshold rounded to bf16, which has to stay above 1e-30 and below 1: 0.998 rounds to 0.996, 0.9981 to 1)
    return head_dim in (64, 128) and S % 8 == 0 and 0 < S <= 4096 and 1e-29 < threshold <= 0.998


def attn_kept_covers(threshold, S, head_dim, share):
    """whether attn_kept, and not scores and probabilities as matrices, serves a calibrated site that is to keep `share` of its
    probabilities: not with a threshold that keeps every positive one, not for rows the softmax kernels refuse, and up to a share of a
    sixteenth (the entry-by-entry half of the backward grows with it: attention at 1 x 2048 x 32 heads x 128 in us, with matrices /
    here: 1 % kept 869 / 386, 3 % 901 / 550, 6 % 926 / 770).  The two forms do not give the same bits (sums in another order, dS rounded
    for dk only), so nothing that depends on a run's timing enters: share is the configured one, not what a KeptBudget has seen."""
    return _attn_kept_shape(threshold, S, head_dim) and slab_room(share * S, S) > 0


def attn_kept_entries(budget, threshold, S, head_dim):
    """slab entries per row for a site of this budget, or 0: nothing seen yet, more kept than a slab is worth, or rows and thresholds
    attn_kept does not take"""
    return _slab_entries(budget, S) if _attn_kept_shape(threshold, S, head_dim) else 0


def attn_kept(q, k, lse, heads, scale, threshold, budget, cap, first, matrices):
    """the probabilities exp(bf16(scale q k^T) - lse) above the threshold of matrices [first, first + matrices) as SparseRows; lse:
    attn_fwd's with round_scores; cap: slab entries per row (rows that keep more are formed a second time, with the same result)"""
    if budget is not None and budget.ready and q.dim() == 3:
        rows = matrices * q.shape[1]
        budget.poll()
        room = budget.capacity(rows)
        done = native.attn_kept(q, k, lse, heads, scale, threshold, cap, room, first, matrices)
        if done is not None:
            budget.watch(done[3], room, rows)
            return SparseRows(done[0], done[1], done[2], (matrices, q.shape[1], q.shape[1]), done[3])
    B, S, H, pq = _need_tokens(q, "q")
    pk = _need_tokens(k, "k")[3]
    if tuple(k.shape) != (B, S, H) or H % heads:
        raise ValueError("q and k must be [B, S, heads*hd] alike, got %s, %s" % (tuple(q.shape), tuple(k.shape)))
    _need_vec(lse, torch.float32, B * heads * S, "lse")
    lib, rows, dev = _abi.load(), matrices * S, q.device
    counts = torch.empty(rows, dtype=torch.int32, device=dev)
    slab = torch.empty((rows, cap), dtype=torch.int32, device=dev)
    args = (_p(q), pq, _p(k), pk, _p(lse), B, S, heads, H // heads, float(scale), float(threshold), first, matrices, _p(counts), _p(slab), cap)
    check(lib.hyc_attn_kept(*args, _stream()))
    row_ptr, nnz, total = _csr_offsets(lib, counts, rows, budget)
    cols = torch.empty(nnz, dtype=torch.int32, device=dev)
    vals = torch.empty(nnz, dtype=BF16, device=dev)
    if nnz:
        check(lib.hyc_attn_kept_fill(*args, _p(row_ptr), _p(cols), _p(vals), _stream()))
    return SparseRows(row_ptr, cols, vals, (matrices, S, S), total)


def attn_kept_bwd(g, q, k, v, kept, heads, scale, cos=None, sin=None, room=None):
    """(dq, dk, dv) of causal attention at the given q, k, v with the probabilities in `kept` (SparseRows of consecutive ranges
    of matrices, all of them together); cos / sin and room as in attn_bwd"""
    B, S, H, pg = _need_tokens(g, "g")
    ptrs = []
    for name, t in (("q", q), ("k", k), ("v", v)):
        if tuple(t.shape) != (B, S, H):
            raise ValueError("%s is %s, the gradient is %s" % (name, tuple(t.shape), tuple(g.shape)))
        ptrs += [_p(t), _need_tokens(t, name)[3]]
    if H % heads or sum(sp.rows for sp in kept) != B * heads * S or any(sp.rows % S or sp.shape[-1] != S for sp in kept):
        raise ValueError("the kept probabilities are %s, the gradient is %s" % ([tuple(sp.shape) for sp in kept], tuple(g.shape)))
    _need_tables(cos, sin, S, H // heads)
    grads, pitch = _grad_rows(g, room)
    at, first = [_p(t) for t in grads], 0
    for sp in kept:
        matrices, n = sp.rows // S, sp.cols.numel()
        _need_vec(sp.row_ptr, torch.int32, sp.rows + 1, "row_ptr")
        _need_vec(sp.cols, torch.int32, n, "cols")
        _need_vec(sp.vals, BF16, n, "vals")
        records = torch.empty((max(n, 1), 2), dtype=torch.int32, device=g.device)
        check(_abi.load().hyc_attn_kept_bwd(_p(g), pg, *ptrs, _p(sp.row_ptr), _p(sp.cols) or _p(records), _p(sp.vals) or _p(records), _p(cos),
                                            _p(sin), B, S, heads, H // heads, float(scale), first, matrices, at[0], pitch, at[1], pitch,
                                            at[2], pitch, _p(records), _stream()))
        first += matrices
    return grads


# ----------------------------------------------------------------------------------------------------
# seeded dropout
# ----------------------------------------------------------------------------------------------------
def dropout(x, p, seed, backward=False):
    """forward: keep ? x / (1 - p) : 0; backward: keep ? x : 0; keep is a pure function of (seed, element index)"""
    _need(x, BF16, "x")
    out = torch.empty_like(x)
    check(_abi.load().hyc_dropout(_p(x), _p(out), x.numel(), float(p), int(seed) & 0xFFFFFFFFFFFFFFFF,
                                  1 if backward else 0, _stream()))
    return out
