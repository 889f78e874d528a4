"""Tensor-level entry points of the HIP optimizer kernels (current stream, no synchronisation)."""
from __future__ import annotations

import ctypes
import math
import os

import torch

from .. import _lib
from ..kernels.launch import device_guard, stream_handle

NS_COEFFICIENTS = (3.4445, -4.7750, 2.0315)
NS_EPS = 1e-7
NS_STEPS = 5

_DTYPE_CODES = {torch.float32: _lib.DT_F32, torch.bfloat16: _lib.DT_BF16}


def adjust_lr(lr: float, adjust_lr_fn: str | None, param_shape) -> float:
    """Muon's shape-dependent learning-rate factor (torch/optim/_muon.py:73-84)."""
    rows, cols = param_shape[:2]
    if adjust_lr_fn is None or adjust_lr_fn == "original":
        ratio = math.sqrt(max(1, rows / cols))
    elif adjust_lr_fn == "match_rms_adamw":
        ratio = 0.2 * math.sqrt(max(rows, cols))
    else:
        ratio = 1.0
    return lr * ratio


def muon_workspace_bytes(rows: int, cols: int) -> int:
    n = int(_lib.lib().mfsdp_muon_workspace_bytes(rows, cols))
    if n <= 0:
        raise ValueError("Param gradient must be a 2D matrix")
    return n


class MuonWorkspace:
    """Scratch memory for the Newton-Schulz iteration, grown on demand and
    reused across matrices (the kernels themselves never allocate)."""

    def __init__(self, device) -> None:
        self.device = torch.device(device)
        self.buffer: torch.Tensor | None = None

    def get(self, rows: int, cols: int) -> torch.Tensor:
        return self.get_bytes(muon_workspace_bytes(rows, cols))

    def get_bytes(self, need: int) -> torch.Tensor:
        if self.buffer is None or self.buffer.numel() < need:
            self.buffer = None  # release before growing
            self.buffer = torch.empty(need, dtype=torch.uint8, device=self.device)
        return self.buffer


def _check_matrix(t: torch.Tensor, what: str) -> None:
    if t.ndim != 2:
        raise ValueError("Param gradient must be a 2D matrix" if what == "grad" else f"{what} must be a 2D matrix")
    if not t.is_cuda or not t.is_contiguous():
        raise RuntimeError(f"{what} must be a contiguous CUDA tensor")
    if t.dtype not in _DTYPE_CODES:
        raise RuntimeError(f"{what} must be float32 or bfloat16, got {t.dtype}")


def _check_step(param: torch.Tensor, grad: torch.Tensor, momentum_buf: torch.Tensor, ns_steps: int) -> None:
    if grad.ndim != 2:
        raise ValueError("Param gradient must be a 2D matrix")
    for t, what in ((param, "param"), (grad, "grad"), (momentum_buf, "momentum buffer")):
        _check_matrix(t, what)
    if not (param.dtype == grad.dtype == momentum_buf.dtype):
        # Tensor.lerp_ rejects mixed dtypes; the reference's local shard, grad shard and state share one dtype
        raise RuntimeError(f"param, grad and momentum buffer must share a dtype, got {param.dtype}, {grad.dtype}, {momentum_buf.dtype}")
    if not (param.shape == grad.shape == momentum_buf.shape):
        raise RuntimeError("param, grad and momentum buffer must share a shape")
    if ns_steps >= 100:
        raise ValueError("Number of steps must be less than 100 for computational efficiency")


def newton_schulz(
    update: torch.Tensor,
    ns_coefficients=NS_COEFFICIENTS,
    ns_steps: int = NS_STEPS,
    eps: float = NS_EPS,
    *,
    workspace: MuonWorkspace | None = None,
    out: torch.Tensor | None = None,
) -> torch.Tensor:
    """bf16 orthogonalisation of ``update`` (torch/optim/_muon.py:31-70)."""
    if ns_steps >= 100:
        raise ValueError("Number of steps must be less than 100 for computational efficiency")
    if update.ndim != 2:
        raise ValueError("Input tensor gradient must be a 2D matrix")
    if len(ns_coefficients) != 3:
        raise ValueError("Coefficients must be a tuple of exactly 3 values")
    _check_matrix(update, "update")
    rows, cols = update.shape
    workspace = workspace or MuonWorkspace(update.device)
    ws = workspace.get(rows, cols)
    if out is None:
        out = torch.empty((rows, cols), dtype=torch.bfloat16, device=update.device)
    a, b, c = ns_coefficients
    stream = stream_handle(update.device)
    with device_guard(update.device):
        _lib.check(
            _lib.lib().mfsdp_newton_schulz(
                update.data_ptr(), _DTYPE_CODES[update.dtype], rows, cols, a, b, c, ns_steps, eps,
                out.data_ptr(), ws.data_ptr(), ws.numel(), stream,
            )
        )
    return out


def muon_step(
    param: torch.Tensor,
    grad: torch.Tensor,
    momentum_buf: torch.Tensor,
    *,
    lr: float,
    weight_decay: float,
    momentum: float,
    nesterov: bool,
    ns_coefficients=NS_COEFFICIENTS,
    ns_steps: int = NS_STEPS,
    eps: float = NS_EPS,
    adjust_lr_fn: str | None = None,
    workspace: MuonWorkspace | None = None,
    shared_machine: bool = False,
) -> None:
    """One matrix of ``_single_tensor_muon`` (torch/optim/_muon.py:285-318), in
    place on ``param`` and ``momentum_buf``.  ``shared_machine`` tells the
    kernels that the caller updates other matrices on other streams at the same
    time."""
    _check_step(param, grad, momentum_buf, ns_steps)
    rows, cols = param.shape
    workspace = workspace or MuonWorkspace(param.device)
    ws = workspace.get(rows, cols)
    a, b, c = ns_coefficients
    stream = stream_handle(param.device)
    with device_guard(param.device):
        _lib.check(
            _lib.lib().mfsdp_muon_step_ex(
                param.data_ptr(), grad.data_ptr(), momentum_buf.data_ptr(), _DTYPE_CODES[param.dtype], rows, cols,
                lr, weight_decay, momentum, int(bool(nesterov)), a, b, c, ns_steps, eps,
                adjust_lr(lr, adjust_lr_fn, param.shape), _lib.MUON_SHARED_MACHINE if shared_machine else 0,
                ws.data_ptr(), ws.numel(), stream,
            )
        )


class MuonStreamPool:
    """Side streams (default priority) with one Newton-Schulz workspace each, for a caller that wants independent matrices
    updated on streams of its own (``muon_step_many(..., pool=...)``)."""

    def __init__(self, device, n_streams: int = 3) -> None:
        self.device = torch.device(device)
        self.streams = [torch.cuda.Stream(device=self.device) for _ in range(n_streams)]
        self.workspaces = [MuonWorkspace(self.device) for _ in range(n_streams)]


def _underfills_the_machine(shape, compute_units: int) -> bool:
    """Would the 256 x 256 tiles of this matrix's symmetric products (the lower triangle of an m x m result, m the
    short side) occupy less than three quarters of the CUs?"""
    t = -(-min(shape) // 256)
    return 4 * (t * (t + 1) // 2) < 3 * compute_units


def _step_on_streams(jobs, pool: MuonStreamPool) -> None:
    """Every matrix on one of the pool's streams, longest first onto the least loaded one; the calling stream waits for
    them before anything enqueued later runs."""
    n = min(len(pool.streams), len(jobs))

    def cost(job):  # flops of the products: 4 m^2 n + 2 m^3 per step
        m, k = min(job[0].shape), max(job[0].shape)
        return 4 * m * m * k + 2 * m**3

    loads, assigned = [0] * n, [[] for _ in range(n)]
    for job in sorted(jobs, key=cost, reverse=True):
        s = loads.index(min(loads))
        assigned[s].append(job)
        loads[s] += cost(job)
    current = torch.cuda.current_stream(jobs[0][0].device)
    fork = torch.cuda.Event()
    fork.record(current)
    for side, workspace, share in zip(pool.streams, pool.workspaces, assigned):
        side.wait_event(fork)
        with torch.cuda.stream(side):
            for param, grad, buf, kw in share:
                for t in (param, grad, buf):
                    t.record_stream(side)
                muon_step(param, grad, buf, workspace=workspace, **{**kw, "shared_machine": True})
        join = torch.cuda.Event()
        join.record(side)
        current.wait_event(join)


def side_by_side_default() -> bool | None:
    """``MATRIX_FSDP_MUON_SIDE_BY_SIDE``: ``0`` updates one matrix after the other (result bits that do not depend on
    which other parameters the optimizer holds), anything else lets them share launches."""
    value = os.environ.get("MATRIX_FSDP_MUON_SIDE_BY_SIDE", "auto").strip().lower()
    if value in ("0", "false", "off", "no"):
        return False
    if value in ("1", "true", "on", "yes"):
        return True
    return None


def _job(param, grad, momentum_buf, *, lr, weight_decay, momentum, nesterov, ns_coefficients=NS_COEFFICIENTS, ns_steps=NS_STEPS, eps=NS_EPS, adjust_lr_fn=None):
    """``(what the jobs of one library call share, fields of mfsdp_muon_job)``."""
    _check_step(param, grad, momentum_buf, ns_steps)
    rows, cols = param.shape
    # plain floats: equal values share a launch whatever number type they come in
    key = (_DTYPE_CODES[param.dtype], float(momentum), int(bool(nesterov)), *map(float, ns_coefficients), ns_steps, float(eps))
    return key, (param.data_ptr(), grad.data_ptr(), momentum_buf.data_ptr(), rows, cols, lr, weight_decay, adjust_lr(lr, adjust_lr_fn, (rows, cols)))


def muon_step_many(jobs, *, workspace: MuonWorkspace | None = None, pool: MuonStreamPool | None = None,
                   side_by_side: bool | None = None) -> None:
    """Updates several matrices; ``jobs`` is a sequence of ``(param, grad, momentum_buf, keywords of muon_step)``.

    The matrices of a rank are independent of each other, so those that share their hyper-parameters (the learning
    rate and weight decay may differ) go through every stage of the update as one launch, up to 32 at a time and as many
    as 1.4 GiB of workspace hold (``mfsdp_muon_step_many``; one that fills the machine goes alone): small matrices fill
    the machine together and the number of launches does not grow with theirs.

    Reproducibility: which tiles a product takes and how its K walk is cut into pieces, and with them the order of its
    fp32 sums, depend on the other matrices of the call.  In bf16 iterations that is 0.0005 to 0.006 of an update (relative
    Frobenius; torch's is 0.0007 to 0.0065 away in either form, whatever the spectrum).  A caller that needs bits independent
    of the optimizer's other parameters passes ``side_by_side=False`` (or sets ``MATRIX_FSDP_MUON_SIDE_BY_SIDE=0``), which
    updates one matrix after the other.

    With a ``pool`` the matrices take launches of their own on the pool's streams instead: those that leave CUs idle, when
    there are at least two of them (all of them with ``side_by_side=True``), the others one after the other on the calling
    stream.  A job whose keywords hold ``shared_machine`` is updated by ``muon_step``."""
    jobs = list(jobs)
    if not jobs:
        return
    device = jobs[0][0].device
    for param, *_ in jobs:
        if param.device != device:
            raise RuntimeError("muon_step_many updates the matrices of one device")
    if side_by_side is None:
        side_by_side = side_by_side_default()
    workspace = workspace or MuonWorkspace(device)
    spread = []
    if side_by_side is False:
        alone, jobs = jobs, []
    elif pool is not None:
        compute_units = torch.cuda.get_device_properties(device).multi_processor_count
        small = [job[0].ndim == 2 and (bool(side_by_side) or _underfills_the_machine(job[0].shape, compute_units)) for job in jobs]
        if sum(small) < 2 and not side_by_side:
            small = [False] * len(jobs)
        alone, spread, jobs = [j for j, s in zip(jobs, small) if not s], [j for j, s in zip(jobs, small) if s], []
    else:
        alone, jobs = [j for j in jobs if "shared_machine" in j[3]], [j for j in jobs if "shared_machine" not in j[3]]
    for param, grad, buf, kw in alone:
        muon_step(param, grad, buf, workspace=workspace, **kw)
    if spread:
        _step_on_streams(spread, pool)
    if not jobs:
        return
    alike: dict[tuple, list[tuple]] = {}
    for param, grad, buf, kw in jobs:
        key, fields = _job(param, grad, buf, **kw)
        alike.setdefault(key, []).append(fields)
    lib = _lib.lib()
    stream = stream_handle(device)
    with device_guard(device):
        for (dtype, momentum, nesterov, a, b, c, ns_steps, eps), fields in alike.items():
            n = len(fields)
            rows, cols = (ctypes.c_int64 * n)(*(f[3] for f in fields)), (ctypes.c_int64 * n)(*(f[4] for f in fields))
            need = lib.mfsdp_muon_many_workspace_bytes(n, rows, cols)
            if need <= 0:
                raise ValueError("Param gradient must be a 2D matrix")
            ws = workspace.get_bytes(need)
            _lib.check(lib.mfsdp_muon_step_many(n, (_lib.MuonJob * n)(*fields), dtype, momentum, nesterov, a, b, c, ns_steps, eps, ws.data_ptr(), ws.numel(), stream))


class AdamWBatch:
    """Spans that ``adamw_step(..., batch=...)`` has checked, updated by one launch per device (``mfsdp_adamw_step_many``)
    when ``launch`` is called.  The tensors are held until then."""

    def __init__(self) -> None:
        self._spans: dict[tuple, list[tuple]] = {}
        self._tensors: list[tuple] = []

    def add(self, device: torch.device, hyper: tuple, span: tuple, tensors: tuple) -> None:
        self._spans.setdefault((device, *hyper), []).append(span)
        self._tensors.append(tensors)

    def launch(self) -> None:
        spans_by_key, self._spans = self._spans, {}
        try:
            for (device, *hyper), spans in spans_by_key.items():
                with device_guard(device):
                    stream = stream_handle(device)
                    _lib.check(_lib.lib().mfsdp_adamw_step_many(len(spans), (_lib.AdamWSpan * len(spans))(*spans), *hyper, stream))
        finally:
            self._tensors.clear()


def adamw_step(
    param: torch.Tensor,
    grad: torch.Tensor,
    exp_avg: torch.Tensor,
    exp_avg_sq: torch.Tensor,
    step: int,
    *,
    lr: float,
    betas=(0.9, 0.999),
    eps: float = 1e-8,
    weight_decay: float = 1e-2,
    max_exp_avg_sq: torch.Tensor | None = None,
    maximize: bool = False,
    batch: AdamWBatch | None = None,
) -> None:
    """Fused AdamW over flat fp32 tensors; ``step`` is the 1-based count after
    this update (torch/optim/adam.py:347-547).  ``max_exp_avg_sq`` turns on
    amsgrad, ``maximize`` negates the gradient.  With ``batch`` the checked span
    is left to ``batch.launch()``."""
    numel = param.numel()
    state = ((param, "param"), (exp_avg, "exp_avg"), (exp_avg_sq, "exp_avg_sq"))
    if max_exp_avg_sq is not None:
        state += ((max_exp_avg_sq, "max_exp_avg_sq"),)
    for t, what in state:
        if not t.is_cuda or not t.is_contiguous() or t.dtype != torch.float32:
            raise RuntimeError(f"{what} must be a contiguous float32 CUDA tensor")
        if t.numel() != numel:
            raise RuntimeError(f"{what} has {t.numel()} elements, param has {numel}")
    if not grad.is_cuda or not grad.is_contiguous() or grad.dtype not in _DTYPE_CODES or grad.numel() != numel:
        raise RuntimeError("grad must be a contiguous float32 or bfloat16 CUDA tensor of the param's size")
    span = (
        param.data_ptr(), grad.data_ptr(), exp_avg.data_ptr(), exp_avg_sq.data_ptr(), None if max_exp_avg_sq is None else max_exp_avg_sq.data_ptr(),
        numel, int(step), _DTYPE_CODES[grad.dtype],
    )
    hyper = (float(lr), float(betas[0]), float(betas[1]), float(eps), float(weight_decay), int(bool(maximize)))
    tensors = (param, grad, exp_avg, exp_avg_sq, max_exp_avg_sq)
    if batch is not None:
        batch.add(param.device, hyper, span, tensors)
        return
    batch = AdamWBatch()
    batch.add(param.device, hyper, span, tensors)
    batch.launch()
