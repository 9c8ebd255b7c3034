"""Launcher of the fused matmul + log-sum-exp kernel
(reference: cut_cross_entropy/cce_lse_forward.py:170-237)."""

import threading
from typing import Optional, Tuple, Union

import torch

from cut_cross_entropy import _hip

REDUCTION_CODES = {"none": 0, "sum": 1, "mean": 2}
_pinned = threading.local()  # the word of pinned host memory that a thread receives its counts in


def lse_forward(
    e: torch.Tensor,
    c: torch.Tensor,
    bias: Optional[torch.Tensor],
    valids: Optional[torch.Tensor],
    softcap: Optional[float],
    want_logit_avg: bool = False,
    want_tile_max: bool = False,
) -> Tuple[torch.Tensor, Optional[torch.Tensor], Optional[torch.Tensor]]:
    """Returns ``(lse[B] fp32, logit_avg[V] fp32 | None, tile_max | None)``.

    ``tile_max`` holds the largest soft-capped logit of every 32-row x 32-class cell;
    the backward uses it to drop tiles without recomputing them.
    """
    assert e.ndim == 2 and c.ndim == 2
    assert e.shape[1] == c.shape[1], "Incompatible dimensions"
    assert e.is_contiguous(), "Matrix A must be contiguous"
    _hip.require_gpu_tensor("e", e)
    assert c.device == e.device and c.dtype == e.dtype
    if valids is not None:
        assert valids.ndim == 1 and valids.dtype == torch.int32
        valids = valids.contiguous()
        B = valids.numel()
    else:
        B = e.shape[0]
    if bias is not None:
        assert bias.ndim == 1
        assert c.shape[0] == bias.shape[0]
        bias = bias.to(e.dtype).contiguous()
    V, D = c.shape
    code = _hip.dtype_code(e.dtype)
    lib = _hip.load()

    lse = torch.empty((B,), dtype=torch.float32, device=e.device)
    logit_avg = torch.empty((V,), dtype=torch.float32, device=e.device) if want_logit_avg else None
    tile_max = None
    if want_tile_max:
        tile_max = torch.empty((lib.cce_tile_stat_elems(B, V),), dtype=torch.float32, device=e.device)
    if B == 0:
        if logit_avg is not None:
            logit_avg.zero_()
        return lse, logit_avg, tile_max

    ws_bytes = lib.cce_lse_forward_workspace_bytes(B, V, D)
    workspace = torch.empty((max(ws_bytes, 8) // 8,), dtype=torch.int64, device=e.device)
    with _hip.on_device(e.device), _hip.timed("lse_forward", e.device):
        status = lib.cce_lse_forward(
            e.data_ptr(), c.data_ptr(), _hip.ptr(bias), _hip.ptr(valids),
            lse.data_ptr(), _hip.ptr(logit_avg), _hip.ptr(tile_max),
            workspace.data_ptr(), workspace.numel() * 8,
            e.shape[0], B, V, D,
            e.stride(0), c.stride(0), c.stride(1),
            float(softcap) if softcap is not None else 0.0, code,
            _hip.current_stream_ptr(e.device),
        )
    _hip.check(status, "cce_lse_forward")
    return lse, logit_avg, tile_max


def loss_forward(
    e: torch.Tensor,
    c: torch.Tensor,
    bias: Optional[torch.Tensor],
    targets: torch.Tensor,
    valids: Optional[torch.Tensor],
    shift: int,
    softcap: Optional[float],
    target_offset: int,
    want_tile_max: bool,
) -> Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]:
    """``(lse, nll, tile_max | None)`` of the valid rows in one library call: ``lse_forward`` plus the logit of each
    row's target (``indexed_neg_dot_forward_kernel``), merged and added up by one kernel."""
    assert e.ndim == 2 and c.ndim == 2 and e.is_contiguous()
    assert e.shape[1] == c.shape[1], "Incompatible dimensions"
    dev = e.device
    _hip.require_one_gpu(e, c, bias, targets, valids)
    assert c.dtype == e.dtype
    assert targets.numel() == e.shape[0]
    V, D = c.shape
    code = _hip.dtype_code(e.dtype)
    lib = _hip.load()
    B = valids.numel() if valids is not None else e.shape[0]
    if bias is not None:
        assert bias.ndim == 1 and bias.shape[0] == V
        bias = bias.to(e.dtype).contiguous()
    targets = targets.to(torch.int64).contiguous()
    lse = torch.empty((B,), dtype=torch.float32, device=dev)
    nll = torch.empty((B,), dtype=torch.float32, device=dev)
    tile_max = None
    if want_tile_max:
        tile_max = torch.empty((lib.cce_tile_stat_elems(B, V),), dtype=torch.float32, device=dev)
    if B == 0:
        return lse, nll, tile_max
    ws_bytes = lib.cce_lse_forward_workspace_bytes(B, V, D)
    workspace = torch.empty((max(ws_bytes, 8) // 8,), dtype=torch.int64, device=dev)
    with _hip.on_device(dev), _hip.timed("lse_forward", dev):
        status = lib.cce_loss_forward(
            e.data_ptr(), c.data_ptr(), _hip.ptr(bias), _hip.ptr(valids), targets.data_ptr(),
            lse.data_ptr(), nll.data_ptr(), _hip.ptr(tile_max), workspace.data_ptr(), workspace.numel() * 8,
            e.shape[0], B, V, D, e.stride(0), c.stride(0), c.stride(1),
            int(shift), int(target_offset), float(softcap) if softcap is not None else 0.0, code,
            _hip.current_stream_ptr(dev),
        )
    _hip.check(status, "cce_loss_forward")
    return lse, nll, tile_max


def loss_call(
    e: torch.Tensor,
    c: torch.Tensor,
    bias: Optional[torch.Tensor],
    targets: torch.Tensor,
    shift: int,
    ignore_index: int,
    softcap: Optional[float],
    target_offset: int,
    reduction: str,
    return_lse: bool,
    want_tile_max: bool,
    terms: int,
):
    """The whole forward in one library call: ``(rows, count, outputs)``.  ``rows[:count]`` are the valid rows of the flattened
    ``e`` for labels ``targets`` [batch.., steps]; ``outputs`` is ``(loss, lse_out | None, lse[count], tile_max | None)``, or
    None where so few rows count that their plan wants more scratch than was set aside (the single calls take any).
    ``terms``: cross terms per product of fp32 inputs, 0 for 16-bit ones."""
    dev = e.device
    _hip.require_one_gpu(e, c, bias, targets)
    assert c.dtype == e.dtype and e.ndim == 2 and c.ndim == 2 and e.shape[1] == c.shape[1]
    n, (v, d), steps = e.shape[0], c.shape, targets.size(-1)
    assert targets.numel() == n
    code = 2 if terms else _hip.dtype_code(e.dtype)
    lib = _hip.load()
    if bias is not None:
        assert bias.ndim == 1 and bias.shape[0] == v
        bias = bias.to(e.dtype).contiguous()
    batch = targets.shape
    kept = batch[:-1] + (steps - shift,) if shift else batch
    targets = targets.to(torch.int64).contiguous()
    rows = torch.empty((n,), dtype=torch.int32, device=dev)
    lse = torch.empty((n,), dtype=torch.float32, device=dev)
    tile_max = torch.empty((lib.cce_tile_stat_elems(n, v),), dtype=torch.float32, device=dev) if want_tile_max else None
    loss = torch.empty(kept if reduction == "none" else (), dtype=torch.float32, device=dev)
    lse_out = torch.empty(kept, dtype=torch.float32, device=dev) if return_lse else None
    ws_bytes = lib.cce_loss_call_workspace_bytes(n, v, d, code, terms)
    ws = torch.empty((ws_bytes + 256,), dtype=torch.uint8, device=dev)
    count = getattr(_pinned, "count", None)
    if count is None:
        count = _pinned.count = torch.zeros((1,), dtype=torch.int64, pin_memory=True)
    with _hip.on_device(dev), _hip.timed("forward_fp32" if terms else "lse_forward", dev):
        status = lib.cce_loss_call(
            e.data_ptr(), c.data_ptr(), _hip.ptr(bias), targets.data_ptr(), rows.data_ptr(), count.data_ptr(), lse.data_ptr(),
            _hip.ptr(tile_max), loss.data_ptr(), _hip.ptr(lse_out), (ws.data_ptr() + 255) // 256 * 256, ws_bytes,
            n, steps, v, d, e.stride(0), c.stride(0), c.stride(1), shift, ignore_index, target_offset,
            float(softcap) if softcap is not None else 0.0, REDUCTION_CODES[reduction], code, terms,
            _hip.current_stream_ptr(dev))
    b = count.item()
    if status == _hip.ERR_WORKSPACE_TOO_SMALL and b >= 0:
        return rows, b, None
    _hip.check(status, "cce_loss_call")
    if return_lse and b == n and not shift:
        lse_out = lse.view(batch)
    if b < n:
        lse = lse[:b]
        if tile_max is not None:
            tile_max = tile_max[: lib.cce_tile_stat_elems(b, v)]
    return rows, b, (loss, lse_out, lse, tile_max)


def cce_lse_forward_kernel(
    e: torch.Tensor,
    c: torch.Tensor,
    bias: Optional[torch.Tensor] = None,
    valids: Optional[torch.Tensor] = None,
    softcap: Optional[float] = None,
    return_logit_avg: bool = False,
) -> Union[Tuple[torch.Tensor, torch.Tensor], torch.Tensor]:
    """Same call as the reference launcher: ``lse`` or ``(lse, logit_avg)``."""
    lse, logit_avg, _ = lse_forward(e, c, bias, valids, softcap, want_logit_avg=return_logit_avg)
    if return_logit_avg:
        assert logit_avg is not None
        return lse, logit_avg
    return lse
