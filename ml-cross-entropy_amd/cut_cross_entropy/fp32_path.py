"""fp32 inputs on matrix cores that multiply 16-bit numbers.

gfx950 has no fast fp32 matrix path (the reference leans on Triton's tf32x3 / ieee dot for fp32 inputs,
cce_lse_forward.py:81, constants via tl_utils).  For the products of the gradients the library splits every fp32 value
into three bfloat16 parts, x = hi + mid + lo (8 + 8 + 8 significant bits), and takes a product as its six leading cross terms

    hi*hi + hi*mid + mid*hi + mid*mid + hi*lo + lo*hi          (what is left is below 2^-24 relative)

in one reduction of its 16-bit kernels with fp32 accumulators.  The logits, in either pass, go by two halves of fp16 (22 - 23
bits) and hi*hi + hi*lo + lo*hi, unless a value of E is past 255.5 or one of C past 15.9: then by the same parts and terms as the
gradients, which the device decides.  ``cce_fp32_forward`` and ``cce_fp32_backward`` run the whole of either pass in one call.  The
gradient filter threshold of fp32 is far below anything a soft-max produces, so the backward is the unfiltered one.

``torch.set_float32_matmul_precision``: "highest" (the default) takes the terms above; with "high" or "medium" the caller has asked
for fast fp32 products (the reference then lets Triton use tf32, 10 mantissa bits, cce_lse_forward.py:129-131), and products of
bf16 parts are formed from two of them and three terms, hi*hi + hi*mid + mid*hi (16 bits), half the work.  dBias is no product: it is a
sum of fp32 values either way.
"""

from typing import Optional, Tuple

import torch

from cut_cross_entropy import _hip


def n_terms() -> int:
    """Cross terms per product of bf16 parts: all six under "highest" float32 matmul precision, the leading three otherwise."""
    return 6 if torch.get_float32_matmul_precision() == "highest" else 3


def _workspace(nbytes: int, dev: torch.device) -> Tuple[torch.Tensor, int]:
    """A 256-byte aligned scratch buffer (torch memory, so that the allocator's peak statistic sees it)."""
    buf = torch.empty((nbytes + 256,), dtype=torch.uint8, device=dev)
    return buf, (buf.data_ptr() + 255) // 256 * 256


def _check(e, c, bias, targets, valids) -> None:
    _hip.require_one_gpu(e, c, bias, targets, valids)
    assert targets.numel() == e.size(0)
    assert bias is None or (bias.ndim == 1 and bias.size(0) == c.size(0))


def _as_fp32(bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    return None if bias is None else bias.to(torch.float32).contiguous()


def fp32_forward(e, c, bias, targets, valids, shift, softcap, target_offset) -> Tuple[torch.Tensor, torch.Tensor]:
    """``(lse, nll)`` of the valid rows: the log-sum-exp over the whole vocabulary, and what is left of it when the
    (soft-capped) logit of the target is taken off (all of it where the target is not a class of this shard)."""
    _check(e, c, bias, targets, valids)
    lib = _hip.load()
    dev = e.device
    b = valids.numel() if valids is not None else e.size(0)
    lse = torch.empty((b,), dtype=torch.float32, device=dev)
    nll = torch.empty((b,), dtype=torch.float32, device=dev)
    if b == 0:
        return lse, nll
    terms = n_terms()
    bias, targets = _as_fp32(bias), targets.to(torch.int64).contiguous()
    ws_bytes = lib.cce_fp32_forward_workspace_bytes(b, c.size(0), c.size(1), terms)
    _buf, ws = _workspace(ws_bytes, dev)
    with _hip.on_device(dev):
        status = lib.cce_fp32_forward(
            e.data_ptr(), c.data_ptr(), _hip.ptr(bias), _hip.ptr(valids), targets.data_ptr(),
            lse.data_ptr(), nll.data_ptr(), ws, ws_bytes,
            e.size(0), b, c.size(0), c.size(1), e.stride(0), c.stride(0), c.stride(1),
            int(shift), int(target_offset), float(softcap) if softcap is not None else 0.0, terms,
            _hip.current_stream_ptr(dev))
    _hip.check(status, "cce_fp32_forward")
    return lse, nll


def fp32_backward(e, c, bias, lse, do, dlse, valids, targets, shift, target_offset, softcap, grad_scale,
                  want_de, want_dc, want_dbias):
    """(dE, dC, dBias) in fp32."""
    _check(e, c, bias, targets, valids)
    _hip.require_one_gpu(e, lse, do, dlse)
    lib = _hip.load()
    dev = e.device
    v, d = c.shape
    b = lse.numel()
    # packed, whatever the strides of e and c (those of a single row say nothing about where the next one would be)
    de = torch.zeros(e.shape, dtype=e.dtype, device=dev) if want_de else None  # added to; rows that do not count stay zeros
    dc = None
    if want_dc:  # written whole, unless there is no valid row
        dc = (torch.empty if b else torch.zeros)((v, d), dtype=c.dtype, device=dev)
    dbias = torch.zeros((v,), dtype=torch.float32, device=dev) if want_dbias else None
    if b == 0 or not (want_de or want_dc or want_dbias):
        return de, dc, dbias
    terms = n_terms()
    bias, targets = _as_fp32(bias), targets.to(torch.int64).contiguous()
    do = do.to(torch.float32).contiguous().view(-1)
    dlse = dlse.to(torch.float32).contiguous().view(-1) if dlse is not None else None
    ws_bytes = lib.cce_fp32_backward_workspace_bytes(b, v, d, terms)
    _buf, ws = _workspace(ws_bytes, dev)
    with _hip.on_device(dev):
        status = lib.cce_fp32_backward(
            e.data_ptr(), c.data_ptr(), _hip.ptr(bias), lse.data_ptr(), do.data_ptr(), 1 if do.numel() == 1 else 0,
            _hip.ptr(dlse), _hip.ptr(valids), targets.data_ptr(), _hip.ptr(de), _hip.ptr(dc), _hip.ptr(dbias), ws, ws_bytes,
            e.size(0), b, v, d, e.stride(0), c.stride(0), c.stride(1), de.stride(0) if de is not None else d,
            dc.stride(0) if dc is not None else d, float(grad_scale), int(shift), int(target_offset),
            float(softcap) if softcap is not None else 0.0, terms, _hip.current_stream_ptr(dev))
    _hip.check(status, "cce_fp32_backward")
    return de, dc, dbias
