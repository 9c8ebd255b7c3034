"""The branches that the sizes of a call choose between, at the sizes where they begin and end: each against dense
logits or gradients formed on the GPU in fp32 / fp64."""

import pytest
import torch

from _util import make_inputs

pytestmark = pytest.mark.gpu


def _lib():
    from cut_cross_entropy import _hip

    return _hip.load()


@pytest.mark.parametrize("shape", [(1, 256 * 255, 128), (40, 256 * 256 + 1, 128), (256, 256 * 257 - 5, 192), (257, 256 * 129, 128),
                                   (700, 256 * 90 + 7, 128), (1025, 256 * 66, 128)])
def test_lse_forward_of_few_rows_fills_the_chip(shape):
    """One to five row blocks against many classes: more than 64 vocabulary spans per row block (up to one span for
    each tile), all merged by the second kernel."""
    lib = _lib()
    dev = torch.device("cuda:0")
    N, V, D = shape
    e, c, _, _ = make_inputs(N, V, D, torch.bfloat16, seed=5)
    ed, cd = e.to(dev), c.to(dev)
    want = torch.logsumexp((ed.float() @ cd.float().T).double(), dim=1)
    lse = torch.full((N,), float("nan"), dtype=torch.float32, device=dev)
    ws = torch.full((lib.cce_lse_forward_workspace_bytes(N, V, D) // 4,), float("nan"), device=dev)
    st = lib.cce_lse_forward(
        ed.data_ptr(), cd.data_ptr(), None, None, lse.data_ptr(), None, None, ws.data_ptr(), ws.numel() * 4,
        N, N, V, D, ed.stride(0), cd.stride(0), cd.stride(1), 0.0, 0, torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.cce_error_string(st)
    # fp32 sums of D <= 192 products of magnitude about 1, and of up to 66000 exponentials: the bound of
    # test_lse_forward_spans_of_many_tiles
    assert torch.allclose(lse.double(), want, atol=2e-4, rtol=2e-5)
