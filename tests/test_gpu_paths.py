"""GPU parity of the kernels' size- and data-dependent branches, at the sizes where they change.

Same tolerance as the parity tests (errors over the reference output's RMS: max 2e-2, mean 2e-3),
against the fp32 oracle.
"""
import pytest
import torch

from oracle import pairformer_ref as ref
from tt_boltz_amd import ops
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


# ------------------------------------------------------------------------------ attention core
@pytest.mark.parametrize("shift", [-24.0, -6.0, 0.0, 12.0, 24.0])
@pytest.mark.parametrize("first_masked", [128, 127, 33, 32, 31])
def test_attention_reference_and_mask_tiles(gpu, shift, first_masked):
    """Tiles ahead of a row's first masked key run without the mask / reference fold while 0 serves
    as the softmax reference.  ``first_masked`` puts that key on both sides of a 32-key tile's
    edge; ``shift`` moves the logits of the first tile below the sum that accepts 0, of later tiles
    above the one that forces a rescale, and both ways at once over the rows.  (|logit| stays below
    32, half of the fp32 spacing at 1e9: beyond it the reference's own fully masked row is not
    the plain mean that its additive mask stands for.)"""
    g = torch.Generator().manual_seed(11)
    B, N, H, D = 1, 128, 4, 32
    q, k, v = (torch.randn((B, N, H, N, D), generator=g) for _ in range(3))
    bias = torch.randn((B, 1, H, N, N), generator=g)
    bias[..., :40] += shift
    bias[:, :, 1, :, 64:] -= shift
    mask = torch.ones((B, N, 1, 1, N))
    mask[..., first_masked:] = 0.0
    mask[:, 7, ..., 3] = 0.0     # one row with a masked key in its first tile
    mask[:, 9] = 0.0             # a fully masked row
    want = ref.triangle_attention_core(q, k, v, bias, mask, D ** -0.5)
    got = ops.triangle_attention(q.to(gpu), k.to(gpu), v.to(gpu), bias.to(gpu), mask.to(gpu))
    check(f"attention shift={shift} first_masked={first_masked}", got, want)
