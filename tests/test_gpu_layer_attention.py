"""``layer_attention`` on MFMAs: every head width of whole 16-value blocks, sequences from one state to
the 16 a fragment holds, and workgroups whose last waves have no item, against FP64; widths with a
remainder take the general kernel."""

import pytest
import torch

from iris_mi355x import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d", [16, 32, 48, 64, 80, 96, 112, 128, 24, 81])
@pytest.mark.parametrize("L", [1, 3, 4, 12, 15, 16])
@pytest.mark.parametrize("seqs,heads", [(1, 1), (7, 3), (5, 8)])
def test_layer_attention_widths(d, L, seqs, heads):
    g = torch.Generator(device=DEV).manual_seed(60)
    qkv = (2.0 * torch.randn(seqs * L, 3 * heads * d, generator=g, device=DEV)).to(torch.bfloat16)
    q, k, v = (t.transpose(1, 2) for t in qkv.double().view(seqs, L, 3, heads, d).unbind(2))
    p = torch.softmax(q @ k.transpose(-1, -2) / d ** 0.5, -1)
    want = (p @ v).transpose(1, 2).reshape(seqs * L, heads * d)
    out = torch.full((seqs * L, heads * d), 9.0, device=DEV, dtype=torch.bfloat16)
    K.layer_attention(qkv, out, L, heads)
    # FP32 scores (error 2^-24 sqrt(d) |q||k| / sqrt(d), about 1e-5 here) and one BF16 rounding of the result
    torch.testing.assert_close(out.double(), want, rtol=2.0 ** -8, atol=1e-4)
