"""What the weights of the matrix-core kernels at head dims 64 and 256 keep of
their 32 bits, and what infinities, NaN and -inf masks give there."""
import math

import pytest
import torch

from helm_amd.runtime.kv_cache import KVPage, perform_streaming_attention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _pages(K, V, sizes):
    pages, t = [], 0
    for i, n in enumerate(sizes):
        k, v = (x[:, :, t:t + n].contiguous().to(DEV) for x in (K, V))
        pages.append(KVPage(page_id=i, layer_id=0, start_token=t, used_tokens=n,
                            capacity_tokens=n, k_tensor=k, v_tensor=v, device=k.device,
                            state="GPU"))
        t += n
    return pages


def _zero_mask(S, T):
    return torch.zeros(1, 1, S, T, device=DEV) if S > 1 else None


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("S", [1, 40])
def test_bf16_weights_keep_all_their_bits(D, S):
    """Two tokens of weight 1 whose values are minus the leading 16 bits of the
    third token's weight (two bf16 parts), the third's value 1: the output is
    what the two parts leave of the weight, up to 2^-18.  The kernel's weight is
    off by the fp32 logit's and exponential's rounding, at most 8 x 2^-24."""
    H = 64
    g = torch.Generator().manual_seed(D + S)
    kb = (-8 * torch.rand(H, generator=g) - 1).bfloat16()
    w = torch.exp(kb.double() / math.sqrt(D))
    hi = w.bfloat16()
    mid = (w - hi.double()).bfloat16()
    K = torch.zeros(1, H, 3, D, dtype=torch.bfloat16)
    K[0, :, 2, 0] = kb
    V = torch.zeros(1, H, 3, D, dtype=torch.bfloat16)
    V[0, :, 0], V[0, :, 1], V[0, :, 2] = -hi[:, None], -mid[:, None], 1
    q = torch.zeros(1, H, S, D, dtype=torch.bfloat16)
    q[..., 0] = 1
    ref = ((w - hi.double() - mid.double()) / (2 + w))[:, None, None].expand(H, S, D)
    assert ref.abs().max().item() > 1e-6
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, [3]),
                                      attention_mask=_zero_mask(S, 3))
    assert (out[0].double().cpu() - ref).abs().max().item() <= 8 * 2.0 ** -24
