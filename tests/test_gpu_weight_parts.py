"""What the weights of the matrix-core kernels at head dims 64 and 256 keep of
their 32 bits, and what infinities, NaN and -inf masks give at 64, 128 and 256."""
import math

import pytest
import torch

from helm_amd.paged import paged_decode_attention
from helm_amd.runtime.kv_cache import KVPage, perform_streaming_attention
from oracle import attention as A

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TOL = {torch.float16: 2e-3, torch.bfloat16: 1e-2}


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


def _one_dominant_key(D, S, gap, T, V, pps, monkeypatch):
    """(f16 attention, the float64 result) of S query rows over T + 1 keys in
    pages of 64: the first key's logit is `gap`, every other's 0.  V [2, T + 1, D]."""
    monkeypatch.setenv("HELM_AMD_PPS", str(pps))
    K = torch.zeros(1, 2, T + 1, D, dtype=torch.float16)
    K[:, :, 0, 0] = gap
    q = torch.zeros(1, 4, S, D, dtype=torch.float16)
    q[..., 0] = math.sqrt(D)
    sizes = [64] * (T // 64) + [T % 64 + 1]
    out = perform_streaming_attention(q.to(DEV), _pages(K, V[None], sizes),
                                      attention_mask=_zero_mask(S, T + 1))[0].double().cpu()
    w = torch.full((T + 1,), math.exp(-gap), dtype=torch.float64)
    w[0] = 1
    ref = (w / w.sum()) @ V.double()                              # [2, D]
    return out, ref.repeat_interleave(2, 0)[:, None].expand(4, S, D)


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("S,T", [(1, 8000), (40, 65536)])       # decode, chunk: one split
@pytest.mark.parametrize("gap", [16.5, 17.0, 18.0])
@pytest.mark.parametrize("values", ["ones", "one_two", "sink_zero", "random"])
def test_f16_keys_far_below_one_dominant_key(D, S, T, gap, values, monkeypatch):
    """Many keys that together weigh 1e-4 to 4e-3 of the row, each below 2^-23 of
    the largest weight (the ones' sum: also below an ulp of the row's).  The output is off by its own rounding (2^-11 relative,
    half an ulp, and 2^-25 where it is subnormal), the weights' floor (2^-34 each)
    and 1e-6 of fp32 rounding."""
    g = torch.Generator().manual_seed(D + S)
    V = torch.ones(2, T + 1, D, dtype=torch.float16)
    if values == "one_two":
        V[:, 1:] = 2
    elif values == "sink_zero":
        V[:, 0] = 0
    elif values == "random":
        V = torch.randn(2, T + 1, D, generator=g).half()
    out, ref = _one_dominant_key(D, S, gap, T, V, 128 if S == 1 else 1025, monkeypatch)
    bound = ref.abs() * 2.0 ** -11 + 2.0 ** -25 + T * 2.0 ** -34 * V.abs().max() + 1e-6 * ref.abs()
    assert ((out - ref).abs() <= bound).all(), ((out - ref).abs() / bound).max().item()


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,sizes", [(1, [16, 16, 7]), (1, [64] * 40), (40, [16, 16, 7]),
                                     (40, [64] * 40), (150, [48] * 30 + [9])])
def test_infinite_values(D, dtype, S, sizes):
    """Infinities in V come out as the fp32 weights give them: +inf, -inf, NaN
    where both signs meet, also under a weight of e^-40; the other columns keep
    their values (tolerance: the output's rounding, as without infinities)."""
    T = sum(sizes)
    g = torch.Generator().manual_seed(D + S + T)
    K, V = (torch.randn(1, 2, T, D, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(1, 6, S, D, generator=g).to(dtype)
    q[..., 0] = 4
    K[:, :, 13] = 0
    K[:, :, 13, 0] = -10 * math.sqrt(D)
    V[:, :, 5, 0] = V[:, :, 9, 2] = V[:, :, 13, 3] = math.inf
    V[:, :, 7, 1] = V[:, :, 11, 2] = -math.inf
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, sizes),
                                      attention_mask=_zero_mask(S, T))[0].double().cpu()
    assert (out[..., 0] == math.inf).all() and (out[..., 1] == -math.inf).all()
    assert out[..., 2].isnan().all() and (out[..., 3] == math.inf).all()
    V[..., :4] = 0
    ref = A.attention_fp64_batched(q[0], K[0], V[0])
    assert (out[..., 4:] - ref[..., 4:]).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("route,cap", [
    ("causal", None),                 # (a soft-capped prompt is not causal)
    ("pool_decode", None), ("pool_decode", 20.0), ("pool_chunk", None), ("pool_chunk", 20.0)])
def test_infinite_values_without_a_mask(D, dtype, route, cap):
    """The same under the causal limit (the rows that see every infinity) and
    over a slot pool, soft-capped or not, in one split and in several."""
    T = 150 if route == "causal" else 700
    S = {"causal": T, "pool_decode": 1, "pool_chunk": 40}[route]
    g = torch.Generator().manual_seed(D + T)
    K, V = (torch.randn(1, 2, T, D, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(1, 6, S, D, generator=g).to(dtype)
    V[:, :, 5, 0] = math.inf
    V[:, :, 7, 1] = -math.inf
    V[:, :, 3, 2], V[:, :, 8, 2] = math.inf, -math.inf
    if route == "causal":
        outs = [perform_streaming_attention(q.to(DEV), _pages(K, V, [64, 64, 22]), softcap=cap)]
    else:
        pad = torch.zeros(1, 2, 704 - T, D, dtype=dtype)
        pool = [torch.cat([x, pad], 2).reshape(2, 44, 16, D).transpose(0, 1).contiguous().to(DEV)
                for x in (K, V)]
        table = torch.arange(44, dtype=torch.int32, device=DEV)[None]
        lens = torch.tensor([T], dtype=torch.int32, device=DEV)
        outs = [paged_decode_attention(q.to(DEV), *pool, table, lens, softcap=cap,
                                       pages_per_split=pps) for pps in (0, 44, 9)]
    V[..., :3] = 0
    mask = None
    if route == "causal":
        mask = torch.zeros(1, S, T).masked_fill_(
            torch.arange(T)[None, :] > torch.arange(S)[:, None], -math.inf)
    ref = A.attention_fp64_batched(q[0], K[0], V[0], mask=mask, softcap=cap)
    seen = slice(8, None) if route == "causal" else slice(None)
    for out in outs:
        out = out[0].double().cpu()[:, seen]
        assert (out[..., 0] == math.inf).all() and (out[..., 1] == -math.inf).all()
        assert out[..., 2].isnan().all()
        assert (out[..., 3:] - ref[:, seen, 3:]).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S", [1, 40])
def test_infinite_values_at_head_dim_128_stay_in_their_column(dtype, S):
    """D = 128, whose weights were parts from the start: the column of an
    infinity is infinite or NaN, the others keep their values."""
    D, T = 128, 200
    q, K, V = _chunk(D, dtype, T, S, S)
    V[:, :, 5, 0] = math.inf
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, [64, 64, 64, 8]),
                                      attention_mask=_zero_mask(S, T))[0].double().cpu()
    assert not out[..., 0].isfinite().any()
    V[..., 0] = 0
    ref = A.attention_fp64_batched(q[0], K[0], V[0])
    assert (out[..., 1:] - ref[..., 1:]).abs().max().item() <= TOL[dtype]


def _chunk(D, dtype, T, S, seed):
    g = torch.Generator().manual_seed(seed)
    K, V = (torch.randn(1, 2, T, D, generator=g).to(dtype) for _ in range(2))
    return (1.5 * torch.randn(1, 4, S, D, generator=g)).to(dtype), K, V


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S", [1, 40])
@pytest.mark.parametrize("mdtype", ["own", "f32"])
@pytest.mark.parametrize("cap", [None, 50.0])
def test_rows_masked_everywhere(D, dtype, S, mdtype, cap):
    """Rows with no visible key: -inf masks leave a row without keys, zeros (a
    chunk at D = 128 bounds its logits: the mean of V); finfo.min masks weigh
    every key alike; -inf beside finfo.min hides."""
    T = 200
    q, K, V = _chunk(D, dtype, T, S, D + S)
    mt = dtype if mdtype == "own" else torch.float32
    low = torch.finfo(mt).min
    mask = torch.zeros(1, 4, S, T, dtype=mt)
    mask[:, 0] = -math.inf
    mask[:, 1] = low
    mask[:, 2] = low
    mask[:, 2, :, ::2] = -math.inf
    mask[:, 3, :, :T // 2] = -math.inf
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, [64, 64, 64, 8]), softcap=cap,
                                      attention_mask=mask.to(DEV))[0].double().cpu()
    mean = V[0].double().mean(1)
    keeps = D == 128 and S > 1
    assert (out[0] - (mean[0] if keeps else 0)).abs().max().item() <= (TOL[dtype] if keeps else 0)
    exact = A.attention_fp64_batched(q[0], K[0], V[0], mask=mask[0].float(), softcap=cap)
    # (an f16 finfo.min is no bound: the scores still count)
    if mt == torch.float16:
        assert (out[1] - exact[1]).abs().max().item() <= TOL[dtype]
    else:
        assert (out[1] - mean[0]).abs().max().item() <= TOL[dtype]
        want = mean[1] if keeps else V[0, 1, 1::2].double().mean(0)
        assert (out[2] - want).abs().max().item() <= TOL[dtype]
    assert (out[3] - exact[3]).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cap", [None, 50.0])
@pytest.mark.parametrize("other", [0.0, -1.0])
def test_nan_keys_under_a_mask_do_not_depend_on_neighbours(D, dtype, cap, other):
    """A chunk with a NaN key whose mask is zero, its neighbours' masks zero or
    not: at D = 64 and 256 every row is NaN; at D = 128 the key is left out.  A
    NaN key under finfo.min is left out at every head dim, also in a step with
    visible keys."""
    T, S = 200, 40
    q, K, V = _chunk(D, dtype, T, S, D + 1)
    mask = torch.zeros(1, 1, S, T)
    mask[..., 40:60] = other
    hidden = mask.clone()
    hidden[..., 50] = torch.finfo(torch.float32).min
    ref = A.attention_fp64_batched(q[0], K[0], V[0], mask=hidden[0], softcap=cap)
    K[:, :, 50] = math.nan
    mask[..., 50] = 0
    for m, left_out in ((hidden, True), (mask, D == 128)):
        out = perform_streaming_attention(q.to(DEV), _pages(K, V, [64, 64, 64, 8]), softcap=cap,
                                          attention_mask=m.to(DEV))[0].double().cpu()
        if left_out:
            assert (out - ref).abs().max().item() <= TOL[dtype]
        else:
            assert out.isnan().all()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("other", [0.0, -1.0])
def test_infinite_logits_under_a_mask_do_not_depend_on_neighbours(D, other):
    """Every logit -inf, the masks zero or not: a chunk's rows are zeros at D = 64
    and 256 and the mean of V at D = 128, where masked logits are bounded."""
    T, S = 200, 40
    q, K, V = _chunk(D, torch.bfloat16, T, S, D + 2)
    q[..., 0] = 1
    K[..., 0] = -math.inf
    mask = torch.zeros(1, 1, S, T)
    mask[..., 20:180] = other
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, [64, 64, 64, 8]),
                                      attention_mask=mask.to(DEV))[0].double().cpu()
    want = V[0].double().mean(1).repeat_interleave(2, 0)[:, None] * (D == 128)
    assert (out - want).abs().max().item() <= (TOL[torch.bfloat16] if D == 128 else 0)
