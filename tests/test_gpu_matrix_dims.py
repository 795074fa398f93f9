"""The matrix-core kernels at head dims 64 and 256 (chunk edges also at 128)
against the float64 oracle.

The sizes sit at the edges of the kernels' tiles: one row, 16-row decode tiles
(full, remainder), 32-row chunk waves and 128-row workgroups, 16-token blocks,
four-block stages, 64-page record windows; one or several splits and both
merges.  Tolerances: the output's own rounding (half an ulp of the largest
element, |out| < 4: 2^-9 relative in bf16, 2^-12 in f16): 7.8e-3 and 1e-3
absolute, with room for the weights' parts (all 24 bits in bf16, 2^-22 and an
absolute 2^-34 of the largest weight in f16, far below it) and at D = 128 for
a chunk's weights rounded once (as much again times the spread of V over its
mean, small against the output's): 1e-2 (bf16) and 2e-3 (f16).
"""
import math

import pytest
import torch

from helm_amd import workloads as W
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


def _mask(kind, S, T, dtype):
    """(the additive mask as given, what the oracle adds) of a later chunk."""
    if kind in ("none", "causal"):
        return None
    pos = torch.arange(T - S, T)[:, None]
    key = torch.arange(T)[None, :]
    seen = key <= pos
    if kind.startswith("window"):
        seen = seen & (key > pos - max(1, T // 3))
    dtype = torch.float32 if kind == "window_f32" else dtype
    low = torch.finfo(dtype).min
    m = torch.zeros(S, T, dtype=dtype).masked_fill_(~seen, low)
    if kind == "first_row_masked":      # one row with no visible key: equal weights
        m[0] = low
    return m[None, None]


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,S,sizes", [
    (4, 4, 1, [1]),                      # one row, one token
    (6, 2, 1, [16, 16, 5]),              # a partial decode tile, a partial block
    (32, 2, 1, [16] * 70 + [3]),         # a full 16-row tile, past one record window
    (40, 2, 1, [64, 64, 17]),            # more than one tile per KV head
    (4, 2, 17, [16, 16, 11]),            # 34 chunk rows: a full wave and two rows
    (14, 2, 19, [64, 64, 64, 30]),       # 133 rows: a workgroup and five rows
    (4, 1, 150, [16] * 68 + [7]),        # several workgroups, past one record window
    (4, 2, 40, [48] * 30 + [7]),         # 48-token pages: windows of 64 blocks start mid-page
    (8, 2, 200, [48] * 30 + [35]),       # the same, several workgroups and a ragged tail
])
@pytest.mark.parametrize("kind,cap", [("none", None), ("causal", None), ("window", None),
                                      ("window", 5.0),      # logits near the cap: tanhf
                                      ("window", 50.0),     # far below it: the polynomial
                                      ("window_f32", None), ("window_f32", 50.0),
                                      ("first_row_masked", None)])
def test_streaming_matches_fp64(D, dtype, Hq, Hkv, S, sizes, kind, cap):
    T = sum(sizes)
    if kind == "causal" and S == 1 or kind == "none" and S > 1 or T < S and kind != "causal":
        pytest.skip("no such call")
    g = torch.Generator().manual_seed(D + 7 * S + T)
    K = torch.randn(1, Hkv, T, D, generator=g).to(dtype)
    V = torch.randn(1, Hkv, T, D, generator=g).to(dtype)
    q = (1.5 * torch.randn(1, Hq, S, D, generator=g)).to(dtype)
    m = _mask(kind, S, T, dtype)
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, sizes), softcap=cap,
                                      attention_mask=None if m is None else m.to(DEV))
    ref_m = m
    if kind == "causal":
        ref_m = torch.zeros(1, 1, S, T).masked_fill_(
            torch.arange(T)[None, :] > torch.arange(S)[:, None], -math.inf)
    ref = A.attention_fp64_batched(q[0], K[0], V[0], softcap=cap,
                                   mask=None if ref_m is None else ref_m[0])
    diff = (out[0].double().cpu() - ref).abs()
    if kind == "first_row_masked" and dtype == torch.float16:
        # f16's finfo.min is -65504: the row's logits, -94,504 in base 2, have an
        # fp32 ulp of 2^-7, so each weight is off by up to 2^-8 ln 2
        assert diff[:, 0].max().item() <= TOL[dtype] + 2.0 ** -8 * math.log(2) * V.abs().max().item()
        diff = diff[:, 1:] if S > 1 else diff * 0
    err = diff.max().item()
    assert err <= TOL[dtype], err


@pytest.mark.parametrize("merge", ["fused", "kernel"])
@pytest.mark.parametrize("D,P", [(64, 16), (64, 64), (256, 16), (256, 64)])
@pytest.mark.parametrize("lens,pps", [([1, 15, 16, 17], 0), ([3001], 0), ([3001], 1),
                                      ([700, 64, 2049], 3)])
def test_pool_decode_matches_fp64(D, P, lens, pps, merge, monkeypatch):
    monkeypatch.setenv("HELM_AMD_MERGE", merge)
    for dtype in (torch.bfloat16, torch.float16):
        w = W.Workload("dims", len(lens), 10, 2, D, dtype, T=max(lens), page_size=P)
        case = W.make_pool_case(w, seed=D + P, device=DEV, lens=lens)
        out = paged_decode_attention(case["q"], case["k_pool"], case["v_pool"], case["table"],
                                     case["lens"], max_pages=case["max_pages"],
                                     pages_per_split=pps)
        for b, T in enumerate(lens):
            rows = case["pool"][case["table"][b, :case["n_pages"][b]].long()].cpu()
            kv = rows.permute(1, 2, 0, 3, 4).reshape(2, w.Hkv, -1, D)[:, :, :T]
            ref = A.attention_fp64_batched(case["q"][b].cpu(), kv[0], kv[1])
            err = (out[b].double().cpu() - ref).abs().max().item()
            assert err <= TOL[dtype], (dtype, b, err)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Hq,Hkv,S", [(32, 32, 1300), (40, 8, 1000), (8, 8, 129)])
def test_first_prompt_block_order(D, Hq, Hkv, S, monkeypatch):
    """One causal split whose blocks of query rows are handed out longest
    first, every second round of workgroups reversed: 11 blocks per head in
    rounds of 8, 40 in rounds of 32, two in one round; every row once."""
    monkeypatch.setenv("HELM_AMD_PPS", "4096")
    g = torch.Generator().manual_seed(S + D)
    K = torch.randn(1, Hkv, S, D, generator=g).to(torch.bfloat16)
    V = torch.randn(1, Hkv, S, D, generator=g).to(torch.bfloat16)
    q = (1.5 * torch.randn(1, Hq, S, D, generator=g)).to(torch.bfloat16)
    out = perform_streaming_attention(q.to(DEV), _pages(K, V, [S // 3, S - S // 3]))
    causal = torch.zeros(1, S, S).masked_fill_(
        torch.arange(S)[None, :] > torch.arange(S)[:, None], -math.inf)
    ref = A.attention_fp64_batched(q[0], K[0], V[0], mask=causal)
    assert (out[0].double().cpu() - ref).abs().max().item() <= TOL[torch.bfloat16]


@pytest.mark.parametrize("D", [64, 128, 256])
def test_pool_chunk_of_few_rows_fits_the_queried_workspace(D):
    """34 query rows per KV head over a long context: the split estimate wants
    as many splits as it may have, and the workspace query covers them."""
    w = W.Workload("rows", 1, 4, 2, D, torch.bfloat16, T=5000, page_size=16)
    case = W.make_pool_case(w, seed=D, device=DEV)
    g = torch.Generator().manual_seed(D)
    q = (1.5 * torch.randn(1, 4, 17, D, generator=g)).to(torch.bfloat16)
    out = paged_decode_attention(q.to(DEV), case["k_pool"], case["v_pool"], case["table"],
                                 case["lens"], max_pages=case["max_pages"])
    rows = case["pool"][case["table"][0].long()].cpu()
    kv = rows.permute(1, 2, 0, 3, 4).reshape(2, 2, -1, D)[:, :, :5000]
    ref = A.attention_fp64_batched(q[0], kv[0], kv[1])
    assert (out[0].double().cpu() - ref).abs().max().item() <= TOL[torch.bfloat16]


@pytest.mark.parametrize("D,S", [(64, 1), (256, 1), (64, 40), (128, 40), (256, 40)])
def test_pool_call_with_smaller_workspaces(D, S):
    """Ever smaller workspaces: fewer splits (chunks) or the element-wise
    kernel's plan (D = 64, 256), the same result, until the call is refused;
    a decode call is served down to what the element-wise plan needs."""
    from helm_amd import _native, paged
    w = W.Workload("ws", 1, 10, 2, D, torch.bfloat16, T=1500, page_size=16)
    case = W.make_pool_case(w, seed=D + S, device=DEV)
    g = torch.Generator().manual_seed(D + S)
    q = (1.5 * torch.randn(1, 10, S, D, generator=g)).to(torch.bfloat16)
    args, keep = paged._decode_args(q.to(DEV), case["k_pool"], case["v_pool"], case["table"],
                                    case["lens"], case["max_pages"], 0, None, None, None, None, 0)
    rows = case["pool"][case["table"][0].long()].cpu()
    kv = rows.permute(1, 2, 0, 3, 4).reshape(2, 2, -1, D)[:, :, :1500]
    ref = A.attention_fp64_batched(q[0], kv[0], kv[1])
    size, served = args[-2], 0
    while size > (64 << 10):
        args[-2] = size
        keep["out"].zero_()
        try:
            _native.call("helm_paged_decode_attn", *args)
        except ValueError as e:
            assert "workspace" in str(e)
            break
        assert (keep["out"][0].double().cpu() - ref).abs().max().item() <= TOL[torch.bfloat16]
        served += 1
        size = size * 3 // 4
    assert served >= 2
