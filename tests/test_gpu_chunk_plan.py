"""How query chunks over the pool are split, read back from the split counts
that a call leaves in its workspace (int32 per 16-row tile, past the 64 KiB
ticket region), and the workspace they need."""
import pytest
import torch

from helm_amd import _native, paged
from helm_amd import workloads as W
from oracle import attention as A

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TICKETS = 64 << 10


def _chunk(D, Hq, Hkv, S, T, seed, lens=None, total_pages=0, dtype=torch.bfloat16):
    """(C arguments, kept tensors, pool case) of S query rows per sequence over
    the last of T tokens in 16-token pages."""
    lens = lens or [T]
    w = W.Workload("plan", len(lens), Hq, Hkv, D, dtype, T=max(lens), page_size=16)
    case = W.make_pool_case(w, seed=seed, device=DEV, lens=lens)
    g = torch.Generator().manual_seed(seed)
    q = (1.5 * torch.randn(len(lens), Hq, S, D, generator=g)).to(dtype)
    args, keep = paged._decode_args(q.to(DEV), case["k_pool"], case["v_pool"], case["table"],
                                    case["lens"], case["max_pages"], total_pages, None, None, None,
                                    None, 0)
    keep["q_cpu"] = q
    return args, keep, case


def _run(args, ws_bytes):
    """The call with a fresh workspace of ws_bytes; returns the workspace."""
    ws = torch.zeros(ws_bytes, dtype=torch.uint8, device=DEV)
    args[-3], args[-2] = ws.data_ptr(), ws_bytes
    _native.call("helm_paged_decode_attn", *args)
    torch.cuda.synchronize()
    return ws


def _check(keep, case, b, T, D, Hkv, tol=1e-2):
    rows = case["pool"][case["table"][b, :-(-T // 16)].long()].cpu()
    kv = rows.permute(1, 2, 0, 3, 4).reshape(2, Hkv, -1, D)[:, :, :T]
    ref = A.attention_fp64_batched(keep["q_cpu"][b], kv[0], kv[1])
    assert (keep["out"][b].double().cpu() - ref).abs().max().item() <= tol


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("Hq,Hkv,S,T", [(10, 2, 40, 500), (4, 1, 17, 300)])
def test_one_split_needs_no_room_for_partials(D, Hq, Hkv, S, T):
    """A chunk call with a workspace of the ticket region and the split counts
    only: one split, which writes the output itself."""
    args, keep, case = _chunk(D, Hq, Hkv, S, T, seed=D + S)
    tiles = Hkv * -(-(Hq // Hkv * S) // 16)
    need = TICKETS + -(-tiles * 4 // 256) * 256
    ws = _run(args, need)
    assert (ws[TICKETS:].view(torch.int32)[:tiles] == 1).all()
    _check(keep, case, 0, T, D, Hkv)
    with pytest.raises(ValueError, match="workspace"):
        _run(args, need - 256)


@pytest.mark.parametrize("D,Hq,Hkv,S,least", [(128, 16, 2, 4, 100), (64, 14, 2, 3, 200)])
def test_few_heads_over_a_long_context_fill_the_chip(D, Hq, Hkv, S, least):
    """Two KV heads over 131,072 tokens: enough splits for every CU (64 leave
    half of them or more idle)."""
    T = 131072
    args, keep, case = _chunk(D, Hq, Hkv, S, T, seed=D)
    ws = _run(args, args[-2])
    assert least <= ws[TICKETS:].view(torch.int32)[0].item() <= 512
    _check(keep, case, 0, T, D, Hkv)
