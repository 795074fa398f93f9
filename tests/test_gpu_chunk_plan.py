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


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("hint", [True, False])
def test_ragged_chunks_take_no_split_below_the_shortest(D, hint):
    """One sequence of 64 pages among 64 of one page, with and without the total
    page count: splits of at least eight 16-token pages, as the workspace query
    counts on, and the call fits what it asks for."""
    lens = [1024] + [16] * 63
    args, keep, case = _chunk(D, 4, 2, 17, 1024, seed=D, lens=lens,
                              total_pages=127 if hint else 0)
    tiles = 2 * 3
    ws = _run(args, args[-2])
    counts = ws[TICKETS:].view(torch.int32)[:64 * tiles].view(64, tiles).cpu()
    assert (counts[0] <= 8).all() and (counts[1:] == 1).all()
    for b in (0, 1, 63):
        _check(keep, case, b, lens[b], D, 2)


def test_split_length_follows_the_sequence_not_the_table():
    """One sequence of 100 pages in a table of 4,096 columns, its page count
    given: the split count of the same call with a table of 100."""
    counts = []
    for width in (100, 4096):
        args, keep, case = _chunk(128, 32, 8, 64, 1600, seed=3, total_pages=100)
        table = torch.zeros(1, width, dtype=torch.int32, device=DEV)
        table[:, :100] = case["table"]
        args[6], args[7], args[15] = table.data_ptr(), width, width
        ws = _run(args, _native.load().helm_query_workspace_bytes(1, 32, 8, 64, 128, width, 16, 0))
        counts.append(ws[TICKETS:].view(torch.int32)[0].item())
        _check(keep, case, 0, 1600, 128, 8)
    assert counts[0] == counts[1]
