"""Prefill grids that leave most of the device idle (few sequences and heads,
many keys) split their keys over several workgroups per 128-row tile and merge
the parts. Against the fp64 oracle: per-head and packed tiles, both head dims,
items on both sides of the 48-tile line in one batch, parts that some rows do
not see, padding rows, an invalid head, no mask, 8-token pages, contiguous
K/V; and a captured call replayed against the eager one."""
import pytest
import torch

from hrm_flashrenderer_amd import flash_attn, flash_attn_paged
from oracle import attention as ora
from paged_ref import assert_close, paged_reference, seeded
from test_gpu_decode_wide import _paged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hk,M,D,PS,lengths,causal,hidden", [
    (8, 2, 200, 128, 16, [1505, 1504, 6000], True, 0),
    (4, 4, 130, 64, 128, [4000, 300], True, 0),
    (8, 2, 70, 128, 16, [9000, 17, 2500], True, 0),      # packed: 280 rows per KV head
    (6, 3, 100, 64, 8, [3333], False, 0),                # packed
    (8, 8, 300, 128, 16, [5000], True, 2600),            # keys past row 2400 unseen: empty parts
    (5, 5, 257, 64, 24, [1536, 40, 2000], False, 0),
])
def test_split(gpu, Hq, Hk, M, D, PS, lengths, causal, hidden):
    B = len(lengths)
    k, v, bt = _paged(gpu, Hk, D, PS, lengths, True, 31)
    q = seeded((B, Hq, M, D), 3)
    hm = (torch.arange(Hq) * Hk // Hq).to(torch.int32)
    seqlen = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    offs = [max(0, n - M - hidden) for n in lengths]
    qo = torch.tensor(offs, dtype=torch.int32, device=gpu) if causal else 0
    q_lens = [M if b != 1 else M - 60 for b in range(B)]
    for b, n in enumerate(q_lens):
        q[b, :, n:] = float("nan")
    ql = torch.tensor(q_lens, dtype=torch.int32, device=gpu)
    out = flash_attn_paged(q, k, v, seqlen, PS, hm.to(gpu), causal, qo, block_table=bt.to(gpu),
                           q_lens=ql).cpu()
    q0 = torch.nan_to_num(q)
    ref = paged_reference(q0, k, v, bt, lengths, PS, hm, causal, offs)
    for (b, h), r in ref.items():
        n = q_lens[b]
        assert_close(out[b, h, :n].numpy(), r[:n], f"b={b} h={h}")
        assert (out[b, h, n:] == 0).all()
    bad = hm.clone()
    bad[1] = Hk
    out2 = flash_attn_paged(q, k, v, seqlen, PS, bad.to(gpu), causal, qo, block_table=bt.to(gpu),
                            q_lens=ql, heads_per_kv=Hq // Hk).cpu()
    assert torch.isnan(out2[0, 1, :q_lens[0]]).all()
    assert torch.isfinite(out2[:, 2:]).all()


def test_split_contiguous(gpu):
    q, k, v = seeded((2, 8, 150, 128), 1), seeded((2, 2, 3001, 128), 2), seeded((2, 2, 3001, 128), 3)
    out = flash_attn(q, k, v, True, 2851)
    kk, vv = (x.repeat_interleave(4, 1).cpu() for x in (k, v))
    assert_close(out.cpu().numpy(), ora.attention_f64(q.cpu(), kk, vv, True, 2851, 0))


def test_split_in_a_graph(gpu):
    q, k, v = seeded((1, 8, 256, 64), 1), seeded((1, 8, 2500, 64), 2), seeded((1, 8, 2500, 64), 3)
    flash_attn(q, k, v, True, 2244)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = flash_attn(q, k, v, True, 2244)
    for i in range(3):
        q.copy_(seeded((1, 8, 256, 64), 10 + i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, flash_attn(q, k, v, True, 2244))


@pytest.mark.parametrize("Hq,Hk,M,N,D,causal", [
    (8, 8, 129, 129, 128, True),    # two items per head, the second with one live row
    (4, 2, 300, 31, 64, False),     # one key tile: group 1 has none
    (6, 3, 200, 1000, 128, True),   # rows that do not see group 1's last tile
    (32, 8, 1024, 1024, 64, True),  # 256 items: the largest such grid
    (33, 3, 1024, 1024, 64, True),  # 264 items: one group
])
def test_two_groups(gpu, Hq, Hk, M, N, D, causal):
    """Grids of at most 256 items run two wave groups per item."""
    q, k, v = seeded((1, Hq, M, D), 1), seeded((1, Hk, N, D), 2), seeded((1, Hk, N, D), 3)
    out = flash_attn(q, k, v, causal, max(0, N - M))
    for h in (0, Hq // 2, Hq - 1):
        ref = ora.attention_f64(q[:, h:h + 1].cpu(), k[:, h * Hk // Hq:h * Hk // Hq + 1].cpu(),
                                v[:, h * Hk // Hq:h * Hk // Hq + 1].cpu(), causal, max(0, N - M), 0)
        assert_close(out[:, h:h + 1].cpu().numpy(), ref, f"h={h}")
