"""Prefill over pages of a multiple of 8 tokens that is not one of 16: the
tile-DMA kernel, whose slabs of 8 keys each lie in one page. The same keys in
16-token pages take the same kernel, so the outputs must agree bit for bit;
both are checked against the fp64 oracle. Pages of 12 tokens stay
on the kernel that looks up every row. Rows per q head on both
sides of a 128-row tile, packed rows, a table and the identity map, lengths
that end inside a slab, NaN in every dead slot."""
import pytest
import torch

from hrm_flashrenderer_amd import flash_attn_paged
from paged_ref import assert_close, paged_reference, seeded

pytestmark = pytest.mark.gpu


def _pages(kv, lengths, PS, table, seed):
    """[Hk, n, D] keys per sequence laid out in PS-token pages -> (pool, table)."""
    Hk, _, D = kv[0].shape
    per = [-(-n // PS) + 1 for n in lengths]
    width = max(per)
    if table:
        ids = torch.randperm(sum(per), generator=torch.Generator().manual_seed(seed)).tolist()
        pool = torch.full((1, Hk, sum(per), PS, D), float("nan"), dtype=torch.float16)
    else:
        pool = torch.full((len(kv), Hk, width, PS, D), float("nan"), dtype=torch.float16)
    bt = torch.full((len(kv), width), -1, dtype=torch.int32)
    for b, n in enumerate(lengths):
        for p in range(per[b]):
            phi = ids.pop() if table else b * width + p
            bt[b, p] = phi
            rows = kv[b][:, p * PS:min(n, (p + 1) * PS)]
            pool[phi // pool.size(2), :, phi % pool.size(2), :rows.size(1)] = rows
    return pool.cuda(), bt.cuda()


@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("B,Hq,Hk,M,D", [(4, 8, 2, 300, 64), (4, 4, 4, 129, 128), (260, 4, 1, 30, 128),
                                         (260, 4, 1, 30, 64)])
@pytest.mark.parametrize("PS", [8, 24, 40, 12])
def test_pages_of_eight(gpu, PS, B, Hq, Hk, M, D, table):
    lengths = [[601, 7, 333, 0][b % 4] + b // 4 for b in range(B)]
    lengths[3] = 0
    k = [seeded((Hk, n, D), 10 + b, device="cpu") for b, n in enumerate(lengths)]
    v = [seeded((Hk, n, D), 500 + b, device="cpu") for b, n in enumerate(lengths)]
    q = seeded((B, Hq, M, D), 1)
    hm = (torch.arange(Hq) // (Hq // Hk)).to(torch.int32).to(gpu)
    seqlen = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    offs = [max(0, n - M) for n in lengths]
    qo = torch.tensor(offs, dtype=torch.int32, device=gpu)
    outs = {}
    for ps in (PS, 16):
        kp, bt = _pages(k, lengths, ps, table, ps)
        vp, _ = _pages(v, lengths, ps, table, ps)
        outs[ps] = flash_attn_paged(q, kp, vp, seqlen, ps, hm, True, qo,
                                    block_table=bt if table else None)
    if PS % 8 == 0:
        assert torch.equal(outs[PS].view(torch.int16), outs[16].view(torch.int16))
    few = [(b, h) for b in range(4) for h in (0, Hq - 1)]
    ref = paged_reference(q, kp, vp, bt, lengths, 16, hm, True, offs, pairs=few)
    for (b, h), r in ref.items():
        assert_close(outs[PS][b, h].cpu().numpy(), r, f"PS={PS} b={b} h={h}")
