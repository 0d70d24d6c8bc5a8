"""Decode on 32-key LDS tiles (more than 16 query rows per KV head, or pages of
8, 24, ... tokens): every row-block count at its edges (16/17, 32/33, 64/65 rows
and a second pass, which calls without a heads_per_kv bound take; with one,
more than 64 rows run on packed prefill tiles in the decode workspace), slabs of 16 and of 8 keys, pages with and without a table,
contiguous K/V, rows that see only part of the keys, padding rows, rotary
queries and lengths that end inside a slab or leave waves without a tile,
against the fp64 oracle; dead slots hold NaN. The one-call decode step equals
its two calls bit for bit where the step leaves the fused kernels."""
import pytest
import torch

from hrm_flashrenderer_amd import (flash_attn, flash_attn_paged, flash_attn_paged_append,
                                   paged_kv_append)
from oracle import attention as ora
from paged_ref import assert_close, paged_reference, poison_dead_slots, seeded
from test_gpu_rope import _tables

pytestmark = pytest.mark.gpu


def _paged(gpu, Hk, D, PS, lengths, table, seed):
    per = [-(-n // PS) + 1 for n in lengths]
    B, width = len(lengths), max(per)
    bt = torch.full((B, width), -1, dtype=torch.int32)
    if table:
        ids = torch.randperm(sum(per), generator=torch.Generator().manual_seed(seed)).tolist()
        shape = (1, Hk, sum(per), PS, D)
        for b in range(B):
            bt[b, :per[b]] = torch.tensor([ids.pop() for _ in range(per[b])], dtype=torch.int32)
    else:
        shape = (B, Hk, width, PS, D)
        bt = torch.arange(B * width, dtype=torch.int32).view(B, width)
    k, v = seeded(shape, seed), seeded(shape, seed + 1)
    poison_dead_slots(k, v, bt, lengths, PS)
    return k, v, bt


@pytest.mark.parametrize("Hq,Hk,M,D,PS,table,causal", [
    (17, 1, 1, 128, 16, True, False),
    (8, 2, 8, 128, 32, False, True),     # 32 rows
    (33, 1, 1, 64, 16, True, False),
    (24, 3, 5, 128, 128, True, True),    # 40 rows
    (16, 2, 8, 64, 64, True, True),      # 64 rows
    (13, 1, 5, 128, 16, True, True),     # 65 rows: a second pass
    (15, 1, 9, 64, 16, True, True),      # 135 rows: a second pass at D = 64
    (4, 4, 1, 128, 8, True, False),      # one row per KV head, 8-token pages
    (10, 2, 1, 64, 24, False, False),
    (20, 2, 4, 128, 24, True, True),     # 40 rows
    (12, 1, 8, 64, 8, True, True),       # 96 rows
    (71, 1, 1, 128, 16, True, False),    # 71 rows of one token
])
def test_wide_decode(gpu, Hq, Hk, M, D, PS, table, causal):
    lengths = [1, 40, 777, 0, 128, 2049]
    B = len(lengths)
    k, v, bt = _paged(gpu, Hk, D, PS, lengths, table, 5)
    q = seeded((B, Hq, M, D), 9)
    hm = (torch.arange(Hq) * Hk // Hq).flip(0).to(torch.int32).to(gpu)
    seqlen = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    offs = [max(0, n - M) for n in lengths]
    qo = torch.tensor(offs, dtype=torch.int32, device=gpu) if causal else 0
    tab = bt.to(gpu) if table else None
    out = flash_attn_paged(q, k, v, seqlen, PS, hm, causal, qo, block_table=tab)
    unbound = torch.ops.hrm_fa.flash_attn_paged(
        q, k, v, seqlen, PS, hm, causal, 0, 0, qo if causal else None, None, tab, None, None, None, 0)
    ref = paged_reference(q, k, v, bt, lengths, PS, hm, causal, offs)
    for (b, h), r in ref.items():
        assert_close(out[b, h].cpu().numpy(), r, f"b={b} h={h}")
        assert_close(unbound[b, h].cpu().numpy(), r, f"no bound b={b} h={h}")
    # padding rows come out as zeros and leave the others alone
    lens = torch.tensor([M, max(0, M - 2), M, M, 1, M], dtype=torch.int32, device=gpu)
    part = flash_attn_paged(q, k, v, seqlen, PS, hm, causal, qo, block_table=tab, q_lens=lens)
    for b, n in enumerate(lens.tolist()):
        assert (part[b, :, n:] == 0).all()
        assert_close(part[b, :, :n].cpu().numpy(), out[b, :, :n].double().cpu().numpy(), f"q_lens b={b}")


@pytest.mark.parametrize("Hq,Hk,M,N,D", [(40, 2, 1, 333, 128), (8, 2, 8, 2000, 64), (64, 2, 1, 31, 128)])
def test_wide_contiguous(gpu, Hq, Hk, M, N, D):
    q, k, v = seeded((3, Hq, M, D), 1), seeded((3, Hk, N, D), 2), seeded((3, Hk, N, D), 3)
    out = flash_attn(q, k, v, True, N - M)
    kk, vv = (x.repeat_interleave(Hq // Hk, 1).cpu() for x in (k, v))
    assert_close(out.cpu().numpy(), ora.attention_f64(q.cpu(), kk, vv, True, N - M, 0))


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("Hq,Hk,D,PS", [(48, 2, 128, 16), (8, 2, 64, 8), (20, 1, 128, 24), (71, 1, 64, 16)])
def test_step_equals_two_calls(gpu, Hq, Hk, D, PS, rope):
    lengths = [5, 0, 300, 127]
    B = len(lengths)
    k, v, bt = _paged(gpu, Hk, D, PS, lengths, True, 21)
    q, kn, vn = seeded((B, Hq, 1, D), 1), seeded((B, Hk, 1, D), 2), seeded((B, Hk, 1, D), 3)
    hm = (torch.arange(Hq) * Hk // Hq).to(torch.int32).to(gpu)
    tab = bt.to(gpu)
    tables = _tables(512, D, gpu) if rope else None
    start = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    k2, v2 = k.clone(), v.clone()
    paged_kv_append(k2, v2, kn, vn, start, PS, block_table=tab, rope=tables)
    want = flash_attn_paged(q, k2, v2, start + 1, PS, hm, False, start, block_table=tab, rope=tables)
    seqlen = start.clone()
    got = flash_attn_paged_append(q, k, v, kn, vn, seqlen, PS, hm, block_table=tab, rope=tables)
    for a, b in ((got, want), (k, k2), (v, v2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(seqlen, start + 1)
