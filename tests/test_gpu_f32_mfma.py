"""fp32 flash_attn on the fp32 matrix instruction, at the edges of its 32-row
and 32-key tiles and of its four-way key split, in both work orders ((sequence,
KV head) pairs divisible by 8 or not), with offsets, GQA and rows that see no
key; and the path that tensors off a 16-byte boundary keep. Bar: the fp32 bar
of the other fp32 tests, against the fp64 oracle."""
import pytest
import torch

from hrm_flashrenderer_amd import flash_attn
from oracle import attention as ora
from paged_ref import assert_close_f32, seeded

pytestmark = pytest.mark.gpu

SHAPES = [  # B, Hq, Hk, M, N, D, causal, q_offset, k_offset
    (1, 8, 8, 1, 1, 64, True, 0, 0),
    (1, 8, 8, 31, 31, 128, True, 0, 0),
    (2, 4, 4, 32, 33, 64, True, 1, 0),
    (1, 3, 1, 33, 129, 128, True, 96, 0),
    (1, 16, 8, 65, 127, 64, False, 0, 0),
    (1, 5, 5, 40, 300, 128, True, 100, 150),   # rows 0..49 see no key: NaN
    (3, 8, 8, 97, 160, 64, True, [0, 63, 500], [0, 7, 0]),
    (1, 2, 2, 1, 1025, 128, False, 0, 0),
]


def _check(gpu, B, Hq, Hk, M, N, D, causal, qo, ko, shift):
    def tensor(shape, seed):
        t = seeded(shape, seed, dtype=torch.float32)
        if not shift:
            return t
        buf = torch.zeros(t.numel() + 1, device=t.device)
        buf[1:] = t.view(-1)
        return buf[1:].view(shape)   # contiguous, 4 bytes off a 16-byte boundary

    q, k, v = tensor((B, Hq, M, D), 1), tensor((B, Hk, N, D), 2), tensor((B, Hk, N, D), 3)
    dev = [torch.tensor(x, dtype=torch.int32, device=gpu) if isinstance(x, list) else x
           for x in (qo, ko)]
    out = flash_attn(q, k, v, causal, *dev).cpu()
    kk, vv = (x.repeat_interleave(Hq // Hk, 1).cpu() for x in (k, v))
    for b in range(B):
        at = [x[b] if isinstance(x, list) else x for x in (qo, ko)]
        ref = ora.attention_f64(q[b:b + 1].cpu(), kk[b:b + 1], vv[b:b + 1], causal, *at)
        assert_close_f32(out[b:b + 1], ref, f"b={b}")


@pytest.mark.parametrize("shape", SHAPES)
def test_tile_edges(gpu, shape):
    _check(gpu, *shape, shift=False)


@pytest.mark.parametrize("shape", SHAPES[3:5])
def test_unaligned_views(gpu, shape):
    _check(gpu, *shape, shift=True)
