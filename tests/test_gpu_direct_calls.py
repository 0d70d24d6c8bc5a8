"""The operators run the body of their custom op without the dispatcher only
where nothing could tell: modes, fake tensors, gradients, subclasses, lazily
negated tensors and the profiler still meet the op, and a direct call bumps the
version counters of what it writes."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from hrm_flashrenderer_amd import (flash_attn, flash_attn_paged_append, ops, paged_kv_append,
                                   paged_kv_scatter)
from paged_ref import seeded

pytestmark = pytest.mark.gpu


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _qkv():
    return [seeded((1, 8, 40, 64), i) for i in range(3)]


def test_plain_call_is_direct_and_equal(gpu):
    q, k, v = _qkv()
    assert ops._direct(q, k, v, None)
    assert torch.equal(flash_attn(q, k, v), torch.ops.hrm_fa.flash_attn(q, k, v, True, 0, 0, None, None))


def test_dispatch_mode_profiler_and_forward_mode_meet_the_op(gpu):
    q, k, v = _qkv()
    with Seen() as seen:
        flash_attn(q, k, v)
    assert any("hrm_fa.flash_attn" in n for n in seen.names)
    with torch.profiler.profile() as prof:
        flash_attn(q, k, v)
    assert any("hrm_fa::flash_attn" in e.key for e in prof.key_averages())
    with torch.autograd.forward_ad.dual_level():
        assert not ops._direct(q)
    seen_by_vmap = []
    torch.vmap(lambda x: (seen_by_vmap.append(ops._direct(q)), x)[1])(torch.zeros(2, device=gpu))
    assert seen_by_vmap == [False]


def test_gradients_and_negated_tensors_meet_the_op(gpu):
    q, k, v = _qkv()
    want = flash_attn(q, k, v)
    out = flash_attn(q.clone().requires_grad_(), k, v)
    assert out.requires_grad and torch.equal(out.detach(), want)
    with pytest.raises(RuntimeError):
        out.sum().backward()
    with torch.no_grad():
        assert ops._direct(q.clone().requires_grad_())
    neg = torch._neg_view(-q)
    assert neg.is_neg() and torch.equal(flash_attn(neg, k, v), want)
    assert not ops._direct(torch.nn.Parameter(q, requires_grad=False))


def test_writes_bump_versions(gpu):
    kp, vp = seeded((1, 2, 4, 16, 64), 1), seeded((1, 2, 4, 16, 64), 2)
    kn, vn = seeded((1, 2, 1, 64), 3), seeded((1, 2, 1, 64), 4)
    seqlen = torch.tensor([5], dtype=torch.int32, device=gpu)
    hm = torch.tensor([0, 0, 1, 1], dtype=torch.int32, device=gpu)
    steps = (lambda: paged_kv_append(kp, vp, kn, vn, 3, 16),
             lambda: paged_kv_scatter(kp, vp, kn, vn, seqlen.view(1, 1), 16),
             lambda: flash_attn_paged_append(seeded((1, 4, 1, 64), 5), kp, vp, kn, vn, seqlen, 16, hm))
    for i, step in enumerate(steps):
        before = kp._version, vp._version, seqlen._version
        step()
        assert kp._version > before[0] and vp._version > before[1]
        assert (seqlen._version > before[2]) == (i == 2)
    with torch.inference_mode():
        paged_kv_append(kp.clone(), vp.clone(), kn, vn, 3, 16)
