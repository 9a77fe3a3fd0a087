"""The 16-byte form of QK-norm + RoPE (+ append) against the general form: the same values laid out at
4-byte aligned, 16-byte misaligned addresses take the general kernels, and both must give the same
bits (they sum in the same order). Token counts around a wave's rows and above one round of
workgroups, every head_dim and dtype, rotations of none, part and all of a head, skipped slots."""
import pytest
import torch

from helpers import bits, say
from tileinfer_amd.kernels import qknorm_rope, qknorm_rope_append

pytestmark = pytest.mark.gpu


def shifted(t):
    """A copy of t two elements past a 16-byte boundary, same strides."""
    flat = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    out = flat[2:2 + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == 4
    return out


@pytest.mark.parametrize("d,dtype", [(256, torch.bfloat16), (256, torch.float16),
                                     (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("t,hq,hkv,rd", [(1, 1, 1, 0), (1, 24, 4, 64), (3, 5, 1, 16), (7, 6, 2, 128),
                                         (65, 3, 3, 64), (2600, 8, 2, 64)])
def test_vector_form_equals_general_form(t, hq, hkv, rd, d, dtype, dev):
    say(f"qknorm vec t={t} hq={hq} hkv={hkv} d={d} rd={rd} {dtype}")
    g = torch.Generator(device=dev).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)  # noqa: E731
    q, k, v = rnd(t, hq, d), rnd(t, hkv, d), rnd(t, hkv, d)
    qw, kw, cos, sin = rnd(d), rnd(d), rnd(t, rd), rnd(t, rd)
    slots = torch.randperm(t + 5, generator=g, device=dev)[:t].to(torch.int32)
    slots[t // 2] = -1 if t > 1 else slots[0]
    caches = [torch.zeros(t + 5, hkv * d, dtype=dtype, device=dev) for _ in range(4)]
    out = qknorm_rope_append(q, k, v, qw, kw, cos, sin, caches[0], caches[1], slots)
    ref = qknorm_rope_append(shifted(q), k, v, qw, kw, cos, sin, caches[2], caches[3], slots)
    for a, b in [(out, ref), (caches[0], caches[2]), (caches[1], caches[3])]:
        assert torch.equal(bits(a), bits(b))
    assert torch.equal(bits(qknorm_rope(q, qw, cos, sin)), bits(out))
    assert torch.equal(bits(qknorm_rope(shifted(q), qw, cos, sin)), bits(out))
    inplace = q.clone()
    qknorm_rope(inplace, qw, cos, sin, out=inplace)
    assert torch.equal(bits(inplace), bits(out))
