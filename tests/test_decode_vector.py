"""The 16-byte paths of the RoPE append and of SiLU-mul against the element paths, which the same
values one element off a 16-byte boundary take: the same arithmetic, so the same bits.  Head sizes at
the smallest group, item counts below and past a workgroup, strided rows, positions outside the cache."""
import pytest
import torch

from spectra_amd import kernels as K

pytestmark = pytest.mark.gpu


def _off(t):
    """The same values and strides one element past a 16-byte boundary."""
    buf = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[1: 1 + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 16 and t.data_ptr() % 16 == 0
    return v


@pytest.mark.parametrize("heads,kv,hd,tokens,pad", [(1, 1, 16, 1, 0), (3, 1, 48, 5, 8), (24, 8, 128, 77, 0),
                                                    (16, 16, 64, 3, 16), (32, 4, 256, 2, 0)])
def test_rope_append(hip, heads, kv, hd, tokens, pad):
    g = torch.Generator(device="cuda").manual_seed(hd + tokens)
    lmax = tokens + 9
    width = (heads + 2 * kv) * hd
    qkv = torch.randn(tokens, width + pad, generator=g, device="cuda").half()
    pos = torch.randperm(lmax, generator=g, device="cuda")[:tokens].contiguous()
    if tokens > 2:
        pos[0], pos[1] = lmax, -1  # nothing is written for these
    ang = torch.rand(lmax, hd // 2, generator=g, device="cuda") * 6
    cos, sin = ang.cos(), ang.sin()
    outs = []
    for q in (qkv, _off(qkv)):
        kc, vc = (torch.full((kv, lmax, hd), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
        rot = torch.full((tokens, heads, hd), 7.0, dtype=torch.float16, device="cuda")
        K.rope_append(q[:, :width], pos, cos, sin, heads, kv, kc, vc, rot)
        outs.append((rot, kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    last = tokens - 1  # and the vector path against the definition
    x = qkv[last, : (heads + kv) * hd].float().view(heads + kv, hd)
    c, s = cos[pos[last]], sin[pos[last]]
    lo, hi = x[:, : hd // 2], x[:, hd // 2:]
    ref = torch.cat([lo * c - hi * s, hi * c + lo * s], 1)
    got = torch.cat([outs[0][0][last], outs[0][1][:, pos[last]]]).float()
    assert (got - ref).abs().max() <= 2.0 ** -10 * ref.abs().max()  # one fp16 rounding


@pytest.mark.parametrize("rows,inter,pad", [(1, 8, 0), (3, 264, 8), (33, 8192, 0), (2, 2048, 24)])
def test_silu_mul(hip, rows, inter, pad):
    g = torch.Generator(device="cuda").manual_seed(inter)
    gu = (torch.randn(rows, 2 * inter + pad, generator=g, device="cuda") * 4).half()
    gu[0, 0], gu[0, 1], gu[0, 2] = float("inf"), float("-inf"), float("nan")
    a, b = K.silu_mul(gu[:, : 2 * inter]), K.silu_mul(_off(gu)[:, : 2 * inter])
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
