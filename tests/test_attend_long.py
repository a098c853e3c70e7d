"""Decode attention past 32 spans of 64 positions (the 8-wave workgroups, several spans each):
the cache lengths around the change of kernel and of the spans a workgroup takes, positions at the
first and last row of a span and of a workgroup's second one, every head size.  Bounds: as the
short-cache tests, fp16 probabilities and outputs (2^-11 each of the values' magnitude)."""
import math

import pytest
import torch

from spectra_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,hd,L,positions", [
    (6, 2, 128, 2048, (0, 2047)), (6, 2, 128, 2049, (0, 127, 128, 2047, 2048)),
    (4, 4, 64, 4095, (63, 4094)), (8, 1, 128, 4097, (4095, 4096)),
    (6, 2, 128, 9000, (130, 4096, 8191, 8192, 8999)), (2, 1, 256, 5000, (4095, 4096, 4999)),
    (3, 1, 64, 20000, (12288, 19999))])
def test_attend_long(hip, heads, kv, hd, L, positions):
    g = torch.Generator(device="cuda").manual_seed(L)
    k0, v0 = (torch.randn(kv, L, hd, generator=g, device="cuda").half() for _ in range(2))
    ws = torch.zeros(K.attend_workspace_bytes(heads, hd, L), dtype=torch.uint8, device="cuda")
    for p in positions:
        k, v = k0.clone(), v0.clone()
        k[:, p:], v[:, p:] = float("nan"), float("nan")  # rows not yet written may hold anything
        qkv = torch.randn((heads + 2 * kv) * hd, generator=g, device="cuda").half()
        pos = torch.tensor([p], device="cuda")
        for _ in range(2):  # the workspace's counters are left ready
            out = K.attend_decode(qkv, pos, None, None, heads, kv, k, v, ws)
        row = qkv.view(-1, hd)
        assert torch.equal(k[:, p], row[heads:heads + kv]) and torch.equal(v[:, p], row[heads + kv:])
        kd, vd = (t[:, :p + 1].double().repeat_interleave(heads // kv, 0) for t in (k, v))
        s = (kd * row[:heads].double()[:, None]).sum(-1) / math.sqrt(hd)
        ref = (torch.softmax(s, -1)[..., None] * vd).sum(1)
        assert (out.double() - ref).abs().max().item() <= 2.0 ** -10 * vd.abs().max().item(), p


@pytest.mark.parametrize("heads,kv,hd,L,positions", [
    (6, 2, 128, 9000, (0, 130, 4096, 4223, 8192, 8999)), (8, 1, 64, 5000, (127, 4100, 4999)),
    (4, 2, 256, 5000, (128, 4097, 4999))])
def test_attend_long_rope(hip, heads, kv, hd, L, positions):
    """With the rotation: the query heads and the new key, appended from a workgroup's first, second or
    third span, as fp32 products and sums rounded to fp16 once (the key bit for bit).  Bound as above."""
    g = torch.Generator(device="cuda").manual_seed(hd)
    k0, v0 = (torch.randn(kv, L, hd, generator=g, device="cuda").half() for _ in range(2))
    ang = torch.rand(L, hd // 2, generator=g, device="cuda") * 6.3
    cos, sin = ang.cos().contiguous(), ang.sin().contiguous()
    ws = torch.zeros(K.attend_workspace_bytes(heads, hd, L), dtype=torch.uint8, device="cuda")
    for p in positions:
        k, v = k0.clone(), v0.clone()
        k[:, p:], v[:, p:] = float("nan"), float("nan")
        qkv = torch.randn((heads + 2 * kv) * hd, generator=g, device="cuda").half()
        out = K.attend_decode(qkv, torch.tensor([p], device="cuda"), cos, sin, heads, kv, k, v, ws)
        row = qkv.view(-1, hd)
        a, b = row[:heads + kv, :hd // 2].float(), row[:heads + kv, hd // 2:].float()
        rot = torch.cat([a * cos[p] - b * sin[p], b * cos[p] + a * sin[p]], 1).half()
        assert torch.equal(k[:, p], rot[heads:]) and torch.equal(v[:, p], row[heads + kv:]), p
        assert bool(k[:, p + 1:].isnan().all()) and torch.equal(k[:, :p], k0[:, :p])
        kd, vd = (t[:, :p + 1].double().repeat_interleave(heads // kv, 0) for t in (k, v))
        s = (kd * rot[:heads].double()[:, None]).sum(-1) / math.sqrt(hd)
        ref = (torch.softmax(s, -1)[..., None] * vd).sum(1)
        assert (out.double() - ref).abs().max().item() <= 2.0 ** -10 * vd.abs().max().item(), p


@pytest.mark.parametrize("L,rows", [(2049, (0, 16)), (9000, (0, 16)), (9000, (4096, 4112)), (9000, (128, 9000))])
def test_attend_long_infinite_scores(hip, L, rows):
    """Scores of -inf weigh nothing, also over all 16 rows that a wave takes of a span, in its first
    span and in a later one.  Bound as above."""
    heads, kv, hd, p = 2, 1, 128, L - 1
    g = torch.Generator(device="cuda").manual_seed(L + rows[0])
    k, v = (torch.randn(kv, L, hd, generator=g, device="cuda").half() for _ in range(2))
    qkv = torch.randn((heads + 2 * kv) * hd, generator=g, device="cuda").half().abs()
    k[:, rows[0]:rows[1], 0] = float("-inf")
    ws = torch.zeros(K.attend_workspace_bytes(heads, hd, L), dtype=torch.uint8, device="cuda")
    out = K.attend_decode(qkv, torch.tensor([p], device="cuda"), None, None, heads, kv, k, v, ws)
    s = (k.double() * qkv.view(-1, hd)[:heads].double()[:, None]).sum(-1) / math.sqrt(hd)
    ref = (torch.softmax(s, -1)[..., None] * v.double()).sum(1)
    assert (out.double() - ref).abs().max().item() <= 2.0 ** -10 * v.double().abs().max().item()
