"""Prefill attention kernel against the fp64 softmax at the edges of its tiles: one token, the
64-query and 128-key borders, grouped queries, a cache longer than the prompt whose unused rows
hold NaN, and scores far apart.  Bounds: probabilities and outputs are fp16 (2^-11 each, relative
to the outputs' magnitude <= max |v|), scores fp32."""
import math

import pytest
import torch

from spectra_amd import kernels as K

pytestmark = pytest.mark.gpu


def _ref(q, k, v):
    T, heads, d = q.shape
    g = heads // k.shape[0]
    kd, vd = (t[:, :T].double().repeat_interleave(g, 0) for t in (k, v))
    s = torch.matmul(q.double().transpose(0, 1).contiguous(), kd.transpose(1, 2).contiguous()) / math.sqrt(d)
    s = s.masked_fill(torch.ones(T, T, device=q.device).triu(1).bool(), float("-inf"))
    return torch.matmul(torch.softmax(s, -1), vd).transpose(0, 1)


@pytest.mark.parametrize("heads,kv,d", [(6, 2, 128), (4, 4, 64), (8, 1, 128)])
@pytest.mark.parametrize("T", [1, 31, 64, 65, 128, 129, 200, 515])
def test_attend_prefill(hip, heads, kv, d, T):
    g = torch.Generator(device="cuda").manual_seed(T + d)
    q = torch.randn(T, heads, d, generator=g, device="cuda").half()
    k = torch.randn(kv, T + 70, d, generator=g, device="cuda").half()
    v = torch.randn(kv, T + 70, d, generator=g, device="cuda").half()
    k[:, T:], v[:, T:] = float("nan"), float("nan")
    out = K.attend_prefill(q, torch.arange(T, device="cuda"), T, k, v)
    err = (out.double() - _ref(q, k, v)).abs().max().item()
    assert err <= 2.0 ** -10 * v[:, :T].abs().max().item(), err


@pytest.mark.parametrize("T,L", [(40, 170), (100, 100), (70, 300)])
def test_attend_prefill_positions(hip, T, L):
    """A chunk at the end of a longer context, and positions in any order."""
    g = torch.Generator(device="cuda").manual_seed(T)
    q = torch.randn(T, 4, 128, generator=g, device="cuda").half()
    k, v = (torch.randn(2, 320, 128, generator=g, device="cuda").half() for _ in range(2))
    for pos in (torch.arange(L - T, L, device="cuda"), torch.randperm(L, generator=g, device="cuda")[:T].contiguous()):
        out = K.attend_prefill(q, pos, L, k, v)
        kd, vd = (t[:, :L].double().repeat_interleave(2, 0) for t in (k, v))
        s = torch.matmul(q.double().transpose(0, 1).contiguous(), kd.transpose(1, 2).contiguous()) / math.sqrt(128)
        s = s.masked_fill(torch.arange(L, device="cuda")[None, None] > pos[None, :, None], float("-inf"))
        ref = torch.matmul(torch.softmax(s, -1), vd).transpose(0, 1)
        assert (out.double() - ref).abs().max().item() <= 2.0 ** -10 * v.abs().max().item()


def test_attend_prefill_peaked_scores(hip):
    """Scores of +-thousands: one key takes all the weight, whichever tile it lies in."""
    T, d = 300, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    q = (torch.randn(T, 2, d, generator=g, device="cuda") * 60).half()
    k = (torch.randn(2, T, d, generator=g, device="cuda") * 60).half()
    v = torch.randn(2, T, d, generator=g, device="cuda").half()
    out, ref = K.attend_prefill(q, torch.arange(T, device="cuda"), T, k, v), _ref(q, k, v)
    assert torch.isfinite(out).all()
    # |score| <= ~6e4 in fp32: absolute error up to 6e4 * 2^-23 * few in the exponent
    assert ((out.double() - ref).norm() / ref.norm()).item() <= 2e-2


def test_attend_prefill_refuses(hip):
    def call(T, L, d, keys):
        z = torch.zeros(2, L, d, device="cuda", dtype=torch.float16)
        return K.attend_prefill(torch.zeros(T, 2, d, device="cuda", dtype=torch.float16),
                                torch.arange(T, device="cuda"), keys, z, z)

    with pytest.raises(RuntimeError):
        call(4, 8, 96, 4)
    with pytest.raises(ValueError):  # more keys than cache rows
        call(9, 8, 64, 9)
