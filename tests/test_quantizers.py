"""The register quantizers and the mask-to-CSR kernels at their edges, bit-exact against the
oracle: ragged segments (K not a multiple of 512), every block size they take and the first
they leave to the LDS kernel, odd group counts, unaligned rows, infinite / NaN / zero / subnormal
groups, quotients on the code steps, masks without entries and with full rows."""
import numpy as np
import pytest
import torch

import oracle as O
from spectra_amd import compressor as C

pytestmark = pytest.mark.gpu


def _w(n, k, dt, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    w[0, :64] = 0.0
    w[-1, :32] = 0.5          # a constant group
    w[n // 2, 64:96] = -1e-7  # fp16 subnormals
    w[n // 3, 96:128] *= 1e-6
    t = torch.from_numpy(w).to({"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}[dt])
    return t


def _np(t, dt):  # the oracle takes bf16 as its bits
    return t.view(torch.int16).numpy().view(np.uint16) if dt == "bfloat16" else t.numpy()


@pytest.mark.parametrize("dt", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("n,k,pad", [(3, 96, 0), (9, 544, 0), (17, 2080, 8), (8, 1024, 3)])
def test_group32_edges(hip, dt, n, k, pad):
    w = _w(n, k + pad, dt, n * k + pad)[:, :k]
    oidx = np.array([0, 7, 8, k - 1])
    got = C.quantize_group32(w.cuda(), 32, torch.from_numpy(oidx))
    ref = O.compute_group32_quant(w.float().numpy(), oidx)
    for g, r, what in zip(got, ref, ("packed", "scales", "zeros")):
        assert np.array_equal(g.cpu().numpy(), r), what


@pytest.mark.parametrize("dt", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("n,k,bs,had,marlin", [(5, 576, 64, 64, True), (3, 1536, 32, 512, False),
                                               (4, 1024, 512, 2, True), (6, 2048, 128, 0, False),
                                               (2, 2048, 64, 1024, True), (2, 2048, 1024, 128, True)])
def test_nf4_edges(hip, dt, n, k, bs, had, marlin):
    w = _w(n, k, dt, n * k + bs + had)
    rng = np.random.default_rng(had)
    mask = rng.random((n, k)) < 0.02
    mask[0], mask[-1] = False, True  # a row without entries, a full one
    q = C.quantize_nf4(w.cuda(), bs, had, torch.from_numpy(mask).cuda(), marlin)
    ref = O.nf4_quantize(_np(w, dt), dt, bs, had, mask, marlin)
    assert np.array_equal(q.rowptr.cpu().numpy(), ref["rowptr"])
    assert np.array_equal(q.col.cpu().numpy(), ref["col"])
    for name in ("val", "absmax"):
        assert np.array_equal(getattr(q, name).cpu().numpy().view(np.uint16), ref[name].view(np.uint16)), name
    assert np.array_equal(q.packed.cpu().numpy(), ref["packed"])


def test_nf4_code_steps(hip):
    """Values whose quotient by the block's absmax lies on either side of every code step (200
    floats around each, for absmax 1 and for absmaxes whose reciprocal is inexact)."""
    codes = O.NF4_CODEBOOK.astype(np.float64)
    rows = []
    for a in (1.0, 0.7939453125, 3.0, 1.7e-4):
        a = float(np.float16(a))
        for i in range(15):
            mid = np.float32((codes[i] + codes[i + 1]) / 2 * a)
            near = (mid.view(np.int32) + np.arange(-100, 100)).astype(np.int32).view(np.float32)
            for c in range(0, 200, 50):
                blk = np.zeros(64, np.float32)
                blk[:50], blk[63] = near[c:c + 50], a
                rows.append(blk)
    w = np.concatenate(rows).reshape(-1, 256)
    q = C.quantize_nf4(torch.from_numpy(w).cuda(), 64, 0, None, True)
    ref = O.nf4_quantize(w, "float32", 64, 0, None, True)
    assert np.array_equal(q.packed.cpu().numpy(), ref["packed"])


def test_nonfinite_groups(hip):
    """An infinity or a NaN stays in its own group (torch's min / max would spread a NaN: the
    quantizer takes the numbers)."""
    w = torch.randn(4, 128, generator=torch.Generator().manual_seed(1)) * 0.02
    ref_a, ref_b = C.quantize_group32(w.cuda()), C.quantize_nf4(w.cuda())
    w[1, 5], w[2, 70] = float("inf"), float("nan")
    for ref, got in ((ref_a[0], C.quantize_group32(w.cuda())[0]), (ref_b.packed, C.quantize_nf4(w.cuda()).packed)):
        same = (ref == got).cpu()
        assert same[0].all() and same[3].all() and same[1, 32:].all() and same[2, :32].all()
    q = C.quantize_nf4(w.cuda())
    assert torch.isinf(q.absmax[1, 0]) and int(q.packed[2, 32 + 6]) & 15 == 0  # NaN: code 0


@pytest.mark.parametrize("n,k,stride", [(1, 1, 1), (5, 33, 33), (4099, 48, 64), (7, 4096, 4096)])
def test_csr_from_mask(hip, n, k, stride):
    g = torch.Generator().manual_seed(n)
    mask = (torch.rand(n, stride, generator=g) < 0.1)
    mask[0, :] = True
    m = mask.cuda()[:, :k]
    rowptr, col = C.csr_from_mask(m)
    want_r, want_c = C.csr_from_mask(mask[:, :k])  # (host masks go through torch)
    assert torch.equal(rowptr.cpu(), want_r) and torch.equal(col.cpu(), want_c)
    empty = C.csr_from_mask(torch.zeros_like(m))
    assert int(empty[0].abs().sum()) == 0 and empty[1].numel() == 0
