"""The row dequant at the edges of its passes and segments: a pass is 512 16-bit (256 fp32) outputs
of a row, of which the last may be partial (its idle lanes still place outliers), a segment at most
4096; rows without outliers, with one in every column of the last run, and past the 128 entries a
wave holds.  Bit-exact: the same roundings as the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from spectra_amd import compressor as C
from spectra_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dt", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("k,bs,marlin", [(64, 64, True), (544, 32, False), (576, 64, True), (3072, 64, True),
                                         (4160, 64, False), (7776, 32, True), (8192, 128, True)])
def test_pass_and_segment_edges(hip, k, bs, marlin, out_dt):
    n = 37
    rng = np.random.default_rng(k + bs)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float16)
    mask = rng.random((n, k)) < 0.01
    mask[0] = False
    mask[1, -32:] = True
    mask[n - 1, : min(k, 200)] = True
    w[mask] *= 10
    q = O.nf4_quantize(w, "float16", bs, 0, mask, marlin)
    ref = O.nf4_dequant(q["packed"], q["absmax"], marlin, out_dt, q["rowptr"], q["col"], q["val"], blocksize=bs)
    d = {name: torch.from_numpy(np.ascontiguousarray(q[name])).cuda() for name in ("packed", "absmax", "col", "val", "rowptr")}
    y = K.w4_dequant(d["packed"], d["absmax"], None, out_dtype=getattr(torch, out_dt), codebook="nf4", group_size=bs,
                     marlin_layout=marlin, outlier_idx=d["col"], outlier_w=d["val"], outlier_rowptr=d["rowptr"])
    y = y.view(torch.int32 if out_dt == "float32" else torch.int16).cpu().numpy()
    assert np.array_equal(y, np.ascontiguousarray(ref).view(y.dtype))


@pytest.mark.parametrize("k,had,off,dt", [(192, 64, 0, torch.float16), (4160, 32, 0, torch.bfloat16),
                                          (4224, 128, 1, torch.float16), (1024, 512, 0, torch.bfloat16)])
def test_activations_rotated_in_the_same_launch(hip, k, had, off, dt):
    """Prompt-size calls that rotate the activations (4 M < N): rows of a partial and of more than one
    4096-element segment, unaligned rows.  Bound: operands and result rounded to the activations'
    dtype, u = 2^-11 (fp16) or 2^-8 (bf16) each: rel-L2 <= 3 u."""
    m, n = 513, 2080
    g = torch.Generator(device="cuda").manual_seed(k)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    mask = torch.rand(n, k, generator=g, device="cuda") < 0.01
    q = C.quantize_nf4(torch.where(mask, w * 10, w).half(), 64, 0, mask, True)
    buf = torch.randn(m * (k + 8) + 8, generator=g, device="cuda").to(dt)
    x = buf[off: off + m * (k + 8)].view(m, k + 8)[:, :k]
    assert not K.prefill_rotates_weights(m, n, k, had)
    y = K.batched_w4a16_gemm(x, q.packed, q.absmax, None, outlier_idx=q.col, outlier_w=q.val, marlin_layout=True,
                             codebook="nf4", group_size=64, hadamard_block=had, outlier_rowptr=q.rowptr)
    dense = O.nf4_dequant(q.packed.cpu().numpy(), q.absmax.cpu().numpy(), True, "float32", q.rowptr.cpu().numpy(),
                          q.col.cpu().numpy(), q.val.cpu().numpy())
    ref = torch.from_numpy(O.rotate_blocks(x.float().cpu().numpy(), had)).double() @ torch.from_numpy(dense).double().t()
    err = (y.double().cpu() - ref).norm() / ref.norm()
    assert err <= 3 * (2.0 ** -11 if dt == torch.float16 else 2.0 ** -8), err
