"""The row dequant at the edges of its passes and segments: a pass is 512 16-bit (256 fp32) outputs
of a row, of which the last may be partial (its idle lanes still place outliers), a segment at most
4096; rows without outliers, with one in every column of the last run, and past the 128 entries a
wave holds.  Bit-exact: the same roundings as the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
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
