"""The mid-size batch family (17 rows up to 96 by outlier density, 160 without outliers, 511 on shapes
with few tiles) and the 256-row tiles beside it against the float64 product of W_eff, at the edges of
the family's tiles: 32-row tiles and the change from
four chunks a stage to two and to one, columns past the last 128, K of an odd number of 64-chunks and
of a partial quad, every number of K splits' remainder, both formats and nibble orders, rotation
blocks, dense and empty outlier rows, codes under the outliers that are not zero, unaligned and
strided operands.  Bound: fp16 operands (weights and activations rounded once, 2^-11 each) and the
result's rounding: rel-L2 <= 1e-3 in fp16, 5e-3 in bf16, as for the GEMM family."""
import numpy as np
import pytest
import torch

import oracle as O
from spectra_amd import _lib as L
from spectra_amd import compressor as C
from spectra_amd import kernels as K

pytestmark = pytest.mark.gpu

DT = {"float16": torch.float16, "bfloat16": torch.bfloat16}


def _nf4(n, k, had, ratio, marlin, bs=64, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + n + k)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    mask = None
    if ratio:
        mask = torch.rand(n, k, generator=g, device="cuda") < ratio
        mask[0] = False
        mask[n - 1, : k // 2] = True
        w = torch.where(mask, w * 10, w)
    return C.quantize_nf4(w.half(), bs, 0, mask, marlin), had


def _dense(q, bs=64):
    rp = q.rowptr.cpu().numpy()
    return O.nf4_dequant(q.packed.cpu().numpy(), q.absmax.cpu().numpy(), q.marlin_layout, "float32",
                         rp, q.col.cpu().numpy(), q.val.cpu().numpy(), blocksize=bs)


def _runs_mid(hip, ops, m, dt):
    """Whether a call with the workspace the library asks for runs on this family."""
    adt = L.F16 if dt == "float16" else L.BF16
    return bool(hip.spectra_w4a16_gemm_mid(ops.ptr(), m, hip.spectra_w4a16_gemm_workspace(ops.ptr(), m, adt)))


def _check(y, x, w, had, bias, dt):
    xr = O.rotate_blocks(x.float().cpu().numpy(), had) if had else x.float().cpu().numpy()
    ref = torch.from_numpy(xr.astype(np.float64)).cuda() @ torch.from_numpy(w.astype(np.float64)).cuda().t()
    if bias is not None:
        ref = ref + bias.double()
    rel = ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()  # the worst row
    assert rel <= (1e-3 if dt == "float16" else 5e-3), rel


@pytest.mark.parametrize("m,n,k,had,ratio,marlin,dt,bs,mid", [
    (17, 128, 1024, 128, 0.01, True, "float16", 64, True),
    (32, 129, 64, 64, 0.05, False, "bfloat16", 64, True),     # one chunk
    (33, 1000, 1088, 64, 0.01, True, "float16", 32, True),    # 17 chunks, 32-blocks
    (64, 3072, 3072, 512, 0.005, True, "float16", 64, False),  # (the 256-row tiles, by density)
    (64, 3072, 3072, 512, 0.0025, True, "float16", 64, True),
    (65, 640, 2112, 32, 0.02, False, "float16", 64, True),    # 33 chunks
    (96, 5120, 1024, 128, 0.005, True, "bfloat16", 64, False),
    (96, 5120, 2048, 128, 0.001, True, "bfloat16", 64, True),
    (97, 1537, 1024, 0, 0.0, True, "float16", 64, True),      # two chunks a stage, 4 row tiles
    (129, 384, 1344, 0, 0.0, False, "float16", 64, True),     # one chunk a stage, 3 + 3 row tiles
    (160, 2048, 2048, 256, 0.0, True, "bfloat16", 64, True),
    (255, 129, 3072, 2, 0.01, True, "float16", 64, True),     # few tiles: any row count
    (257, 77, 4096, 128, 0.01, False, "float16", 64, True),   # two row blocks
    (511, 33, 6144, 0, 0.01, True, "float16", 128, True),
])
def test_mid_nf4(hip, m, n, k, had, ratio, marlin, dt, bs, mid):
    q, _ = _nf4(n, k, had, ratio, marlin, bs)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").to(DT[dt])
    x[m - 1] *= 1000.0  # rows of very different size
    x[0] *= 1e-3
    bias = torch.randn(n, generator=g, device="cuda")
    col, val = q.outliers()
    rowptr = q.rowptr if col is not None else None
    ops = K.QWeightOperands(q.packed, q.absmax, None, k, codebook="nf4", group_size=bs, hadamard_block=had,
                            marlin_layout=marlin, outlier_idx=col, outlier_w=val, outlier_rowptr=rowptr)
    assert _runs_mid(hip, ops, m, dt) == mid
    y = K.batched_w4a16_gemm(x, q.packed, q.absmax, None, col, val, marlin, codebook="nf4", group_size=bs,
                             hadamard_block=had, outlier_rowptr=rowptr, bias=bias)
    _check(y, x, _dense(q, bs), had, bias, dt)


def _format_a(m, n, k, n_out, marlin, dt):
    """Operands, W_eff and activations; the codes under the outlier columns are not zero."""
    rng = np.random.default_rng(m + n)
    qc = rng.integers(0, 16, (n, k)).astype(np.uint8)
    z = rng.integers(0, 16, (n, k // 32)).astype(np.uint8)
    s = (rng.random((n, k // 32)) * 0.01 + 0.001).astype(np.float16)
    packed = O.pack_nibbles(qc, marlin)
    w = (qc.astype(np.float32) - np.repeat(z, 32, 1)) * np.repeat(s.astype(np.float32), 32, 1)
    idx = np.sort(rng.permutation(k)[:n_out]) if n_out else None
    ow = None
    if n_out:
        ow = torch.from_numpy((rng.standard_normal((n, n_out)) * 0.2).astype(np.float32)).to(DT[dt]).cuda()
        w[:, idx] = ow.float().cpu().numpy()
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").to(DT[dt])
    args = (torch.from_numpy(packed).cuda(), torch.from_numpy(s).cuda(), torch.from_numpy(z).cuda(),
            torch.from_numpy(idx).cuda() if n_out else None, ow, marlin)
    ops = K.QWeightOperands(*args[:3], k, marlin_layout=marlin, outlier_idx=args[3], outlier_w=ow)
    return args, ops, w, x


@pytest.mark.parametrize("m,n,k,n_out,marlin,dt,mid", [
    (17, 256, 96 * 2, 3, True, "float16", True), (40, 1001, 2112, 20, False, "bfloat16", True),
    (96, 3072, 3072, 30, True, "float16", False), (96, 3072, 3072, 4, True, "float16", True),
    (160, 640, 1024, 0, True, "float16", True), (300, 99, 2048, 7, True, "float16", True),
    (128, 1536, 1024, 0, False, "float16", True),    # two chunks a stage, 4 row tiles
    (255, 77, 1024, 3, True, "bfloat16", True),      # one chunk a stage, 4 + 4 row tiles
    (511, 65, 1088, 5, False, "float16", True)])
def test_mid_format_a(hip, m, n, k, n_out, marlin, dt, mid):
    args, ops, w, x = _format_a(m, n, k, n_out, marlin, dt)
    assert _runs_mid(hip, ops, m, dt) == mid
    _check(K.batched_w4a16_gemm(x, *args), x, w, 0, None, dt)


def _on_tiles(hip, ops, x, n):
    """The product on the 256-row tiles: where the mid-size family serves the call, in the largest
    workspace that does not hold its buffers."""
    m, k = x.shape
    adt = L.F16 if x.dtype == torch.float16 else L.BF16
    size = hip.spectra_w4a16_gemm_workspace(ops.ptr(), m, adt)
    if hip.spectra_w4a16_gemm_mid(ops.ptr(), m, size):
        lo = 0
        while size - lo > 1:
            at = (lo + size) // 2
            lo, size = (lo, at) if hip.spectra_w4a16_gemm_mid(ops.ptr(), m, at) else (at, size)
        size = lo
    ws = torch.empty(size, device="cuda", dtype=torch.uint8)
    out = torch.empty(m, n, device="cuda", dtype=x.dtype)
    L.check("spectra_w4a16_gemm", hip.spectra_w4a16_gemm(
        ops.ptr(), x.data_ptr(), x.stride(0), m, adt, out.data_ptr(), n, ws.data_ptr(), size,
        torch.cuda.current_stream().cuda_stream))
    return out


@pytest.mark.parametrize("m,n,k,had", [(40, 256, 4096, 128), (300, 256, 4096, 128), (33, 130, 1024, 0), (97, 512, 3072, 64)])
def test_tiles_nf4_split_k_outliers(hip, m, n, k, had):
    """The 256-row tiles on shapes that split K (8 splits of 512 at K = 4096): entries on both sides of
    every split's edge, a fully dense row, a half-dense one and an empty one."""
    g = torch.Generator(device="cuda").manual_seed(m)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    mask = torch.rand(n, k, generator=g, device="cuda") < 0.005
    mask[3, 480:560] = True
    mask[n - 2, 1000:1100] = True
    mask[77, :] = True
    mask[n - 1, ::2] = True
    mask[5] = False
    q = C.quantize_nf4(torch.where(mask, w * 10, w).half(), 64, 0, mask, True)
    ops = K.QWeightOperands(q.packed, q.absmax, None, k, codebook="nf4", hadamard_block=had, marlin_layout=True,
                            outlier_idx=q.col, outlier_w=q.val, outlier_rowptr=q.rowptr)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    y = _on_tiles(hip, ops, x, n)
    _check(y, x, _dense(q), had, None, "float16")
    assert torch.equal(_on_tiles(hip, ops, x, n), y)  # the split partials are summed in a fixed order


@pytest.mark.parametrize("m,n,k,n_out,marlin,dt", [
    (130, 8192, 1024, 10, True, "float16"), (300, 8192, 512, 3, False, "bfloat16"), (33, 256, 4096, 20, True, "float16"),
    (40, 1000, 1024, 12, False, "float16")])
def test_tiles_format_a(hip, m, n, k, n_out, marlin, dt):
    args, ops, w, x = _format_a(m, n, k, n_out, marlin, dt)
    _check(_on_tiles(hip, ops, x, n), x, w, 0, None, dt)


def test_mid_strides_alignment_and_workspace(hip):
    """The C entry with x and out rows padded and x off 16-byte alignment; a workspace that holds only
    the 256-row-tile GEMM's buffers still runs (that GEMM)."""
    m, n, k = 50, 333, 1024
    q, had = _nf4(n, k, 128, 0.01, True)
    ops = K.QWeightOperands(q.packed, q.absmax, None, k, codebook="nf4", hadamard_block=128, marlin_layout=True,
                            outlier_idx=q.col, outlier_w=q.val, outlier_rowptr=q.rowptr)
    g = torch.Generator(device="cuda").manual_seed(5)
    xb = torch.randn(m, k + 9, generator=g, device="cuda").half()
    out = torch.full((m, n + 3), 7.0, device="cuda", dtype=torch.float16)
    need = hip.spectra_w4a16_gemm_workspace(ops.ptr(), m, L.F16)
    stream = torch.cuda.current_stream().cuda_stream
    small = next(b for b in range(need, 0, -256) if not hip.spectra_w4a16_gemm_mid(ops.ptr(), m, b))
    assert small < need
    for off, size in ((1, need), (0, need), (0, small)):
        x = xb[:, off:off + k]
        ws = torch.empty(size, device="cuda", dtype=torch.uint8)
        st = hip.spectra_w4a16_gemm(ops.ptr(), x.data_ptr(), xb.stride(0), m, L.F16, out.data_ptr(), out.stride(0),
                                    ws.data_ptr(), size, stream)
        assert st == 0
        _check(out[:, :n], x, _dense(q), 128, None, "float16")
        assert bool((out[:, n:] == 7.0).all())


@pytest.mark.parametrize("had", [0, 4, 32, 128, 256, 512])
def test_mid_row_scale(hip, had):
    """Small activations beside one huge one, whose block meets only zero weights: the row scale is
    that of the rotated row (60000 / sqrt(b)), so the others, down to 2^-24 of it, keep fp16's 11
    bits.  Bound as above."""
    m, n, k = 40, 256, 1024
    g = torch.Generator(device="cuda").manual_seed(had)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    w[:, :512] = 0
    q = C.quantize_nf4(w.half(), 64, 0, None, True)
    x = (torch.rand(m, k, generator=g, device="cuda") + 0.5) * (2e-4 if had >= 128 else 8e-3)
    x[:, :512] = 0
    x[:, 3] = 60000.0
    x = x.half()
    y = K.batched_w4a16_gemm(x, q.packed, q.absmax, None, None, None, True, codebook="nf4", group_size=64,
                             hadamard_block=had)
    _check(y, x, _dense(q), had, None, "float16")


@pytest.mark.parametrize("fmt", ["nf4", "asym"])
def test_mid_infinite_activations(hip, fmt):
    """An infinite activation at an outlier gives value x inf, not NaN (the code under an outlier is
    0); one elsewhere meets codes of 0 too and gives NaN there, as the product of W_eff does."""
    m, n, k = 40, 256, 1024
    g = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    if fmt == "nf4":
        mask = torch.rand(n, k, generator=g, device="cuda") < 0.01
        mask[:, 5] = True
        mask[:, 700] = True
        q = C.quantize_nf4(torch.where(mask, w * 10, w).half(), 64, 0, mask, True)
        args = (q.packed, q.absmax, None, q.col, q.val, True)
        kw = dict(codebook="nf4", group_size=64, outlier_rowptr=q.rowptr)
    else:
        idx = torch.tensor([5, 300, 700], device="cuda")
        packed, scales, pz = C.quantize_group32(w, 32, idx)
        args = (packed, scales, C.unpack_zeros(pz, k).contiguous(), idx, (w[:, idx] * 10).half().contiguous(), True)
        kw = {}
    x = torch.randn(m, k, generator=g, device="cuda").half()
    inf = float("inf")
    x[3, 5], x[4, 5], x[4, 700], x[38, 700], x[39, 6], x[20, 9] = inf, -inf, inf, -inf, inf, float("nan")
    y = K.batched_w4a16_gemm(x, *args, **kw).cpu()
    dkw = {a: b for a, b in kw.items() if a != "group_size"}
    weff = K.w4_dequant(*args[:3], out_dtype=torch.float32, marlin_layout=True, outlier_idx=args[3],
                        outlier_w=args[4], **dkw).cpu()
    ref = (x.cpu().double()[:, None] * weff.double()[None]).sum(-1)
    special = ~ref.isfinite()
    assert special[[3, 4, 20, 38, 39]].all() and ref[3].isinf().all() and ref[38].isinf().all()
    assert torch.equal(y.double()[special].nan_to_num(7.0, 8.0, 9.0), ref[special].nan_to_num(7.0, 8.0, 9.0))
    fin = ~special
    assert ((y.double() - ref)[fin].norm() / ref[fin].norm()).item() <= 1e-3


def test_mid_long_outlier_rows(hip):
    """Rows far longer than the others (every column, every second one, one tile's worth more than the
    lanes of a row add by themselves): right, and shared among the workgroup's lanes: one row of 8192
    entries took 16 times a call with short rows only when its own lanes added it, 1.9 times now."""
    n, k = 3072, 8192
    g = torch.Generator(device="cuda").manual_seed(9)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    mask = torch.rand(n, k, generator=g, device="cuda") < 0.005
    times = []
    for dense in (False, True):
        if dense:
            mask[7], mask[40, ::2], mask[41, :200], mask[n - 1, 5:] = True, True, True, True
        q = C.quantize_nf4(torch.where(mask, w * 10, w).half(), 64, 0, mask, True)
        for m in (20, 48):
            x = torch.randn(m, k, generator=g, device="cuda").half()

            def call():
                return K.batched_w4a16_gemm(x, q.packed, q.absmax, None, q.col, q.val, True, codebook="nf4",
                                            group_size=64, outlier_rowptr=q.rowptr)
            y = call()
            _check(y, x, _dense(q), 0, None, "float16")
            assert torch.equal(call(), y)
        call()
        best = 1e9
        for _ in range(10):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                call()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        times.append(best)
    assert times[1] <= 6 * times[0], times
