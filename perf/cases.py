"""The work that programs on this framework spend their time in, as measurable cases.

Four kinds of case, each through public entry points:

* ``linear``    ``SpectraFusedLinear`` modules: M = 1 decode, 2..16 rows of a verify batch, a few
                dozen to a few hundred rows of batched serving and chunked prompts, 2048-row prefill;
                both weight formats, both activation types.  Up to 16 rows the calls of a pass are
                captured in one HIP graph over a model's layers, as a decode loop runs them.
* ``attend``    decode attention over the fp16 or the 4-bit KV cache, one call per layer in a graph.
* ``prefill`` / ``decode``   ``SpectraDecoder`` whole calls: a prompt, and one token by graph replay.
* ``quantize``  the compressor's side: a checkpoint tensor to packed weights, scales and outliers.

Sizes are the layer shapes of the 3B-shaped decoder (hidden 3072, 24 query / 8 KV heads of 128,
intermediate 8192, vocabulary 128256), the 4096 / 14336 prefill shapes of ``bench.py``, and
generic ones.
"""
import math

import torch

from spectra_amd import compressor as C
from spectra_amd import kernels as K
from spectra_amd.engine import DecoderConfig, SpectraDecoder, SpectraFusedLinear

_DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _linear(name=None, fmt="nf4", m=1, k=4096, n=4096, dtype="fp16", had=128, ratio=0.005, bias=False,
            marlin=True, layers=1, graph=False):
    c = dict(kind="linear", fmt=fmt, m=m, k=k, n=n, dtype=dtype, had=had, ratio=ratio, bias=bias, marlin=marlin,
             layers=layers, graph=graph)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest call of all: one eager module call on one token, no rotation, no outliers
        _linear("gemv_eager_4096", m=1, k=4096, n=4096, had=0, ratio=0.0),
        # one token through the down projections of a 28-layer decoder: the format's full path
        _linear("gemv_down", m=1, k=8192, n=3072, layers=28, graph=True),
        # eight drafted tokens verified at once, the widest layer (bench.py's verify batch)
        _linear("verify_gate_up_m8", m=8, k=3072, n=16384, layers=28, graph=True),
        # batched serving of 48 sequences: the fused QKV projection, with a bias, in bf16
        _linear("serve_qkv_m48", m=48, k=3072, n=5120, dtype="bf16", bias=True),
        # a chunk of a prompt, ragged row count: the down projection
        _linear("chunk_down_m200", m=200, k=8192, n=3072),
        # a long prompt: bench.py's first prefill GEMM at full size
        _linear("prefill_up_m2048", m=2048, k=4096, n=14336, dtype="bf16"),
        # Format A (the reference's own format): one token, dense outlier columns
        _linear("format_a_gemv", fmt="asym", m=1, k=3072, n=8192, had=0, ratio=0.01, dtype="bf16", layers=28,
                graph=True),
        # Format A: a short prompt, ragged, plain nibble order is the container's Marlin order here
        _linear("format_a_prompt_m130", fmt="asym", m=130, k=3072, n=8192, had=0, ratio=0.01),
        # long-context decode attention, 6001 of 8192 positions filled
        dict(name="attend_8k", kind="attend", heads=24, kv_heads=8, head_dim=128, max_seq=8192, pos=6001, kv_bits=16,
             window=128, layers=28),
        # a prompt of ragged length through four decoder layers and the lm_head
        dict(name="decoder_prefill_777", kind="prefill", layers=4, prompt=777, max_seq=1024),
        # one token of batch-1 generation: eight layers, the tied lm_head and the greedy pick
        dict(name="decoder_token", kind="decode", layers=8, prompt=640, max_seq=1024),
        # compressing one projection of a checkpoint to the NF4 container format
        dict(name="quantize_nf4_down", kind="quantize", fmt="nf4", n=3072, k=8192, dtype="bf16", had=128, ratio=0.005),
    ]


_LARGEST = 2048 * 4096 * 14336


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "attend", "prefill", "decode", "quantize"], [10, 2, 1.5, 1, 1.5])[0]
    if kind == "linear":
        fmt = rng.choices(["nf4", "asym"], [3, 1])[0]
        m = _log(rng, 1, 2048)
        k = rng.choice([2048, 3072, 4096, 8192, 128 * _log(rng, 8, 112)])
        n = rng.choice([3072, 5120, 16384, _log(rng, 256, 16384)])
        m = max(1, min(m, _LARGEST // (k * n)))
        small = m <= 16
        return _linear(fmt=fmt, m=m, k=k, n=n, dtype=rng.choice(["fp16", "bf16"]),
                       had=rng.choice([0, 128, 128]) if fmt == "nf4" else 0,
                       ratio=rng.choice([0.0, 0.005, 0.01]), bias=rng.random() < 0.3, marlin=rng.random() < 0.8,
                       layers=rng.randint(8, 28) if small else 1, graph=small)
    if kind == "attend":
        max_seq = _log(rng, 512, 16384)
        heads, kv = rng.choice([(24, 8), (32, 8), (32, 4), (16, 16)])
        return dict(kind="attend", heads=heads, kv_heads=kv, head_dim=rng.choice([64, 128, 128]), max_seq=max_seq,
                    pos=rng.randint(1, max_seq - 1), kv_bits=rng.choice([16, 4]), window=128, layers=rng.randint(4, 28))
    if kind == "prefill":
        return dict(kind="prefill", layers=rng.randint(1, 4), prompt=_log(rng, 16, 2040), max_seq=2048)
    if kind == "decode":
        return dict(kind="decode", layers=rng.randint(2, 8), prompt=_log(rng, 16, 2000), max_seq=2048)
    fmt = rng.choice(["nf4", "asym"])
    return dict(kind="quantize", fmt=fmt, n=_log(rng, 256, 16384), k=rng.choice([2048, 3072, 4096, 8192]),
                dtype=rng.choice(["fp16", "bf16", "fp32"]), had=rng.choice([0, 128]) if fmt == "nf4" else 0,
                ratio=rng.choice([0.0, 0.005, 0.01]))


# -- inputs --------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1 + int(seed))


def _capture(fn):
    """``fn`` once eagerly, then captured; returns the graph and the outputs it writes."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _weight(case, gen):
    """Quantized operands of one layer, W ~ N(0, 0.02) with outliers ~ N(0, 0.2)."""
    n, k, ratio = case["n"], case["k"], case["ratio"]
    w = torch.randn(n, k, generator=gen, device="cuda").mul_(0.02)
    if case["fmt"] == "nf4":
        mask = torch.rand(n, k, generator=gen, device="cuda") < ratio if ratio else None
        if mask is not None:
            w = torch.where(mask, w * 10.0, w)
        return C.quantize_nf4(w.half(), 64, 0, mask, case.get("marlin", True))
    idx = ow = None
    if ratio:
        idx = torch.randperm(k, generator=gen, device="cuda")[:max(1, int(k * ratio))].sort().values
        w[:, idx] *= 10.0
        ow = w[:, idx].to(_DT[case["dtype"]]).contiguous()
    packed, scales, pz = C.quantize_group32(w, 32, idx)
    if not case.get("marlin", True):  # the same codes in the plain order: byte j = q[2j] | q[2j+1] << 4
        q = _codes(packed, True)
        packed = (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8)
    return packed, scales, C.unpack_zeros(pz, k).contiguous(), idx, ow


def _prepare_linear(case, seed):
    gen = _gen(seed)
    dt = _DT[case["dtype"]]
    mods, xs, ws = [], [], []
    for _ in range(case["layers"]):
        w = _weight(case, gen)
        nf4 = case["fmt"] == "nf4"
        lin = SpectraFusedLinear(case["k"], case["n"], 64 if nf4 else 32, marlin_layout=case["marlin"],
                                 codebook=case["fmt"], hadamard_block=case["had"])
        bias = torch.randn(case["n"], generator=gen, device="cuda").to(dt) if case["bias"] else None
        if nf4:
            col, val = w.outliers()
            lin.set_weights(w.packed, w.absmax, None, bias, col, val, case["marlin"],
                            outlier_rowptr=w.rowptr if col is not None else None)
        else:
            lin.set_weights(w[0], w[1], w[2], bias, w[3], w[4], case["marlin"])
        mods.append(lin)
        ws.append((w, bias))
        xs.append(torch.randn(case["m"], case["k"], generator=gen, device="cuda").to(dt))
    state = dict(kind="linear", mods=mods, xs=xs, ws=ws)
    if case["graph"]:
        with torch.no_grad():
            state["graph"], state["out"] = _capture(lambda: [f(x) for f, x in zip(mods, xs)])
    return state


def _prepare_attend(case, seed):
    gen = _gen(seed)
    h, kv, d, n = case["heads"], case["kv_heads"], case["head_dim"], case["max_seq"]

    def f16(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float16)

    inv = 1.0 / (500000.0 ** (torch.arange(0, d, 2, dtype=torch.float32, device="cuda") / d))
    ang = torch.arange(n, dtype=torch.float32, device="cuda")[:, None] * inv
    pos = torch.tensor([case["pos"]], dtype=torch.int64, device="cuda")
    ws = torch.zeros(K.attend_workspace_bytes(h, d, n), dtype=torch.uint8, device="cuda")
    cos, sin = ang.cos(), ang.sin()
    # the caches of all layers in one tensor, as the decoder keeps them: fp16 rows of every
    # position, or of the last ``window`` beside 4-bit codes of all
    rows = n if case["kv_bits"] == 16 else min(case["window"], n)
    kcs, vcs = (torch.zeros(case["layers"], kv, rows, d, device="cuda", dtype=torch.float16) for _ in range(2))
    layers = []
    for i in range(case["layers"]):
        kc, vc = f16(kv, n, d), f16(kv, n, d)
        lay = dict(qkv=f16((h + 2 * kv) * d), k=kcs[i], v=vcs[i])
        if case["kv_bits"] == 16:
            lay["k"].copy_(kc)
            lay["v"].copy_(vc)
        else:
            at = torch.arange(max(0, case["pos"] - rows + 1), case["pos"], device="cuda")
            lay["k"][:, at % rows], lay["v"][:, at % rows] = kc[:, at], vc[:, at]
            lay.update(k4=K.kv4_quantize(kc), v4=K.kv4_quantize(vc))
        layers.append(lay)

    def step():
        outs = []
        for t in layers:
            if case["kv_bits"] == 16:
                outs.append(K.attend_decode(t["qkv"], pos, cos, sin, h, kv, t["k"], t["v"], ws))
            else:
                outs.append(K.attend_decode_q4(t["qkv"], pos, cos, sin, h, kv, t["k"], t["v"], t["k4"], t["v4"], ws))
        return outs

    graph, out = _capture(step)
    # the appended rows are state that a pass writes
    out = dict(out=out, k_row=kcs[:, :, case["pos"] % rows], v_row=vcs[:, :, case["pos"] % rows])
    return dict(kind="attend", graph=graph, out=out, layers=layers, pos=pos, cos=cos, sin=sin, ws=ws)


def _decoder(case, seed):
    return SpectraDecoder(DecoderConfig(layers=case["layers"], max_seq=case["max_seq"], seed=int(seed)))


def _prompt(dec, case, seed):
    return torch.randint(0, dec.cfg.vocab, (case["prompt"],), generator=_gen(seed), device="cuda")


def _prepare_prefill(case, seed):
    dec = _decoder(case, seed)
    return dict(kind="prefill", dec=dec, prompt=_prompt(dec, case, seed))


def _prepare_decode(case, seed):
    dec = _decoder(case, seed)
    dec.prefill(_prompt(dec, case, seed))
    dec.capture_decode()
    return dict(kind="decode", dec=dec, tok=dec.cur_id.clone(), pos=dec.cur_pos.clone(), at=case["prompt"])


def _prepare_quantize(case, seed):
    gen = _gen(seed)
    n, k = case["n"], case["k"]
    w = torch.randn(n, k, generator=gen, device="cuda").mul_(0.02)
    s = dict(kind="quantize", fmt=case["fmt"], had=case["had"], ratio=case["ratio"])
    if case["fmt"] == "nf4":
        mask = None
        if case["ratio"]:  # a fixed share of the tensor, anywhere in it
            mask = torch.zeros(n * k, dtype=torch.bool, device="cuda")
            mask[torch.randperm(n * k, generator=gen, device="cuda")[:int(n * k * case["ratio"])]] = True
            mask = mask.view(n, k)
            w = torch.where(mask, w * 10.0, w)
        s["mask"] = mask
    else:  # columns of unequal size, the largest kept as outliers
        w *= torch.exp(0.5 * torch.randn(k, generator=gen, device="cuda"))
    s["w"] = w.to(_DT[case["dtype"]])
    return s


def prepare(case, seed):
    return {"linear": _prepare_linear, "attend": _prepare_attend, "prefill": _prepare_prefill,
            "decode": _prepare_decode, "quantize": _prepare_quantize}[case["kind"]](case, seed)


# -- one pass ------------------------------------------------------------------------------------
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear" and "graph" not in state:
        return [f(x) for f, x in zip(state["mods"], state["xs"])]
    if kind in ("linear", "attend"):
        state["graph"].replay()
        return state["out"]
    if kind == "prefill":
        dec, t = state["dec"], state["prompt"].numel()
        logits = dec.prefill(state["prompt"])
        return dict(logits=logits, k=dec.k_cache[:, :, :t], v=dec.v_cache[:, :, :t])
    if kind == "decode":
        dec = state["dec"]
        dec.cur_id.copy_(state["tok"])
        dec.cur_pos.copy_(state["pos"])
        dec.decode(1)
        at = state["at"]
        return dict(logits=dec.graph_logits, k=dec.k_cache[:, :, at:at + 1], v=dec.v_cache[:, :, at:at + 1])
    if state["fmt"] == "nf4":
        q = C.quantize_nf4(state["w"], 64, state["had"], state["mask"], True)
        return [q.packed, q.absmax, q.rowptr, q.col, q.val]
    idx = None
    if state["ratio"]:
        idx, _, _ = C.select_outlier_columns(state["w"], None, state["ratio"], False)
    packed, scales, zeros = C.quantize_group32(state["w"], 32, idx)
    return [packed, scales, zeros] + ([idx, state["w"][:, idx.long()]] if idx is not None else [])


# -- what a pass cannot do without ---------------------------------------------------------------
def _weight_bytes(fmt, n, k, ratio):
    if fmt == "nf4":
        nnz = int(n * k * ratio)
        return n * k / 2 + n * (k // 64) * 2 + (nnz * 6 + (n + 1) * 4 if nnz else 0)
    cols = max(1, int(k * ratio)) if ratio else 0
    return n * k / 2 + n * (k // 32) * 3 + cols * (8 + 2 * n)


def _decoder_linears(layers):
    per = [(5120, 3072), (3072, 3072), (16384, 3072), (3072, 8192)]
    return per * layers, (128256, 3072)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n, layers = case["m"], case["k"], case["n"], case["layers"]
        b = _weight_bytes(case["fmt"], n, k, case["ratio"]) + 2 * m * (n + k) + (2 * n if case["bias"] else 0)
        return {"bytes": layers * b, "flops": layers * 2 * m * n * k}
    if kind == "attend":
        h, kv, d, p, w = case["heads"], case["kv_heads"], case["head_dim"], case["pos"] + 1, case["window"]
        row = 2 * 2 * kv * d  # k and v of one position in fp16
        cache = p * row if case["kv_bits"] == 16 else min(p, w) * row + max(0, p - w) * 2 * kv * (d // 2 + 3 * d // 32)
        return {"bytes": case["layers"] * (cache + 2 * (2 * h + 2 * kv) * d),
                "flops": case["layers"] * 4 * h * d * p}
    if kind in ("prefill", "decode"):
        lins, head = _decoder_linears(case["layers"])
        t = case["prompt"] if kind == "prefill" else 1
        ctx = case["prompt"] if kind == "prefill" else case["prompt"] + 1
        wb = sum(_weight_bytes("nf4", n, k, 0.005) for n, k in lins + [head])
        flops = 2 * t * sum(n * k for n, k in lins) + 2 * head[0] * head[1]
        pairs = ctx * (ctx + 1) / 2 if kind == "prefill" else ctx
        flops += case["layers"] * 4 * 3072 * pairs
        return {"bytes": wb + case["layers"] * ctx * 2 * 2 * 1024 + 2 * 128256, "flops": flops}
    n, k = case["n"], case["k"]
    es = 4 if case["dtype"] == "fp32" else 2
    out = _weight_bytes(case["fmt"], n, k, case["ratio"])
    mask = n * k if case["fmt"] == "nf4" and case["ratio"] else 0
    return {"bytes": n * k * es + mask + out,
            "flops": n * k * (2 + (math.log2(case["had"]) if case["had"] else 0))}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "linear":
        # fp16 / bf16 rounding of the result and of the rotated operands
        return {"rel": 1.5e-3 if case["dtype"] == "fp16" else 8e-3, "max": 0.05}
    if kind == "attend":
        return {"rel": 2e-3, "max": 0.05}
    return {"rel": 1.5e-2, "max": 0.1}  # fp16 activations rounded in every layer


# -- the same in 64 bits -------------------------------------------------------------------------
# the 16 levels of NormalFloat-4 (Dettmers et al., "QLoRA", 2023, appendix E)
_NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
        -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
        0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def _codes(packed, marlin):
    lo, hi = (packed & 15).long(), (packed >> 4).long()
    if marlin:
        n = packed.shape[0]
        return torch.cat([lo.view(n, -1, 16), hi.view(n, -1, 16)], -1).reshape(n, -1)
    return torch.stack([lo, hi], -1).reshape(packed.shape[0], -1)


def _nf4_dense(q):
    lev = torch.tensor(_NF4, dtype=torch.float64, device="cuda")
    w = lev[_codes(q.packed, q.marlin_layout)] * q.absmax.double().repeat_interleave(q.blocksize, 1)
    if q.col.numel():
        rows = torch.repeat_interleave(torch.arange(q.n, device="cuda"), torch.diff(q.rowptr.long()))
        w[rows, q.col.long()] = q.val.double()
    return w


def _rotate(x, block):
    if not block:
        return x
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < block:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((x.reshape(-1, block) @ h) / math.sqrt(block)).reshape(x.shape)


def _exact_linear(case, s):
    outs = []
    for x, (w, bias) in zip(s["xs"], s["ws"]):
        if case["fmt"] == "nf4":
            dense = _nf4_dense(w)
        else:
            dense = (_codes(w[0], case["marlin"]).double() - w[2].double().repeat_interleave(32, 1)) * \
                w[1].double().repeat_interleave(32, 1)
            if w[3] is not None:
                dense[:, w[3]] = w[4].double()
        y = _rotate(x.double(), case["had"]) @ dense.t()
        outs.append(y + bias.double() if bias is not None else y)
    return outs


def _rope(x, pos, base=500000.0):
    """x [T, heads, d], rotated in pairs (i, i + d/2)."""
    d = x.shape[-1]
    ang = pos.double()[:, None] / base ** (torch.arange(0, d, 2, device="cuda").double() / d)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _softmax_v(q, k, v, mask=None):
    """q [heads, T, d], k and v [kv, L, d]."""
    g = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(g, 0), v.repeat_interleave(g, 0)
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v)


def _exact_attend(case, s):
    h, kv, d, p, n = case["heads"], case["kv_heads"], case["head_dim"], case["pos"], case["max_seq"]
    outs = dict(out=[], k_row=[], v_row=[])
    pos = torch.tensor([p], device="cuda")
    for t in s["layers"]:
        row = t["qkv"].double().view(1, h + 2 * kv, d)
        q, kn, vn = _rope(row[:, :h], pos), _rope(row[:, h:h + kv], pos)[0], row[0, h + kv:]
        if case["kv_bits"] == 16:
            k, v = t["k"].double()[:, :p + 1].clone(), t["v"].double()[:, :p + 1].clone()
        else:
            w = t["k"].shape[1]
            k, v = [(_codes(c.reshape(kv * n, d // 2), False).double() - z.reshape(kv * n, -1).double()
                     .repeat_interleave(32, 1)).mul(sc.reshape(kv * n, -1).double().repeat_interleave(32, 1))
                    .view(kv, n, d)[:, :p + 1].clone() for c, sc, z in (t["k4"], t["v4"])]
            at = torch.arange(max(0, p + 1 - w), p, device="cuda")
            k[:, at], v[:, at] = t["k"].double()[:, at % w], t["v"].double()[:, at % w]
        k[:, p], v[:, p] = kn, vn
        outs["out"].append(_softmax_v(q[0][:, None], k, v)[:, 0])
        outs["k_row"].append(kn)
        outs["v_row"].append(vn)
    outs["k_row"], outs["v_row"] = torch.stack(outs["k_row"]), torch.stack(outs["v_row"])
    return outs


def _exact_decoder(case, s):
    dec = s["dec"]
    c = dec.cfg
    h_, kv, d = c.heads, c.kv_heads, c.head_dim
    if case["kind"] == "prefill":
        ids, first = s["prompt"], 0
    else:
        ids, first = s["tok"], s["at"]
    t = ids.numel()
    pos = torch.arange(first, first + t, device="cuda")
    mask = torch.arange(first + t, device="cuda")[None, :] <= pos[:, None]
    emb = _nf4_dense(dec.embed_q)
    x = emb[ids]
    ks, vs = [], []

    def norm(v, w):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + c.rms_eps) * w.double()

    def lin(q, v):
        return _rotate(v, q.hadamard_block) @ _nf4_dense(q).t()

    for i, (wqkv, wo, wgu, wd) in enumerate(dec.layers_q):
        qkv = lin(wqkv, norm(x, dec.norm_w[2 * i])).view(t, h_ + 2 * kv, d)
        q, k, v = _rope(qkv[:, :h_], pos), _rope(qkv[:, h_:h_ + kv], pos).transpose(0, 1), qkv[:, h_ + kv:].transpose(0, 1)
        ks.append(k)
        vs.append(v)
        if first:
            k = torch.cat([dec.k_cache[i, :, :first].double(), k], 1)
            v = torch.cat([dec.v_cache[i, :, :first].double(), v], 1)
        a = _softmax_v(q.transpose(0, 1).contiguous(), k.contiguous(), v.contiguous(), mask)
        x = x + lin(wo, a.transpose(0, 1).reshape(t, c.hidden))
        g, u = lin(wgu, norm(x, dec.norm_w[2 * i + 1])).chunk(2, -1)
        x = x + lin(wd, torch.nn.functional.silu(g) * u)
    return dict(logits=norm(x[-1:], dec.norm_w[-1]) @ emb.t(), k=torch.stack(ks), v=torch.stack(vs))


def _exact_quantize(case, s):
    if case["fmt"] != "nf4":
        return None
    w = _rotate(s["w"].double(), case["had"])
    val = w.masked_select(s["mask"]) if s["mask"] is not None else None
    if s["mask"] is not None:
        w = w.masked_fill(s["mask"], 0.0)
    absmax = w.reshape(case["n"], -1, 64).abs().amax(-1)
    return [None, absmax, None, None, val]


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "linear":
        return _exact_linear(case, s)
    if case["kind"] == "attend":
        return _exact_attend(case, s)
    if case["kind"] in ("prefill", "decode"):
        return _exact_decoder(case, s)
    return _exact_quantize(case, s)
