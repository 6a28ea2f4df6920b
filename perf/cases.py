"""The work that a user of this framework has it do, as cases to be measured.

Every family below goes through the public entry points (stark_amd.qmm,
stark_amd.decode) as a user's program calls them: arguments marshalled once
(prepare_many and its like), weights and workspaces kept, one pass per call.
Weights are N(0, 0.02) quantized by each format's rule, activations N(0, 1);
the passes of the bandwidth-bound families run over several layers of distinct
weights, as a model's pass does.
"""
from __future__ import annotations

import math

import torch

from stark_amd import decode as D
from stark_amd import qmm as Q

BF = torch.bfloat16


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # One small product of a 0.6B-sized model's MLP at decode: a call that is all launch and latency.
        dict(name="matvec_3072x1024", family="layer", m=1, bits=4, layers=1, hidden=1024, kv=0, inter=3072, layout=1),
        # Decode: one token through the seven projections of each of four 8B-sized layers, W4 group 64.
        dict(name="decode_w4", family="layer", m=1, bits=4, layers=4, hidden=4096, kv=1024, inter=12288, layout=1),
        # Decode with 8-bit weights, the other MLX width, at sizes that are no powers of two, planes row by row.
        dict(name="decode_w8_ragged", family="layer", m=1, bits=8, layers=4, hidden=2560, kv=640, inter=6912,
             layout=0),
        # Speculative verify: a draft of five tokens checked in one pass.
        dict(name="verify_w4_m5", family="layer", m=5, bits=4, layers=4, hidden=4096, kv=1024, inter=12288, layout=1),
        # A short prompt (or the ragged end of a chunked one) of 100 tokens.
        dict(name="short_prefill_w4_m100", family="layer", m=100, bits=4, layers=2, hidden=4096, kv=1024,
             inter=12288, layout=1),
        # A prefill chunk of 2048 tokens through one layer's projections.
        dict(name="prefill_w4_m2048", family="layer", m=2048, bits=4, layers=1, hidden=4096, kv=1024, inter=12288,
             layout=1),
        # Int8 activations (A8W4): the MLP of a 512-token prompt, quantized on the way in and between the products.
        dict(name="mlp_a8w4_m512", family="mlp_a8", m=512, layers=2, hidden=4096, inter=12288, act_group=128),
        # The hybrid engine's decode: GGUF Q4_K projections of four layers, f32 activations, one call a layer.
        dict(name="hybrid_q4_k", family="hybrid", m=1, kind=12, layers=4, hidden=4096, kv=1024, inter=12288),
        # A mixture-of-experts layer at decode with four sequences: bf16 router, top 8 of 128 experts.
        dict(name="moe_decode_t4", family="moe", tokens=4, layers=4, model=2048, hidden=768, experts=128, active=8),
        # The same layer over a 512-token prompt.
        dict(name="moe_prefill_t512", family="moe", tokens=512, layers=1, model=2048, hidden=768, experts=128,
             active=8),
        # Token sampling after the lm_head: four sequences, temperature, top-k and top-p over a 151936-word vocabulary.
        dict(name="sample_v151936_b4", family="sample", batch=4, vocab=151936, temperature=0.7, top_k=50, top_p=0.95),
        # A whole greedy decode step (eight layers, attention over 4096 tokens, 8-bit lm_head) as one graph replay.
        dict(name="decode_step_ctx4096", family="decode", layers=8, context=4096, capacity=4352, vocab=151936),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["layer", "layer", "layer", "layer", "mlp_a8", "hybrid", "moe", "moe", "sample", "decode"])
    if family == "layer":
        # decode (one row), verify (2-16) and prompts (17-2048) alike often
        m = rng.choice([1, rng.randint(2, 16), _log(rng, 17, 2048)])
        hidden = 64 * _log(rng, 16, 64)
        inter = 64 * _log(rng, hidden // 64, 3 * hidden // 64)
        return dict(family=family, m=m, bits=rng.choice([4, 4, 8]), layers=1 if m > 256 else rng.randint(2, 4),
                    hidden=hidden, kv=hidden // rng.choice([2, 4]) // 64 * 64, inter=inter,
                    layout=rng.choice([0, 1, 1]))
    if family == "mlp_a8":
        hidden = 128 * _log(rng, 8, 32)
        return dict(family=family, m=_log(rng, 1, 1024), layers=1, hidden=hidden,
                    inter=128 * _log(rng, hidden // 128, 3 * hidden // 128), act_group=rng.choice([64, 128]))
    if family == "hybrid":
        hidden = 256 * _log(rng, 4, 16)
        return dict(family=family, m=rng.choice([1, 1, rng.randint(2, 8)]), kind=rng.choice([8, 12]),
                    layers=rng.randint(2, 4), hidden=hidden, kv=hidden // 4,
                    inter=256 * _log(rng, hidden // 256, 3 * hidden // 256))
    if family == "moe":
        return dict(family=family, tokens=rng.choice([rng.randint(1, 16), _log(rng, 17, 1024)]), layers=1,
                    model=256 * rng.randint(4, 10), hidden=64 * rng.randint(8, 16),
                    experts=rng.choice([32, 64, 96, 128]), active=rng.choice([2, 4, 6, 8]))
    if family == "sample":
        return dict(family=family, batch=_log(rng, 1, 32), vocab=_log(rng, 32000, 152064),
                    temperature=rng.choice([0.0, 0.6, 1.0]), top_k=rng.choice([0, 20, 64]),
                    top_p=rng.choice([0.0, 0.8, 0.95]))
    context = _log(rng, 64, 4096)
    return dict(family="decode", layers=rng.randint(2, 6), context=context, capacity=context + rng.randint(1, 300),
                vocab=_log(rng, 32000, 152064))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * std


def _affine(gen, n, k, bits, layout=1, group=64):
    """N(0, 0.02) rows by the MLX affine rule: codes [n, k*bits/8] and bf16
    scale and bias planes, [k/group, n] (layout 1, n a multiple of 4) or
    [n, k/group] (layout 0)."""
    g = _randn(gen, n, k // group, group, std=0.02)
    lo, hi = g.amin(dim=2), g.amax(dim=2)
    levels = (1 << bits) - 1
    s, b = ((hi - lo) / float(levels)).to(BF), lo.to(BF)
    q = torch.round((g - b.float().unsqueeze(2)) / s.float().unsqueeze(2)).clamp_(0, levels).to(torch.uint8)
    q = q.view(n, k)
    codes = (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous() if bits == 4 else q.contiguous()
    if layout == 1:
        s, b = s.t().contiguous(), b.t().contiguous()
    return dict(n=n, k=k, bits=bits, layout=layout, group=group, codes=codes, s=s, b=b)


def _affine_f64(w):
    """The dequantized rows in 64 bits."""
    q = w["codes"]
    if w["bits"] == 4:
        q = torch.stack([q & 15, q >> 4], dim=2)
    s, b = (w["s"], w["b"]) if w["layout"] == 0 else (w["s"].t(), w["b"].t())
    g = q.reshape(w["n"], w["k"] // w["group"], w["group"]).double()
    return (g * s.double().unsqueeze(2) + b.double().unsqueeze(2)).view(w["n"], w["k"])


def _quantized(w):
    return Q.QuantizedB(codes=w["codes"], scales=w["s"], correction_data=w["b"],
                        mode=Q.MODE_U4 if w["bits"] == 4 else Q.MODE_U8, group_size=w["group"],
                        params=Q.QuantParams(Q.GROUP_OUTPUT if w["layout"] == 1 else Q.OUTPUT_GROUP, w["n"],
                                             w["k"] // w["group"]))


def _gguf(gen, n, k, kind):
    """N(0, 0.02) rows as GGUF blocks, and the pieces they decode from."""
    w = _randn(gen, n, k, std=0.02)
    if kind == 8:
        g = w.view(n, k // 32, 32)
        d = (g.abs().amax(dim=2) / 127.0).to(torch.float16)
        q = torch.round(g / d.float().unsqueeze(2)).clamp(-127, 127).to(torch.int8)
        out = torch.empty(n, k // 32, 34, dtype=torch.uint8, device="cuda")
        out[:, :, 0:2] = d.view(torch.uint8).view(n, k // 32, 2)
        out[:, :, 2:] = q.view(torch.uint8)
        return out.view(-1), (d, q)
    g = w.view(n, k // 256, 8, 32)
    m = -torch.clamp(g.amin(dim=3), max=0.0)
    sc = (g.amax(dim=3) + m) / 15.0
    d, dmin = (sc.amax(dim=2) / 63.0).to(torch.float16), (m.amax(dim=2) / 63.0).to(torch.float16)
    si = torch.round(sc / d.float().unsqueeze(2)).clamp(0, 63)
    mi = torch.round(m / dmin.float().unsqueeze(2)).clamp(0, 63)
    step = (d.float().unsqueeze(2) * si).unsqueeze(3).clamp(min=1e-12)
    q = torch.round((g + (dmin.float().unsqueeze(2) * mi).unsqueeze(3)) / step).clamp(0, 15).to(torch.uint8)
    a, b = si.to(torch.uint8), mi.to(torch.uint8)
    packed = torch.cat([(a[..., :4] & 63) | ((a[..., 4:] >> 4) << 6), (b[..., :4] & 63) | ((b[..., 4:] >> 4) << 6),
                        (a[..., 4:] & 15) | ((b[..., 4:] & 15) << 4)], dim=2)
    qv = q.view(n, k // 256, 4, 2, 32)
    out = torch.empty(n, k // 256, 144, dtype=torch.uint8, device="cuda")
    out[:, :, 0:2] = d.view(torch.uint8).view(n, k // 256, 2)
    out[:, :, 2:4] = dmin.view(torch.uint8).view(n, k // 256, 2)
    out[:, :, 4:16] = packed
    out[:, :, 16:] = (qv[:, :, :, 0] | (qv[:, :, :, 1] << 4)).reshape(n, k // 256, 128)
    return out.view(-1), (d, dmin, si, mi, q)


def _gguf_f64(parts, n, k):
    if len(parts) == 2:
        d, q = parts
        return (d.double().unsqueeze(2) * q.double()).view(n, k)
    d, dmin, si, mi, q = parts
    w = (d.double().unsqueeze(2) * si.double()).unsqueeze(3) * q.double() \
        - (dmin.double().unsqueeze(2) * mi.double()).unsqueeze(3)
    return w.view(n, k)


def _shapes(c):
    """(input, rows, columns) of the products of one layer; input names the activation read."""
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    if kv == 0:
        return [("x", i, h)]  # a lone product
    return [("x", h, h), ("x", kv, h), ("x", kv, h), ("o", h, h), ("y", i, h), ("y", i, h), ("g", h, i)]


def _activations(gen, c, dtype):
    return {name: _randn(gen, c["m"], k).to(dtype) for name, k in {n: k for n, _, k in _shapes(c)}.items()}


# ---------------------------------------------------------------- one transformer layer's products

def _layer_inputs(c, seed):
    gen = _gen(seed)
    layers = []
    for _ in range(c["layers"]):
        acts = _activations(gen, c, BF)
        layers.append([(acts[a], _affine(gen, n, k, c["bits"], c["layout"])) for a, n, k in _shapes(c)])
    return layers


def _layer_prepare(c, seed):
    kern = Q.MatmulKernel(Q.BF16, Q.BF16, Q.BF16)
    batches, outs = [], []
    for layer in _layer_inputs(c, seed):
        args = []
        for x, w in layer:
            d = torch.empty(c["m"], w["n"], dtype=BF, device="cuda")
            outs.append(d)
            args.append(Q.MatmulArguments(a=x, b=_quantized(w), d=d, m=c["m"], n=w["n"], k=w["k"]))
        batches.append(kern.prepare_many(args))
    return dict(kern=kern, batches=batches, outs=outs)


def _layer_run(s):
    for b in s["batches"]:
        s["kern"].encode_prepared(b)
    return s["outs"]


def _layer_exact(c, seed):
    return [x.double() @ _affine_f64(w).t() for layer in _layer_inputs(c, seed) for x, w in layer]


def _affine_bytes(n, k, bits):
    return n * k * bits // 8 + 2 * 2 * n * (k // 64)


def _layer_work(c):
    sh = _shapes(c)
    by = sum(_affine_bytes(n, k, c["bits"]) + 2 * c["m"] * n for _, n, k in sh)
    by += sum(2 * c["m"] * k for k in {a: k for a, _, k in sh}.values())
    return dict(bytes=c["layers"] * by, flops=c["layers"] * sum(2 * c["m"] * n * k for _, n, k in sh))


# ---------------------------------------------------------------- MLP with int8 activations

def _a8_inputs(c, seed):
    gen = _gen(seed)
    h, i = c["hidden"], c["inter"]
    layers = []
    for _ in range(c["layers"]):
        signs = [torch.randint(0, 2, (k,), generator=gen, device="cuda", dtype=torch.int32) * 2 - 1 for k in (h, i)]
        layers.append(dict(x=_randn(gen, c["m"], h).to(BF), signs=signs, up=_affine(gen, 2 * i, h, 4),
                           down=_affine(gen, h, i, 4)))
    return layers


def _a8_prepare(c, seed):
    m, h, i, ag = c["m"], c["hidden"], c["inter"], c["act_group"]
    kern = Q.MatmulKernel(Q.BF16, Q.BF16, Q.BF16)
    quant = Q.ActivationQuantization.new(ag, 64, False, Q.GROUPED_BY_NIBBLE)

    def codes(k):
        return Q.Int8SymmetricA(values=torch.empty(m, k, dtype=torch.int8, device="cuda"),
                                scales=torch.empty(m, k // ag, dtype=torch.float32, device="cuda"),
                                scale_group_size=ag, code_layout=Q.GROUPED_BY_NIBBLE)

    layers = []
    for L in _a8_inputs(c, seed):
        qx, qg = codes(h), codes(i)
        gu, y = torch.empty(m, 2 * i, dtype=BF, device="cuda"), torch.empty(m, h, dtype=BF, device="cuda")
        up = kern.prepare_many([Q.MatmulArguments(a=qx, b=_quantized(L["up"]), d=gu, m=m, n=2 * i, k=h)])
        down = kern.prepare_many([Q.MatmulArguments(a=qg, b=_quantized(L["down"]), d=y, m=m, n=h, k=i)])
        layers.append(dict(L, qx=qx, qg=qg, gu=gu, y=y, up_batch=up, down_batch=down))
    return dict(c=c, kern=kern, layers=layers, quant=Q.ActivationTransform.quantize(Q.BF16, quant),
                gated=Q.GatedActMul.quantized(Q.BF16, quant))


def _a8_run(s):
    c, outs = s["c"], []
    for L in s["layers"]:
        s["quant"].encode_quantize(L["x"], L["qx"].values, L["qx"].scales, None, L["signs"][0], c["m"], c["hidden"])
        s["kern"].encode_prepared(L["up_batch"])
        s["gated"].encode_quantized(L["gu"], L["qg"].values, L["qg"].scales, None, L["signs"][1], c["inter"], c["m"],
                                    Q.ACT_SILU)
        s["kern"].encode_prepared(L["down_batch"])
        outs += [L["gu"], L["y"]]
    return outs


def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < 32:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(32.0)


def _a8_quantize_f64(t, signs, ag):
    """What the int8 codes stand for, in 64 bits: signs, Hadamard blocks of 32, symmetric rounding per group."""
    m, k = t.shape
    r = ((t * signs.double()).view(m, k // 32, 32) @ _hadamard()).view(m, k // ag, ag)
    s = r.abs().amax(dim=2, keepdim=True) / 127.0
    return (torch.round(r / s).clamp(-127, 127) * s).view(m, k)


def _a8_exact(c, seed):
    outs, i = [], c["inter"]
    for L in _a8_inputs(c, seed):
        gu = _a8_quantize_f64(L["x"].double(), L["signs"][0], c["act_group"]) @ _affine_f64(L["up"]).t()
        v, g = gu[:, :i], gu[:, i:]
        a = _a8_quantize_f64(v * g * torch.sigmoid(g), L["signs"][1], c["act_group"])
        outs += [gu, a @ _affine_f64(L["down"]).t()]
    return outs


def _a8_work(c):
    m, h, i = c["m"], c["hidden"], c["inter"]
    by = _affine_bytes(2 * i, h, 4) + _affine_bytes(h, i, 4) + 4 * (h + i) + 2 * m * h + 2 * m * 2 * i + 2 * m * h
    return dict(bytes=c["layers"] * by, flops=c["layers"] * 2 * m * 3 * h * i)


# ---------------------------------------------------------------- hybrid engine (GGUF blocks, f32 activations)

def _hybrid_inputs(c, seed):
    gen = _gen(seed)
    layers = []
    for _ in range(c["layers"]):
        acts = _activations(gen, c, torch.float32)
        layers.append([(acts[a], n, k, _gguf(gen, n, k, c["kind"])) for a, n, k in _shapes(c)])
    return layers


def _hybrid_prepare(c, seed):
    prepared, outs = [], []
    for layer in _hybrid_inputs(c, seed):
        ops = [Q.MappedOperation(matrices=[Q.MappedMatrix(codes=blocks)] * c["m"], inputs=x.view(-1), rows=n,
                                 columns=k, format=("packed", c["kind"])) for x, n, k, (blocks, _) in layer]
        p, o = Q.mapped_prepare(ops)
        prepared.append(p)
        outs += o
    return dict(prepared=prepared, outs=outs, status=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _hybrid_run(s):
    for p in s["prepared"]:
        Q.mapped_many_async(p, s["status"])
    return s["outs"] + [s["status"]]


def _hybrid_exact(c, seed):
    return [(x.double() @ _gguf_f64(parts, n, k).t()).view(-1)
            for layer in _hybrid_inputs(c, seed) for x, n, k, (_, parts) in layer] + [None]


def _hybrid_work(c):
    sh, m = _shapes(c), c["m"]
    by = sum((n * k // 256 * 144 if c["kind"] == 12 else n * k // 32 * 34) + 4 * m * n for _, n, k in sh)
    by += sum(4 * m * k for k in {a: k for a, _, k in sh}.values())
    return dict(bytes=c["layers"] * by, flops=c["layers"] * sum(2 * m * n * k for _, n, k in sh))


# ---------------------------------------------------------------- mixture of experts

def _moe_inputs(c, seed):
    gen = _gen(seed)
    e, h, model = c["experts"], c["hidden"], c["model"]
    return [dict(x=_randn(gen, c["tokens"], model).to(BF), router=_randn(gen, e, model, std=0.02).to(BF),
                 up=_affine(gen, e * 2 * h, model, 4), down=_affine(gen, e * model, h, 4))
            for _ in range(c["layers"])]


def _moe_prepare(c, seed):
    t, e, h, model, a = c["tokens"], c["experts"], c["hidden"], c["model"], c["active"]
    kern = Q.MatmulKernel(Q.BF16, Q.BF16, Q.F32)
    ws = torch.empty(Q.routed_experts_workspace_size(t, model, h, e, a), dtype=torch.uint8, device="cuda")
    steps = []
    for L in _moe_inputs(c, seed):
        logits = torch.empty(t, e, dtype=torch.float32, device="cuda")
        out = torch.empty(t, model, dtype=BF, device="cuda")
        router = kern.prepare_many([Q.MatmulArguments(a=L["x"], b=Q.FullPrecisionB(values=L["router"]), d=logits,
                                                      m=t, n=e, k=model)])
        experts = Q.routed_experts(L["x"], logits, _quantized(L["up"]), _quantized(L["down"]), t, model, h, e, a,
                                   workspace=ws, output=out, prepare_only=True)
        steps.append((router, experts, logits, out))
    return dict(kern=kern, steps=steps)


def _moe_run(s):
    outs = []
    for router, experts, logits, out in s["steps"]:
        s["kern"].encode_prepared(router)
        Q.routed_experts_prepared(experts)
        outs += [logits, out]
    return outs


def _moe_exact(c, seed):
    e, h, model, a = c["experts"], c["hidden"], c["model"], c["active"]
    outs = []
    for L in _moe_inputs(c, seed):
        x = L["x"].double()
        logits = x @ L["router"].double().t()
        p, ids = logits.topk(a, dim=1)
        p = torch.softmax(p, dim=1)
        up, down = _affine_f64(L["up"]).view(e, 2 * h, model), _affine_f64(L["down"]).view(e, model, h)
        y = torch.zeros(c["tokens"], model, dtype=torch.float64, device="cuda")
        for k in range(e):
            rows, rank = (ids == k).nonzero(as_tuple=True)
            if rows.numel():
                vg = x[rows] @ up[k].t()
                v, g = vg[:, :h], vg[:, h:]
                y.index_add_(0, rows, p[rows, rank].unsqueeze(1) * ((v * g * torch.sigmoid(g)) @ down[k].t()))
        outs += [logits, y]
    return outs


def _moe_work(c):
    t, e, h, model, a = c["tokens"], c["experts"], c["hidden"], c["model"], c["active"]
    used = e * (1.0 - (1.0 - a / e) ** t)  # experts that some token reaches, on average
    by = used * (_affine_bytes(2 * h, model, 4) + _affine_bytes(model, h, 4)) + 2 * e * model + 4 * t * model + 4 * t * e
    return dict(bytes=int(c["layers"] * by), flops=c["layers"] * (2 * t * a * 3 * h * model + 2 * t * e * model))


# ---------------------------------------------------------------- sampling

def _sample_inputs(c, seed):
    gen = _gen(seed)
    # a language model's logits: most words far below a few likely ones
    z = _randn(gen, c["batch"], c["vocab"]) * 2.0
    for _ in range(24):
        z.scatter_add_(1, torch.randint(0, c["vocab"], (c["batch"], 1), generator=gen, device="cuda"),
                       4.0 + 8.0 * torch.rand(c["batch"], 1, generator=gen, device="cuda"))
    seeds = torch.randint(0, 1 << 62, (c["batch"],), generator=gen, device="cuda", dtype=torch.int64)
    return z.to(torch.float32).contiguous(), seeds


def _sample_prepare(c, seed):
    z, seeds = _sample_inputs(c, seed)
    method = Q.SamplingMethod(stochastic=c["temperature"] > 0, temperature=c["temperature"] or None,
                              top_k=c["top_k"] or None, top_p=c["top_p"] or None)
    return dict(c=c, z=z, seeds=seeds, method=method)


def _sample_run(s):
    return Q.unified_sampling(s["z"], Q.F32, s["c"]["vocab"], s["c"]["batch"], s["method"], s["seeds"])


def _philox(offset, word, seed):
    """Philox4x32-10 (Salmon et al. 2011) of the counters `offset`; word[i] picks the output."""
    mask = 0xFFFFFFFF
    c = [offset, torch.zeros_like(offset), torch.zeros_like(offset), torch.zeros_like(offset)]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
    return torch.stack(c).gather(0, word.unsqueeze(0)).squeeze(0)


def _sample_exact(c, seed):
    z, seeds = _sample_inputs(c, seed)
    if c["temperature"] == 0:
        return z.argmax(dim=1).to(torch.int32)
    v = c["vocab"]
    idx = torch.arange(v, device="cuda")
    offset, word = ((v + 4095) // 4096) * (idx % 1024) + idx // 4096, (idx // 1024) % 4
    out = []
    for row, seed_row in zip(z.double() / c["temperature"], seeds.tolist()):
        s, order = torch.sort(row, descending=True, stable=True)
        keep = torch.ones(v, dtype=torch.bool, device="cuda")
        if c["top_k"]:
            keep[c["top_k"]:] = False
        if c["top_p"]:
            p = torch.softmax(s, dim=0)
            keep &= (p.cumsum(0) - p) < c["top_p"]
        keep[0] = True
        bits = (_philox(offset, word, seed_row) >> 8).clamp(min=1)
        noise = -torch.log(-torch.log(bits.double() / 16777216.0))
        score = torch.full_like(row, -math.inf)
        score[order[keep]] = s[keep] + noise[order[keep]]
        out.append(score.argmax())
    return torch.stack(out).to(torch.int32)


def _sample_work(c):
    n = c["batch"] * c["vocab"]
    return dict(bytes=4 * n + 12 * c["batch"], flops=4 * n)


# ---------------------------------------------------------------- whole decode step

def _config(c):
    return D.Qwen3Config(layers=c["layers"], vocab=c["vocab"] // 32 * 32)


_PRODUCTS = ("q", "k", "v", "o", "gate", "up", "down")


def _decode_inputs(c, seed):
    cfg, gen = _config(c), _gen(seed)
    h, i, hd = cfg.hidden, cfg.intermediate, cfg.head_dim
    qd, kd = cfg.q_heads * hd, cfg.kv_heads * hd
    shapes = dict(q=(qd, h), k=(kd, h), v=(kd, h), o=(h, qd), gate=(i, h), up=(i, h), down=(h, i))

    def norm(n):
        return (1.0 + _randn(gen, n, std=0.05)).to(BF)

    layers = []
    for _ in range(cfg.layers):
        kv = [torch.zeros(cfg.kv_heads, c["capacity"], hd, dtype=BF, device="cuda") for _ in range(2)]
        for t in kv:
            t[:, :c["context"]] = _randn(gen, cfg.kv_heads, c["context"], hd).to(BF)
        layers.append(dict(attn_norm=norm(h), mlp_norm=norm(h), q_norm=norm(hd), k_norm=norm(hd), kcache=kv[0],
                           vcache=kv[1], **{w: _affine(gen, *shapes[w], 4) for w in _PRODUCTS}))
    return dict(layers=layers, embed=_randn(gen, cfg.vocab, h, std=0.02).to(BF), final_norm=norm(h),
                lm_head=_affine(gen, cfg.vocab, h, 8),
                token=torch.randint(0, cfg.vocab, (1,), generator=gen, device="cuda", dtype=torch.int32))


def _load(dst, w):
    dst["codes"].copy_(w["codes"])
    dst["scales"].copy_(w["s"].view(torch.int16))
    dst["biases"].copy_(w["b"].view(torch.int16))


def _decode_prepare(c, seed):
    inp = _decode_inputs(c, seed)
    dec = D.Qwen3Decoder(_config(c), c["capacity"])
    dec.embed.copy_(inp["embed"])
    dec.final_norm.copy_(inp["final_norm"])
    _load(dec.lm_head, inp["lm_head"])
    for dst, src in zip(dec.layers, inp["layers"]):
        for name in ("attn_norm", "mlp_norm", "q_norm", "k_norm", "kcache", "vcache"):
            dst[name].copy_(src[name])
        for name in _PRODUCTS:
            _load(dst[name], src[name])
    pos = torch.full((1,), c["context"], dtype=torch.int32, device="cuda")
    state = dict(dec=dec, token=inp["token"], pos=pos)
    del inp
    dec.token.copy_(state["token"])
    dec.pos.copy_(pos)
    dec.step()
    torch.cuda.synchronize()
    dec.capture()
    return state


def _decode_run(s):
    """The token at one position again, as after a rejected draft: set the token and the position, replay."""
    dec = s["dec"]
    dec.token.copy_(s["token"])
    dec.pos.copy_(s["pos"])
    dec.graph.replay()
    return [dec.logits] + [L[n] for L in dec.layers for n in ("kcache", "vcache")]


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.double()


def _decode_exact(c, seed):
    inp, cfg = _decode_inputs(c, seed), _config(c)
    hd, n = cfg.head_dim, c["context"] + 1
    i = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    angle = float(c["context"]) * cfg.rope_theta ** (-2.0 * i / hd)
    cs, sn = torch.cos(angle), torch.sin(angle)

    def rope(t):
        a, b = t[:, :hd // 2], t[:, hd // 2:]
        return torch.cat([a * cs - b * sn, b * cs + a * sn], dim=1)

    def mv(w, x):
        return _affine_f64(w) @ x

    x = inp["embed"][inp["token"].long()].double().view(-1)
    caches = []
    for L in inp["layers"]:
        h = _rms64(x, L["attn_norm"], cfg.eps)
        q = rope(_rms64(mv(L["q"], h).view(cfg.q_heads, hd), L["q_norm"], cfg.eps))
        k = rope(_rms64(mv(L["k"], h).view(cfg.kv_heads, hd), L["k_norm"], cfg.eps))
        kc, vc = L["kcache"].double(), L["vcache"].double()
        kc[:, c["context"]] = k
        vc[:, c["context"]] = mv(L["v"], h).view(cfg.kv_heads, hd)
        qg = q.view(cfg.kv_heads, -1, hd)
        p = torch.softmax(qg @ kc[:, :n].transpose(1, 2).contiguous() / math.sqrt(hd), dim=2)
        x = x + mv(L["o"], (p @ vc[:, :n].contiguous()).reshape(-1))
        h = _rms64(x, L["mlp_norm"], cfg.eps)
        g = mv(L["gate"], h)
        x = x + mv(L["down"], g * torch.sigmoid(g) * mv(L["up"], h))
        caches += [kc, vc]
    return [mv(inp["lm_head"], _rms64(x, inp["final_norm"], cfg.eps))] + caches


def _decode_work(c):
    cfg = _config(c)
    h, i, hd = cfg.hidden, cfg.intermediate, cfg.head_dim
    qd, kd = cfg.q_heads * hd, cfg.kv_heads * hd
    shapes = [(qd, h), (kd, h), (kd, h), (h, qd), (i, h), (i, h), (h, i)]
    kv = 2 * 2 * kd * (c["context"] + 2)
    layer = sum(_affine_bytes(n, k, 4) for n, k in shapes) + kv + 2 * 2 * h + 2 * 2 * hd
    by = cfg.layers * layer + _affine_bytes(cfg.vocab, h, 8) + 4 * cfg.vocab + 2 * 2 * h
    fl = cfg.layers * (sum(2 * n * k for n, k in shapes) + 4 * qd * (c["context"] + 1)) + 2 * cfg.vocab * h
    return dict(bytes=by, flops=fl)


# ---------------------------------------------------------------- the interface

_FAMILIES = {
    "layer": (_layer_prepare, _layer_run, _layer_exact, _layer_work),
    "mlp_a8": (_a8_prepare, _a8_run, _a8_exact, _a8_work),
    "hybrid": (_hybrid_prepare, _hybrid_run, _hybrid_exact, _hybrid_work),
    "moe": (_moe_prepare, _moe_run, _moe_exact, _moe_work),
    "sample": (_sample_prepare, _sample_run, _sample_exact, _sample_work),
    "decode": (_decode_prepare, _decode_run, _decode_exact, _decode_work),
}


def prepare(case, seed):
    state = _FAMILIES[case["family"]][0](case, seed)
    return dict(family=case["family"], state=state)


def run(state):
    return _FAMILIES[state["family"]][1](state["state"])


def exact(case, seed):
    return _FAMILIES[case["family"]][2](case, seed)


def work(case):
    return _FAMILIES[case["family"]][3](case)


def tolerance(case):
    """About four times the distance from exact() (in brackets)."""
    return dict(
        # bf16 outputs of 32-bit sums (1.7e-3); from 17 rows on the weights are rounded to bf16 too (2.3e-3)
        layer={"rel": 7e-3 if case.get("m", 0) <= 16 else 9e-3},
        # two products and an int8 requantization of bf16 values between them (7.9e-3)
        mlp_a8={"rel": 3e-2},
        # f32 activations as bf16 pairs, 32-bit sums, f32 outputs (2.9e-6)
        hybrid={"rel": 1.2e-5},
        # bf16 at each of the stages of an expert and in the sum over the ranks (4.4e-3)
        moe={"rel": 1.7e-2},
        # tokens
        sample="exact",
        # bf16 between all stages of the layers (2.3e-2)
        decode={"rel": 9e-2},
    )[case["family"]]
