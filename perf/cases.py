"""The work a model's runtime hands to this library, as measurable cases.

Three kinds of pass, each through the public entry points in the way a decoder or a prefill loop calls them:

``decode``  one transformer layer's projections for a batch of m sequences: q+k+v (one shared step), o, the gated MLP
            projection and down, as a dispatch plan captured once and replayed with one graph launch per token.
``prompt``  the same layer for a prompt of m tokens, eager calls (a prompt's length is new each time), with the
            quantized KV cache written from and read back over the prompt's positions.
``token``   what stands at both ends of a token: the quantized embedding gather and the output head with its greedy
            arg-max, on one tied table.

Layer sizes are hidden / kv / ffn: q and o are hidden x hidden, k and v hidden -> kv, gate and up hidden -> ffn, down
ffn -> hidden.  4096 / 1024 / 14336 is the layer of the benchmark at the root of the repository; 2048 / 512 / 8192 are
the sizes of its smallest configuration and of its output head.
"""
import importlib
import math

import numpy as np
import torch

mi355q = importlib.import_module("swift-mlx-lm_amd")

DTYPES = {"f16": (mi355q.F16, torch.float16), "bf16": (mi355q.BF16, torch.bfloat16), "f32": (mi355q.F32, torch.float32)}
LAYOUTS = {"planes": mi355q.LAYOUT_PLANES, "blocks": mi355q.LAYOUT_STAF_BLOCKS, "tile16": mi355q.LAYOUT_TILE16}
KV_Q8_G32 = 0x10
HEAD_DIMENSION = 128


def _decode(name, m, bits=4, group=64, layout="planes", x="bf16", hidden=4096, kv=1024, ffn=14336):
    return {"name": name, "kind": "decode", "m": m, "bits": bits, "group": group, "layout": layout, "x": x,
            "hidden": hidden, "kv": kv, "ffn": ffn}


def listed():
    return [
        # one sequence on a small model: four launches of a few microseconds, where latency is everything
        _decode("decode_small_m1", 1, hidden=2048, kv=512, ffn=8192),
        # one sequence on the benchmark's layer: the headline
        _decode("decode_m1", 1),
        # one sequence, weights left where model.staf was uploaded, f16 activations (the reference's decode type)
        _decode("decode_blocks_f16_m1", 1, layout="blocks", x="f16"),
        # one sequence on a 6-bit model in groups of 32, the format of the reference's own 6-bit benchmark
        _decode("decode_q6g32_f16_m1", 1, bits=6, group=32, x="f16"),
        # four sequences on an 8-bit model
        _decode("decode_q8g32_m4", 4, bits=8, group=32),
        # eight sequences on the records laid out for batches
        _decode("decode_tile16_m8", 8, layout="tile16"),
        # a batch that fills no power of two
        _decode("decode_m13", 13),
        # a serving batch on weights in place
        _decode("decode_blocks_f16_m32", 32, layout="blocks", x="f16"),
        # both ends of a token on a tied table
        {"name": "token_2048_65536", "kind": "token", "m": 1, "bits": 4, "group": 64, "layout": "planes", "x": "bf16",
         "hidden": 2048, "vocabulary": 65536},
        # a short prompt
        {**_decode("prompt_m128", 128), "kind": "prompt"},
        # a prompt of ragged length in fp32, the reference's prefill type
        {**_decode("prompt_f32_m517", 517, x="f32"), "kind": "prompt"},
        # a long prompt
        {**_decode("prompt_m2048", 2048), "kind": "prompt"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["decode", "prompt", "token"], [6, 4, 1])[0]
    bits, group = rng.choice([(4, 64)] * 6 + [(4, 128), (8, 32), (8, 64), (6, 32), (6, 64), (5, 64), (3, 64), (2, 64)])
    layout = rng.choice(["planes", "planes", "blocks", "tile16"])
    x = rng.choice(["bf16", "f16"])
    unit = max(64, group)
    if kind == "prompt":
        m = _log_int(rng, 97, 2048)
        if bits not in (4, 8):
            bits, group = 4, 64
        if m <= 1024 and rng.random() < 0.35:
            x = "f32"
        layout = "planes" if layout == "tile16" else layout
    elif kind == "token":
        m = _log_int(rng, 1, 64)
        layout = "planes" if layout == "tile16" else layout
    else:
        m = _log_int(rng, 1, 96)
    if layout == "tile16":
        bits, group, unit = 4, 64, 128
        m = min(m, 16)
    hidden = unit * (_log_int(rng, 1024, 4096) // unit)
    case = {"kind": kind, "m": m, "bits": bits, "group": group, "layout": layout, "x": x, "hidden": hidden}
    if kind == "token":
        case["vocabulary"] = _log_int(rng, 8192, 65536)
    else:
        case["kv"] = HEAD_DIMENSION * rng.randint(1, max(1, hidden // 512))
        case["ffn"] = unit * (rng.randint(2 * hidden, 7 * hidden // 2) // unit)
    return case


class _State:
    """What a pass needs, released with its last reference."""

    def __init__(self):
        self.weights, self.plan = [], None

    def __del__(self):
        if self.plan is not None:
            self.plan.destroy()
        for w in self.weights:
            w.destroy()


_runtime = None


def _context():
    """The program's one context and stream."""
    global _runtime
    if _runtime is None:
        ctx = mi355q.Context(0)
        _runtime = (ctx, ctx.stream_create())
    return _runtime


def _levels(generator, n, k, bits, group, spread):
    """A random matrix quantized as MLX quantizes it, some rows at a time: (first row, code words, steps, lowest values)."""
    levels = (1 << bits) - 1
    rows = max(1, (1 << 26) // k)
    for r in range(0, n, rows):
        c = min(rows, n - r)
        w = torch.randn((c, k // group, group), device="cuda", generator=generator) * spread
        low = w.amin(2, keepdim=True).half().float()
        step = ((w.amax(2, keepdim=True) - low) / levels).half().float()
        yield r, ((w - low) / step).round_().clamp_(0, levels).to(torch.int32), step, low


def _quantize(generator, n, k, bits, group, spread):
    """The matrix as a file holds it: (code words, scales and biases as fp16 bits), on the host."""
    words = torch.empty((n, k * bits // 32), dtype=torch.int32)
    scales = torch.empty((n, k // group), dtype=torch.float16)
    biases = torch.empty((n, k // group), dtype=torch.float16)
    shifts = torch.arange(0, 32, bits, device="cuda", dtype=torch.int32) if 32 % bits == 0 else None
    for r, codes, step, low in _levels(generator, n, k, bits, group, spread):
        c = codes.shape[0]
        codes = codes.view(c, k)
        if shifts is not None:
            packed = (codes.view(c, -1, 32 // bits) << shifts).sum(2, dtype=torch.int64)
        else:                                             # widths that straddle words: 32 codes fill `bits` words
            packed = torch.zeros((c, k // 32, bits), device="cuda", dtype=torch.int64)
            lanes = codes.view(c, k // 32, 32).to(torch.int64)
            for i in range(32):
                word, at = divmod(i * bits, 32)
                packed[:, :, word] |= (lanes[:, :, i] << at) & 0xFFFFFFFF
                if at + bits > 32:
                    packed[:, :, word + 1] |= lanes[:, :, i] >> (32 - at)
            packed = packed.view(c, -1)
        words[r:r + c] = packed.to(torch.int32).cpu()      # (the low 32 bits)
        scales[r:r + c], biases[r:r + c] = step.view(c, -1).half().cpu(), low.view(c, -1).half().cpu()
    return words.numpy().view(np.uint32), scales.numpy().view(np.uint16), biases.numpy().view(np.uint16)


def _matrix(generator, case, n, k, spread=0.02):
    """The same matrix as the numbers it stands for, in 64 bits."""
    w = torch.empty((n, k), device="cuda", dtype=torch.float64)
    for r, codes, step, low in _levels(generator, n, k, case["bits"], case["group"], spread):
        w[r:r + codes.shape[0]] = (codes.double() * step.double() + low.double()).view(-1, k)
    return w


def _weight(state, generator, case, n, k, spread=0.02):
    """A weight as a program loads it: packed on the host, laid out once on the device."""
    ctx, _ = _context()
    fmt = mi355q.QuantizationFormatRegistry.format_for_mlx_quantization(case["bits"], case["group"])
    words, scales, biases = _quantize(generator, n, k, case["bits"], case["group"], spread)
    state.weights.append(ctx.weight_prepare_mlx(fmt, words, scales, biases, mi355q.F16, LAYOUTS[case["layout"]]))
    return state.weights[-1]


def prepare(case, seed):
    ctx, stream = _context()
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = _State()
    s.case, s.ctx, s.stream = case, ctx, stream
    m, hidden = case["m"], case["hidden"]
    s.x_dtype, dtype = DTYPES[case["x"]]

    def rows(width):
        return torch.randn((m, width), device="cuda", generator=g).to(dtype)      # activations behind a normalisation

    def result(width, kind=dtype):
        return torch.empty((m, width), device="cuda", dtype=kind)

    if case["kind"] == "token":
        vocabulary = case["vocabulary"]
        s.table = _weight(s, g, case, vocabulary, hidden)
        s.ids = torch.randint(0, vocabulary, (m,), device="cuda", dtype=torch.int32, generator=g)
        s.embedded = result(hidden)
        s.last = torch.randn((1, hidden), device="cuda", generator=g).to(dtype)
        s.logits = torch.empty(vocabulary, device="cuda")
        s.token = torch.empty(1, device="cuda", dtype=torch.int32)
        s.outputs = [s.embedded, s.logits, s.token]
        torch.cuda.synchronize()
        return s
    kv, ffn = case["kv"], case["ffn"]
    s.q, s.k, s.v = (_weight(s, g, case, n, hidden) for n in (hidden, kv, kv))
    s.o = _weight(s, g, case, hidden, hidden)
    s.gate, s.up = _weight(s, g, case, ffn, hidden), _weight(s, g, case, ffn, hidden)
    s.down = _weight(s, g, case, hidden, ffn)
    s.x_attention, s.attended, s.x_mlp = rows(hidden), rows(hidden), rows(hidden)
    s.yq, s.yk, s.yv, s.yo = result(hidden), result(kv), result(kv), result(hidden)
    s.act, s.y = result(ffn), result(hidden)
    s.gated = result(ffn) if case["x"] == "f32" else None
    s.outputs = [s.yq, s.yk, s.yv, s.yo, s.act, s.y]
    if case["kind"] == "decode":
        s.plan = mi355q.DispatchPlan(ctx)
        t = s.x_dtype
        s.plan.add_batched_linear([s.q, s.k, s.v], s.x_attention.data_ptr(), t,
                                  [s.yq.data_ptr(), s.yk.data_ptr(), s.yv.data_ptr()], t, m)
        s.plan.add_linear(s.o, s.attended.data_ptr(), t, s.yo.data_ptr(), t, m)
        s.plan.add_gated_mlp(s.gate, s.up, s.x_mlp.data_ptr(), t, s.act.data_ptr(), t, m)
        s.plan.add_linear(s.down, s.act.data_ptr(), t, s.y.data_ptr(), t, m)
        torch.cuda.synchronize()
        s.plan.graph_build(stream)
    else:
        # the rotated keys and the values of the prompt, and one layer's caches
        s.keys, s.values = rows(kv), rows(kv)
        s.cache = mi355q.KVCacheSpecification(KV_Q8_G32, mi355q.KV_SEQUENCE_MAJOR, kv // HEAD_DIMENSION, HEAD_DIMENSION, m)
        s.k_cache, s.v_cache = (torch.zeros(s.cache.bytes_per_layer, device="cuda", dtype=torch.uint8) for _ in range(2))
        s.k_read, s.v_read = result(kv), result(kv)
        s.outputs += [s.k_cache, s.v_cache, s.k_read, s.v_read]
        torch.cuda.synchronize()
    return s


def run(s):
    ctx, stream, case = s.ctx, s.stream, s.case
    m, t = case["m"], s.x_dtype
    if case["kind"] == "decode":
        s.plan.graph_launch(stream)
    elif case["kind"] == "token":
        ctx.embedding_lookup(s.table, s.ids.data_ptr(), m, s.embedded.data_ptr(), t, stream=stream)
        ctx.lmhead_argmax(s.table, s.last.data_ptr(), t, s.logits.data_ptr(), s.token.data_ptr(), stream=stream)
    else:
        ctx.batched_qgemm([s.q, s.k, s.v], s.x_attention.data_ptr(), t,
                          [s.yq.data_ptr(), s.yk.data_ptr(), s.yv.data_ptr()], t, m, stream=stream)
        for cache, source, read in ((s.k_cache, s.keys, s.k_read), (s.v_cache, s.values, s.v_read)):
            ctx.kv_cache_write(s.cache, cache.data_ptr(), source.data_ptr(), t, 0, m, stream=stream)
            ctx.kv_cache_read(s.cache, cache.data_ptr(), read.data_ptr(), t, 0, m, stream=stream)
        ctx.qgemm(s.o, s.attended.data_ptr(), t, s.yo.data_ptr(), t, m, stream=stream)
        if t == mi355q.F32:      # the gated projection takes 16-bit rows: the shared projection and the elementwise step
            ctx.batched_qgemm([s.gate, s.up], s.x_mlp.data_ptr(), t, [s.gated.data_ptr(), s.act.data_ptr()], t, m, stream=stream)
            ctx.gated_activation(s.gated.data_ptr(), s.act.data_ptr(), s.act.data_ptr(), t, case["ffn"], m, stream=stream)
        else:
            ctx.gated_qgemm(s.gate, s.up, s.x_mlp.data_ptr(), t, s.act.data_ptr(), t, m, stream=stream)
        ctx.qgemm(s.down, s.act.data_ptr(), t, s.y.data_ptr(), t, m, stream=stream)
    return s.outputs


def exact(case, seed):
    """What run() returns, in 64 bits from the numbers the quantized weights stand for; the caches, whose bytes are a
    quantization of their own, have no such value."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    m, hidden, dtype = case["m"], case["hidden"], DTYPES[case["x"]][1]

    def rows(count, width):
        return torch.randn((count, width), device="cuda", generator=g).to(dtype).double()

    if case["kind"] == "token":
        table = _matrix(g, case, case["vocabulary"], hidden)
        ids = torch.randint(0, case["vocabulary"], (m,), device="cuda", dtype=torch.int32, generator=g)
        logits = table @ rows(1, hidden)[0]
        return [table[ids.long()], logits, logits.argmax().view(1).to(torch.int32)]
    kv, ffn = case["kv"], case["ffn"]
    shapes = [(hidden, hidden), (kv, hidden), (kv, hidden), (hidden, hidden), (ffn, hidden), (ffn, hidden), (hidden, ffn)]
    wq, wk, wv, wo, gate, up, down = (_matrix(g, case, n, k) for n, k in shapes)
    x_attention, attended, x_mlp = (rows(m, hidden) for _ in range(3))
    act = torch.nn.functional.silu(x_mlp @ gate.t()) * (x_mlp @ up.t())
    outputs = [x_attention @ wq.t(), x_attention @ wk.t(), x_attention @ wv.t(), attended @ wo.t(), act, act @ down.t()]
    return outputs + [None] * 4 if case["kind"] == "prompt" else outputs


def work(case):
    m, hidden, size = case["m"], case["hidden"], DTYPES[case["x"]][1].itemsize
    per_weight = (case["bits"] * case["group"] / 8 + 4) / case["group"]
    if case["kind"] == "token":
        vocabulary = case["vocabulary"]
        return {"bytes": vocabulary * hidden * per_weight + m * hidden * (per_weight + size) + hidden * size + vocabulary * 4,
                "flops": 2.0 * vocabulary * hidden}
    kv, ffn = case["kv"], case["ffn"]
    weights = 2 * hidden * hidden + 2 * hidden * kv + 3 * hidden * ffn
    values = m * (3 * hidden + 2 * hidden + 2 * kv + 2 * ffn + hidden)      # read and written rows, the MLP's inner rows both
    total = weights * per_weight + values * size
    if case["kind"] == "prompt":
        total += 2 * m * kv * (2 * size + 2 * (8 * 32 / 8 + 4) / 32)       # the caches: values in and out, slots both ways
    return {"bytes": total, "flops": 2.0 * m * weights}


def tolerance(case):
    # The difference between two right results is a few times what one of them is off a 64-bit evaluation of the same
    # dequantised weights, measured over layouts, widths and row counts (worst output of a layer, down behind the
    # rounded MLP rows): 4.6e-3 in bf16, 5.5e-4 in f16, 2.9e-3 for fp32 rows against weights rounded to bf16, and
    # 1.4e-6 for the fp32 logits of the head.
    if case["kind"] == "token":
        return {"rel": 1e-5}
    return {"rel": {"f16": 2e-3, "bf16": 1e-2, "f32": 1e-2}[case["x"]]}
