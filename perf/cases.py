"""The work that a user of this framework has it do, as cases that can be timed and compared.

One step of a continuous-batching server is: append the step's K/V to the paged pool and attend
over it (single-token decodes, chunked-prefill slices, or both packed together), weight-only INT8
and INT4 linears on the step's tokens, and the whole decoder around them. The listed cases are one
of each kind, from the smallest call to the largest; ``draw`` gives others of the same ranges:

* attention (``kernels.paged_attention_append`` with the step's plan): fp16, bf16 and fp32 pools of
  16-token blocks, head_dim 64 or 128, multi-head and grouped-query heads, 1 to 64 decodes over
  contexts of 16 to 8,192 tokens, prefill slices of 9 to 512 tokens behind cached prefixes of up
  to 6,656, and batches that hold both;
* linears (``QuantLinear.forward``): INT8 per output channel and INT4 in groups of 128, fp16
  activations of 1 to 2,048 tokens, 1,152 to 8,192 inputs, 1,024 to 16,384 outputs;
* decoder (``EdgeRagDecoder.greedy``): blocks of the 1.7B shape, a decode batch replayed from a
  HIP graph as the executor does, or an eager step with a prefill slice beside decodes.
"""

import dataclasses
import math
import random

import numpy as np
import torch

from edgerag_amd import kernels
from edgerag_amd.core.linear import QuantLinear
from edgerag_amd.core.model import EdgeRagDecoder, StepInputs
from edgerag_amd.core.quant import QuantConfig
from edgerag_amd.core.spec import SMOLLM2_1_7B

BLOCK = 16
LAYERS = 4  # blocks of a decoder case: every block is alike
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
DEVICE = "cuda"


# --- the cases ---------------------------------------------------------------------------------


def _attention(dtype, heads, kv_heads, head_dim, decodes=0, ctx=(0, 0), slices=0, chunk=0,
               prefix=(0, 0), spread=0, **more):
    """``decodes`` single-token requests with contexts drawn from ``ctx``, and ``slices`` of
    ``chunk`` tokens behind prefixes spread over ``prefix``."""
    return dict(op="attention", dtype=dtype, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                decodes=decodes, ctx_lo=ctx[0], ctx_hi=ctx[1], slices=slices, chunk=chunk,
                prefix_lo=prefix[0], prefix_hi=prefix[1], spread=spread, **more)


def _linear(bits, m, k, n, **more):
    return dict(op="linear", bits=bits, m=m, k=k, n=n, **more)


def _decoder(graph, decodes, ctx, slices=0, chunk=0, prefix=(0, 0), spread=0, **more):
    return dict(op="decoder", graph=graph, decodes=decodes, ctx_lo=ctx[0], ctx_hi=ctx[1],
                slices=slices, chunk=chunk, prefix_lo=prefix[0], prefix_hi=prefix[1],
                spread=spread, **more)


def listed():
    return [
        # One user's next token: the latency of a single sequence in the middle of a chat.
        _attention("fp16", 32, 32, 64, 1, (2048, 2048), name="decode_one"),
        # A loaded server's decode step: 32 requests, ragged contexts (the benchmark's batch).
        _attention("fp16", 32, 32, 64, 32, (256, 7472), spread=2, name="decode_batch"),
        # The same for a grouped-query model in bf16 with heads of 128.
        _attention("bf16", 32, 8, 128, 48, (256, 8192), spread=5, name="decode_gqa_bf16"),
        # Continuous batching: three 512-token slices of long prompts beside 24 decodes.
        _attention("fp16", 32, 32, 64, 24, (512, 7472), 3, 512, (0, 6656), 3, name="mixed"),
        # Two slices of long prompts and a few decodes for the grouped-query bf16 model.
        _attention("bf16", 32, 8, 128, 7, (256, 4096), 2, 512, (1536, 3584), 4,
                   name="prefill_gqa_bf16"),
        # Short prompts of odd length at full precision, 9 query heads over 3 (how results are
        # checked against a reference), with a few decodes.
        _attention("fp32", 9, 3, 64, 4, (37, 511), 2, 300, (0, 211), 1, name="short_fp32"),
        # The smallest linear calls: one token through an INT8 up projection, ...
        _linear(8, 1, 2048, 8192, name="linear_int8_one"),
        # ... and eight through an INT4 layer whose width is no power of two.
        _linear(4, 8, 1152, 4608, name="linear_int4_batch"),
        # A prefill slice with the decode tokens packed behind it, through a down projection.
        _linear(8, 544, 8192, 2048, name="linear_int8_slice"),
        # Four slices at once through the fused gate/up projection: the largest linear.
        _linear(8, 2048, 2048, 16384, name="linear_int8_long"),
        # A whole decode iteration (4 blocks and the head) of 8 requests, replayed from a graph.
        _decoder(True, 8, (256, 3000), spread=6, name="decoder_decode"),
        # A whole prefill iteration: one 512-token slice beside 7 decodes, launched eagerly.
        _decoder(False, 7, (256, 3000), 1, 512, (2560, 2560), 7, name="decoder_prefill"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.30:
        bits = rng.choice((8, 8, 4))
        k = rng.choice((2048, 4096, 8192)) if bits == 8 else rng.choice((1152, 2304, 4608))
        n = rng.choice((1024, 2048, 4096, 6144, 8192, 16384)) if bits == 8 else \
            rng.choice((1152, 3456, 4608))
        m = _log(rng, 1, 2048)
        while m * k * n > 2048 * 2048 * 16384:
            m = _log(rng, 1, 2048)
        return _linear(bits, m, k, n)
    if kind < 0.40:
        lo = _log(rng, 16, 1024)
        if rng.random() < 0.5:
            return _decoder(True, rng.randint(1, 24), (lo, lo + _log(rng, 1, 2048)),
                            spread=rng.randrange(1 << 20))
        prefix = 16 * rng.randint(0, 160)
        return _decoder(False, rng.randint(0, 7), (lo, lo + _log(rng, 1, 2048)), 1,
                        _log(rng, 33, 512), (prefix, prefix), rng.randrange(1 << 20))
    dtype = rng.choice(("fp16", "fp16", "bf16", "bf16", "fp32"))
    heads, kv_heads, head_dim = rng.choice((
        (32, 32, 64), (9, 3, 64), (15, 5, 64), (32, 8, 64), (32, 8, 128), (16, 16, 128),
        (24, 8, 128)))
    decodes = slices = chunk = 0
    ctx = prefix = (0, 0)
    what = rng.choice(("decode", "prefill", "mixed"))
    token = 2 * kv_heads * head_dim * (4 if dtype == "fp32" else 2)
    if what != "prefill":
        decodes = _log(rng, 1, 48)
        lo = _log(rng, 16, 4096)
        hi = min(8192, lo + _log(rng, 1, 4096))
        # The reads of a step stay below those of the listed decode batches.
        while decodes > 1 and decodes * hi * token > 800 << 20:
            decodes -= 1
        ctx = (lo, hi)
    if what != "decode":
        # Full-precision prompts stay short: they are how results are checked.
        slices = rng.randint(1, 3 if dtype == "fp16" else 2)
        chunk = _log(rng, 9, 300 if dtype == "fp32" else 512)
        p = _log(rng, 1, 512 if dtype == "fp32" else 3584) - 1
        prefix = (p // 2, p)
    return _attention(dtype, heads, kv_heads, head_dim, decodes, ctx, slices, chunk, prefix,
                      rng.randrange(1 << 20))


# --- shapes of a step, from the case alone --------------------------------------------------------


def _lens(case):
    """``(context lengths, query lengths)``: the prefill slices first, then the decodes."""
    rng = random.Random(case["spread"])
    n = case["slices"]
    step = (case["prefix_hi"] - case["prefix_lo"]) / max(1, n - 1)
    ctx = [case["prefix_lo"] + int(step * i) + case["chunk"] for i in range(n)]
    q = [case["chunk"]] * n
    ctx += [rng.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["decodes"])]
    return ctx, q + [1] * case["decodes"]


def _tables(ctx, q, seed):
    """Disjoint shuffled block tables, and the step's slots and positions."""
    nb = [-(-L // BLOCK) for L in ctx]
    total = sum(nb) + sum(nb) // 8 + 8
    perm = np.random.RandomState(seed % (1 << 32)).permutation(total).astype(np.int32)
    bt = np.full((len(ctx), max(nb)), -1, np.int32)
    at, slots, pos = 0, [], []
    for r, (L, c, b) in enumerate(zip(ctx, q, nb)):
        bt[r, :b] = perm[at : at + b]
        at += b
        p = np.arange(L - c, L)
        slots.append(bt[r, p // BLOCK].astype(np.int64) * BLOCK + p % BLOCK)
        pos.append(p)
    return bt, total, np.concatenate(slots).astype(np.int32), np.concatenate(pos).astype(np.int32)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _codes(g, bits, n, k):
    """A weight ~ N(0, 0.02) as its quantised codes and scales, in plain torch: INT8 with one
    scale per output channel, or INT4 in groups of 128 packed two to a byte."""
    group = k if bits == 8 else 128
    w = torch.randn(n, k // group, group, generator=g, device=DEVICE) * 0.02
    qmax = 127 if bits == 8 else 7
    scales = (w.abs().amax(-1, keepdim=True) / qmax).half()
    codes = (w / scales.float()).round_().clamp_(-qmax, qmax).to(torch.int16).view(n, k)
    if bits == 8:
        packed = (codes & 0xFF).to(torch.uint8)
    else:
        nibbles = (codes + 8).to(torch.uint8)
        packed = nibbles[:, 0::2] | (nibbles[:, 1::2] << 4)
    return packed.contiguous(), scales.view(n, -1).contiguous()


def _weight64(packed, scales, bits):
    """The float64 weight that codes and scales stand for (code * scale, rounded to fp16)."""
    if bits == 8:
        codes = packed.view(torch.int8).half()
    else:
        codes = torch.stack((packed & 15, packed >> 4), -1).view(packed.shape[0], -1).half() - 8
    n, k = codes.shape
    return (codes.view(n, scales.shape[1], -1) * scales[:, :, None]).view(n, k).double()


# --- preparation ----------------------------------------------------------------------------------


def prepare(case, seed):
    return {"attention": _prepare_attention, "linear": _prepare_linear,
            "decoder": _prepare_decoder}[case["op"]](case, seed)


def _prepare_attention(case, seed):
    dtype, d, hkv = DTYPES[case["dtype"]], case["head_dim"], case["kv_heads"]
    ctx, q_lens = _lens(case)
    bt, blocks, slots, _ = _tables(ctx, q_lens, seed)
    g = _generator(seed)
    t = sum(q_lens)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE, dtype=dtype)

    state = {"kp": normal(hkv, blocks, BLOCK, d), "vp": normal(hkv, blocks, BLOCK, d),
             "q": normal(t, case["heads"], d), "k": normal(t, hkv, d), "v": normal(t, hkv, d),
             "scale": d**-0.5, "tables": bt}
    qsl = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    state["plan"], (state["slots"],) = kernels.plan_attention(
        qsl, np.asarray(ctx, np.int32), bt, case["heads"], hkv, d, BLOCK, dtype,
        torch.device(DEVICE), [slots])
    state["out"] = torch.empty_like(state["q"])
    return state


def _prepare_linear(case, seed):
    g = _generator(seed)
    packed, scales = _codes(g, case["bits"], case["n"], case["k"])
    cfg = QuantConfig(group_size=case["k"] if case["bits"] == 8 else 128, bits=case["bits"])
    layer = QuantLinear(case["k"], case["n"], config=cfg, device=DEVICE)
    layer.load_quantized(packed, scales)
    x = torch.randn(case["m"], case["k"], generator=g, device=DEVICE, dtype=torch.float16)
    return {"layer": layer, "x": x}


def _prepare_decoder(case, seed):
    spec = dataclasses.replace(SMOLLM2_1_7B, n_layers=LAYERS)
    g = _generator(seed)
    h, inter, d, heads = spec.hidden_size, spec.intermediate_size, spec.head_dim, spec.n_q_heads
    model = EdgeRagDecoder(spec, device=DEVICE)
    for layer in model.layers:
        layer.qkv.load_quantized(*_codes(g, 8, 3 * heads * d, h))
        layer.o_proj.load_quantized(*_codes(g, 8, h, heads * d))
        layer.gate_up.load_quantized(*_codes(g, 8, 2 * inter, h))
        layer.down_proj.load_quantized(*_codes(g, 8, h, inter))
        for norm in (layer.input_layernorm, layer.post_attention_layernorm):
            norm.weight.copy_(1 + 0.1 * torch.randn(h, generator=g, device=DEVICE))
    model.embed_tokens.copy_(torch.randn(spec.vocab_size, h, generator=g, device=DEVICE) * 0.02)
    model.lm_head.copy_(torch.randn(spec.vocab_size, h, generator=g, device=DEVICE) * 0.02)
    ctx, q_lens = _lens(case)
    bt, blocks, slots, pos = _tables(ctx, q_lens, seed)
    pools = [[torch.randn(spec.n_kv_heads, blocks, BLOCK, d, generator=g, device=DEVICE,
                          dtype=torch.float16) for _ in range(LAYERS)] for _ in range(2)]
    ids = np.random.RandomState(seed % (1 << 32)).randint(0, spec.vocab_size, len(pos))
    ids = ids.astype(np.int32)
    qsl = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    state = {"model": model, "kp": pools[0], "vp": pools[1], "tables": bt, "ids": ids,
             "slots": slots, "positions": pos}
    if not case["graph"]:
        plan, (s, p, i, rows) = kernels.plan_attention(
            qsl, np.asarray(ctx, np.int32), bt, heads, spec.n_kv_heads, d, BLOCK, torch.float16,
            torch.device(DEVICE), [slots, pos, ids, qsl[1:] - 1])
        state["step"] = StepInputs(i, p, s, rows, plan)
        return state
    # A decode batch as the executor runs it: metadata staged once, the iteration captured.
    n = len(ctx)
    fixed = kernels.FixedAttention(torch.device(DEVICE), heads, spec.n_kv_heads, d, BLOCK,
                                   torch.float16, n, bt.shape[1], [n, n, n, n])
    if not fixed.update(None, ctx, [bt[r, : -(-ctx[r] // BLOCK)] for r in range(n)],
                        [slots, pos, ids, np.arange(n, dtype=np.int32)]):
        raise RuntimeError("the decode batch does not fit its own staging")
    s, p, i, rows = (e[:n] for e in fixed.extras)
    step = StepInputs(i, p, s, rows, fixed, all_rows=True)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        model.greedy(step, state["kp"], state["vp"])
        with torch.cuda.graph(graph, stream=stream):
            state["logits"], _ = model.greedy(step, state["kp"], state["vp"])
    torch.cuda.current_stream().wait_stream(stream)
    state.update(graph=graph, step=step)
    return state


# --- one pass ----------------------------------------------------------------------------------


def run(state):
    if "layer" in state:
        return state["layer"](state["x"])
    if "model" in state:
        if "graph" in state:
            state["graph"].replay()
            logits = state["logits"]
        else:
            logits, _ = state["model"].greedy(state["step"], state["kp"], state["vp"])
        return [logits, state["kp"], state["vp"]]
    out = kernels.paged_attention_append(
        state["k"], state["v"], state["slots"], state["q"], state["kp"], state["vp"],
        state["plan"], state["scale"], out=state["out"])
    return [out, state["kp"], state["vp"]]


# --- what a pass cannot do without ------------------------------------------------------------------


def work(case):
    if case["op"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        scales = n * 2 * (1 if case["bits"] == 8 else k // 128)
        return {"bytes": n * k * case["bits"] // 8 + scales + 2 * m * (k + n),
                "flops": 2 * m * n * k}
    ctx, q_lens = _lens(case)
    t = sum(q_lens)
    pairs = sum(c * (L - c) + c * (c + 1) // 2 for L, c in zip(ctx, q_lens))
    if case["op"] == "attention":
        es = 4 if case["dtype"] == "fp32" else 2
        h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
        # Cached K and V read, new K and V read and written, q read, out written.
        cached = sum(L - c for L, c in zip(ctx, q_lens))
        return {"bytes": es * d * (2 * hkv * (cached + 2 * t) + 2 * h * t),
                "flops": 4 * d * h * pairs}
    s = SMOLLM2_1_7B
    h, inter, d, heads = s.hidden_size, s.intermediate_size, s.head_dim, s.n_q_heads
    weights = 4 * heads * d * h + 3 * inter * h
    cached = sum(L - c for L, c in zip(ctx, q_lens))
    kv = 2 * 2 * heads * d * (cached + t)
    return {"bytes": LAYERS * (weights + kv) + 2 * s.vocab_size * (h + len(ctx)) + 2 * t * h,
            "flops": LAYERS * (2 * t * weights + 4 * d * heads * pairs)
            + 2 * len(ctx) * h * s.vocab_size}


def tolerance(case):
    """Four times the error against 64 bits that the path shows: the rounding of its results to
    the dtype (fp16 2e-4 to 3e-4, bf16 1.7e-3, fp32 1.5e-7), and in a decoder the fp16 roundings
    of every layer, which travel on through the residual stream (2.1e-3)."""
    if case["op"] == "linear":
        return {"rel": 1.2e-3}
    if case["op"] == "decoder":
        return {"rel": 8e-3}
    return {"rel": {"fp16": 1.2e-3, "bf16": 7e-3, "fp32": 1e-6}[case["dtype"]]}


# --- the same in 64 bits, in plain torch ----------------------------------------------------------


def _attend64(q, kp, vp, tables, ctx, q_lens, scale):
    """Attention of the packed float64 ``q`` over pools that hold the step's rows already."""
    t, h, d = q.shape
    hkv = kp.shape[0]
    out, at = torch.empty_like(q), 0
    for r, (L, c) in enumerate(zip(ctx, q_lens)):
        blocks = torch.from_numpy(tables[r, : -(-L // BLOCK)].astype(np.int64)).to(q.device)
        k, v = (p[:, blocks].reshape(hkv, -1, d)[:, :L].double() for p in (kp, vp))
        hidden = torch.ones(c, L, dtype=torch.bool, device=q.device).triu_(L - c + 1)
        for j in range(hkv):
            rep = h // hkv
            qj = q[at : at + c, j * rep : (j + 1) * rep].reshape(c * rep, d)
            s = (qj @ k[j].t() * scale).view(c, rep, L)
            s.masked_fill_(hidden[:, None], -math.inf)
            o = torch.softmax(s, -1).view(c * rep, L) @ v[j]
            out[at : at + c, j * rep : (j + 1) * rep] = o.view(c, rep, d)
        at += c
    return out


def _write(pool, slots, rows):
    hkv, blocks, _, d = pool.shape
    at = torch.from_numpy(slots.astype(np.int64)).to(pool.device)
    pool.view(hkv, blocks * BLOCK, d)[:, at] = rows.transpose(0, 1).to(pool.dtype)


def exact(case, seed):
    state = prepare(case, seed)
    torch.cuda.synchronize()
    with torch.no_grad():
        if case["op"] == "linear":
            layer = state["layer"]
            return state["x"].double() @ _weight64(layer.packed, layer.scales, case["bits"]).t()
        ctx, q_lens = _lens(case)
        if case["op"] == "attention":
            slots = state["slots"].cpu().numpy()
            _write(state["kp"], slots, state["k"])
            _write(state["vp"], slots, state["v"])
            out = _attend64(state["q"].double(), state["kp"], state["vp"], state["tables"], ctx,
                            q_lens, state["scale"])
            return [out, None, None]
        return [_decoder64(state, ctx, q_lens), None, None]


def _decoder64(state, ctx, q_lens):
    model, spec = state["model"], state["model"].spec
    d, heads, inter = spec.head_dim, spec.n_q_heads, spec.intermediate_size
    ids = torch.from_numpy(state["ids"].astype(np.int64)).to(DEVICE)
    pos = torch.from_numpy(state["positions"].astype(np.float64)).to(DEVICE)
    freq = spec.rope_theta ** (-torch.arange(0, d, 2, device=DEVICE, dtype=torch.float64) / d)
    angle = torch.cat([pos[:, None] * freq] * 2, -1)[:, None]

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + spec.rms_norm_eps) * w.double()

    def rope(x):
        half = torch.cat([-x[..., d // 2 :], x[..., : d // 2]], -1)
        return x * angle.cos() + half * angle.sin()

    def linear(x, lin):
        return x @ _weight64(lin.packed, lin.scales, 8).t()

    x = model.embed_tokens[ids].double()
    for i, layer in enumerate(model.layers):
        qkv = linear(norm(x, layer.input_layernorm.weight), layer.qkv)
        q, k, v = (p.reshape(-1, heads, d) for p in qkv.chunk(3, -1))
        _write(state["kp"][i], state["slots"], rope(k))
        _write(state["vp"][i], state["slots"], v)
        a = _attend64(rope(q), state["kp"][i], state["vp"][i], state["tables"], ctx, q_lens,
                      d**-0.5)
        x = x + linear(a.reshape(-1, heads * d), layer.o_proj)
        gu = linear(norm(x, layer.post_attention_layernorm.weight), layer.gate_up)
        x = x + linear(torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:], layer.down_proj)
    rows = torch.tensor(np.cumsum(q_lens) - 1, device=DEVICE)
    return norm(x[rows], model.norm.weight) @ model.lm_head.double().t()
