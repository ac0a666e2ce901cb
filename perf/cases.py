"""The work this framework is used for, as cases that can be timed and checked.

A case is a dict of plain values.  `kind` names the public entry point that
runs it, the other fields its sizes and options.  Shapes are those of the
gpt-oss-20b and gpt-oss-120b presets (hidden 2880, 64 query / 8 kv heads of 64,
intermediate 2880, 32 or 128 experts, top-4, vocabulary 201088, sliding window
128).  Inputs are drawn on the device from the seed alone.

kinds
  turn         a whole engine call in the default (exact) modes: prompts in,
               a few generated tokens, tokens and logits out
  score        matrix-core decode steps of a batch over given tokens (every
               step teacher-forced), the logits of the last step out
  moe_layer    neon_moe_layer: router + top-4 experts, the decode-step MoE block
  moe_prompt   neon_moe_prefill / neon_moe_prefill_mx8: the expert FFN of a prompt
  attn_step    neon_attn_decode: one decode step's attention over a KV cache
  attn_prompt  neon_attn_prefill: causal attention over a prompt
  proj_prompt  neon_gemm_bf16: the prompt pass's QKV and O projections
  gemv_mxfp4   neon_mxfp4_gemv: one MXFP4 matrix times a small batch
"""
import math
import random

import numpy as np
import torch

import neonengine_amd as ne

HID, INTER, VOCAB = 2880, 2880, 201088
HQ, HKV, HD = 64, 8, 64
TOP_K, WINDOW = 4, 128
QKV = (HQ + 2 * HKV) * HD
ALPHA, LIMIT = 1.702, 7.0
GAIN = 3.0


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one user's chat turn in the default modes: a prompt of a few hundred
        # tokens, then a short greedy answer at batch 1 (the headline decode)
        dict(name="turn_single", kind="turn", batch=1, lo=333, hi=333, steps=24, temperature=0.0),
        # sixteen sequences of different prompt lengths decoding together,
        # sampled at temperature 0.8 within the 0.95 nucleus
        dict(name="turn_batch", kind="turn", batch=16, lo=5, hi=77, steps=8, temperature=0.8),
        # the throughput decode mode at its largest batch, two layers deep
        dict(name="score_b64", kind="score", batch=64, tokens=24, layers=2, mx8=False),
        # the MoE block of a batch-1 decode step, layer after layer (six layers'
        # own experts, so that the weights come from memory as in a model)
        dict(name="moe_step_b1", kind="moe_layer", batch=1, experts=32, layers=6),
        # the MoE block of a batched decode step of the 128-expert model
        dict(name="moe_step_b16", kind="moe_layer", batch=16, experts=128, layers=1),
        # the expert FFN of a long prompt on the scaled fp8 x fp4 instruction
        dict(name="moe_prompt_mx8", kind="moe_prompt", rows=2047, experts=32, mx8=True),
        # the expert FFN of a medium, ragged prompt in the bf16 form
        dict(name="moe_prompt_bf16", kind="moe_prompt", rows=333, experts=32, mx8=False),
        # the smallest call: a sliding layer's attention of one decode step
        dict(name="attn_step_window", kind="attn_step", batch=1, cache=256, window=WINDOW),
        # long-context decode: eight sequences of different lengths up to 8192 keys
        dict(name="attn_step_long", kind="attn_step", batch=8, cache=8192, window=0),
        # a full layer's attention over a long prompt
        dict(name="attn_prompt_full", kind="attn_prompt", rows=2047, window=0),
        # the QKV projection of a long prompt
        dict(name="proj_prompt_qkv", kind="proj_prompt", rows=2047, which="qkv"),
        # an MXFP4 matrix of gate_up size at the largest batch of its range
        dict(name="gemv_mxfp4_b64", kind="gemv_mxfp4", n=5760, k=HID, batch=64),
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["turn", "score", "moe_layer", "moe_layer", "moe_prompt", "moe_prompt",
                       "attn_step", "attn_step", "attn_prompt", "proj_prompt", "gemv_mxfp4"])
    if kind == "turn":
        batch = _log_int(rng, 1, 16)
        hi = _log_int(rng, 2, max(2, 640 // batch))
        return dict(kind=kind, batch=batch, lo=rng.randint(1, hi), hi=hi,
                    steps=rng.randint(1, 24 if batch == 1 else 8),
                    temperature=rng.choice([0.0, 0.8]))
    if kind == "score":
        return dict(kind=kind, batch=rng.randint(16, 64), tokens=rng.randint(3, 24), layers=2,
                    mx8=rng.random() < 0.3)
    if kind == "moe_layer":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), experts=rng.choice([32, 128]), layers=1)
    if kind == "moe_prompt":
        return dict(kind=kind, rows=_log_int(rng, 2, 2048), experts=rng.choice([32, 32, 128]),
                    mx8=rng.random() < 0.5)
    if kind == "attn_step":
        cache = _log_int(rng, 64, 32768)
        return dict(kind=kind, batch=_log_int(rng, 1, max(1, min(32, 131072 // cache))),
                    cache=cache, window=rng.choice([0, 0, WINDOW]))
    if kind == "attn_prompt":
        return dict(kind=kind, rows=_log_int(rng, 2, 2560), window=rng.choice([0, WINDOW]))
    if kind == "proj_prompt":
        return dict(kind=kind, rows=_log_int(rng, 2, 2560), which=rng.choice(["qkv", "o"]))
    return dict(kind=kind, n=16 * rng.randint(16, 500), k=32 * rng.randint(8, 128),
                batch=_log_int(rng, 1, 64))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + salt)
    return g


def _bf16(shape, g, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x.mul_(std).add_(mean)).to(torch.bfloat16)


def _codes(n, g):
    return torch.randint(0, 256, (n,), generator=g, device="cuda", dtype=torch.uint8)


def _scales(n, g):
    """E8M0 bytes that put uniform E2M1 codes at a standard deviation of about 0.02."""
    return torch.randint(118, 122, (n,), generator=g, device="cuda", dtype=torch.uint8)


def _expert_weights(E, g):
    return dict(
        guc=_codes(E * 2 * INTER * HID // 2, g), gus=_scales(E * 2 * INTER * HID // 32, g),
        gub=_bf16((E, 2 * INTER), g, 0.02),
        dnc=_codes(E * HID * INTER // 2, g), dns=_scales(E * HID * INTER // 32, g),
        dnb=_bf16((E, HID), g, 0.02))


def _prompts(case, seed):
    rng = random.Random(int(seed) * 31 + 5)
    lens = [case["hi"]] + [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"] - 1)]
    return [[rng.randrange(VOCAB) for _ in range(n)] for n in lens]


def _positions(case, seed):
    """Lengths of the sequences of a batch: between half the cache and all of it."""
    rng = random.Random(int(seed) * 17 + 3)
    T = case["cache"]
    return [T - 1] + [rng.randint(T // 2, T - 1) for _ in range(case["batch"] - 1)]


def _routing(case, seed, g):
    """Expert ids and weights of prompt rows: top-4 of logits in which some
    experts are more popular than others."""
    logits = torch.randn((case["rows"], case["experts"]), generator=g, device="cuda")
    logits += 0.5 * torch.randn((case["experts"],), generator=g, device="cuda")
    v, i = torch.topk(logits, TOP_K, dim=1)
    return i.to(torch.int32).contiguous(), torch.softmax(v, dim=1).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    s = dict(case=dict(case))
    if kind == "turn":
        prompts = _prompts(case, seed)
        eng = ne.Engine("gpt-oss-20b", max_seq=4096, max_batch=max(2, case["batch"]))
        eng.init_random(int(seed))
        if case["temperature"] > 0:
            eng.set_sampling(case["temperature"], 0.95, int(seed) + 1)
        s.update(engine=eng, prompts=prompts)
    elif kind == "score":
        eng = ne.Engine("gpt-oss-20b", n_layers=case["layers"], max_seq=4096,
                        max_batch=case["batch"])
        eng.init_random(int(seed))
        # a trained router is decided: with a gain of GAIN on the random one the
        # 4th expert's weight is a few percent, so that a near-tie for its place
        # does not make two correct implementations differ by a whole expert
        for l in range(case["layers"]):
            w = _bf16((32, HID), g, 0.02 * GAIN).view(torch.int16).cpu().numpy()
            eng.load_tensor("model.layers.%d.mlp.router.weight" % l, w)
        eng.set_prefill_mode(ne.PREFILL_STEPWISE)
        eng.set_decode_mode(ne.DECODE_MATRIX_MX8 if case["mx8"] else ne.DECODE_MATRIX)
        rng = random.Random(int(seed) * 13 + 1)
        s.update(engine=eng, prompts=[[rng.randrange(VOCAB) for _ in range(case["tokens"])]
                                      for _ in range(case["batch"])])
    elif kind == "moe_layer":
        B, E = case["batch"], case["experts"]
        s["layers"] = []
        for _ in range(case["layers"]):
            w = _expert_weights(E, g)
            w.update(x=_bf16((B, HID), g), rw=_bf16((E, HID), g, 0.02), rb=_bf16((E,), g, 0.02),
                     h=_bf16((B, HID), g), out=torch.empty((B, HID), dtype=torch.bfloat16,
                                                          device="cuda"),
                     idx=torch.empty((B, TOP_K), dtype=torch.int32, device="cuda"),
                     score=torch.empty((B, TOP_K), dtype=torch.float32, device="cuda"))
            s["layers"].append(w)
        s["ws"] = torch.empty(ne.moe_layer_workspace(B, E, INTER, TOP_K), dtype=torch.uint8,
                              device="cuda")
    elif kind == "moe_prompt":
        M, E = case["rows"], case["experts"]
        s.update(_expert_weights(E, g))
        idx, score = _routing(case, seed, g)
        s.update(x=_bf16((M, HID), g), h=_bf16((M, HID), g), idx=idx, score=score,
                 ws=torch.empty(ne.moe_prefill_workspace(M, E, HID, INTER, TOP_K,
                                                         mx8=case["mx8"]),
                                dtype=torch.uint8, device="cuda"))
    elif kind == "attn_step":
        B, T = case["batch"], case["cache"]
        wb, cb = ne.attn_decode_workspace(B, HQ, HKV, HD, T, case["window"])
        s.update(q=_bf16((B, HQ * HD), g), k=_bf16((B, HKV, T, HD), g),
                 v=_bf16((B, HKV, T, HD), g), sinks=_bf16((HQ,), g),
                 pos=torch.tensor(_positions(case, seed), dtype=torch.int32, device="cuda"),
                 out=torch.empty((B, HQ * HD), dtype=torch.bfloat16, device="cuda"),
                 ws=torch.empty(max(wb, 4), dtype=torch.uint8, device="cuda"),
                 counters=torch.zeros(max(cb, 4), dtype=torch.uint8, device="cuda"))
    elif kind == "attn_prompt":
        M = case["rows"]
        s.update(q=_bf16((M, HQ, HD), g), k=_bf16((HKV, M, HD), g), v=_bf16((HKV, M, HD), g),
                 sinks=_bf16((HQ,), g),
                 out=torch.empty((M, HQ * HD), dtype=torch.bfloat16, device="cuda"))
    elif kind == "proj_prompt":
        M = case["rows"]
        N, K = (QKV, HID) if case["which"] == "qkv" else (HID, HQ * HD)
        s.update(a=_bf16((M, K), g), w=_bf16((N, K), g, 0.02), b=_bf16((N,), g, 0.02),
                 c=_bf16((M, N), g), m=M, n=N, k=K)
    else:
        B, N, K = case["batch"], case["n"], case["k"]
        s.update(codes=_codes(N * K // 2, g), scales=_scales(N * K // 32, g),
                 b=_bf16((N,), g, 0.02), x=_bf16((B, K), g),
                 y=torch.empty((B, N), dtype=torch.bfloat16, device="cuda"))
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "turn":
        eng = s["engine"]
        eng.prefill(s["prompts"])
        eng.decode(case["steps"])
        return dict(tokens=eng.read_tokens(), logits=eng.read_logits())
    if kind == "score":
        eng = s["engine"]
        eng.prefill(s["prompts"])
        return dict(logits=eng.read_logits())
    if kind == "moe_layer":
        outs = []
        for w in s["layers"]:
            ne.moe_layer(w["x"], w["rw"], w["rb"], w["guc"], w["gus"], w["gub"], w["dnc"],
                         w["dns"], w["dnb"], w["h"], w["out"], w["idx"], w["score"],
                         case["batch"], case["experts"], HID, INTER, TOP_K, ALPHA, LIMIT,
                         workspace=s["ws"])
            outs.append(dict(out=w["out"], idx=w["idx"], score=w["score"]))
        return outs
    if kind == "moe_prompt":
        f = ne.moe_prefill_mx8 if case["mx8"] else ne.moe_prefill
        f(s["x"], s["idx"], s["score"], s["guc"], s["gus"], s["gub"], s["dnc"], s["dns"],
          s["dnb"], s["h"], case["rows"], case["experts"], HID, INTER, TOP_K, ALPHA, LIMIT,
          workspace=s["ws"])
        return s["h"]
    if kind == "attn_step":
        ne.attn_decode(s["q"], s["k"], s["v"], s["sinks"], s["pos"], s["out"], case["batch"], HQ,
                       HKV, HD, case["cache"], case["window"], workspace=s["ws"],
                       counters=s["counters"])
        return s["out"]
    if kind == "attn_prompt":
        ne.attn_prefill(s["q"], s["k"], s["v"], s["sinks"], s["out"], case["rows"], HQ, HKV, HD,
                        case["rows"], case["window"])
        return s["out"]
    if kind == "proj_prompt":
        # the O projection adds into the residual stream in place
        ne.gemm_bf16(s["a"], s["w"], s["b"], s["c"], s["m"], s["n"], s["k"],
                     accumulate=case["which"] == "o")
        return s["c"]
    ne.mxfp4_gemv(s["codes"], s["scales"], s["b"], s["x"], s["y"], case["n"], case["k"],
                  case["batch"])
    return s["y"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _fp4(n, k):
    return n * k * 17 / 32


def _used(pairs, experts):
    """Experts that `pairs` random choices are expected to touch."""
    return experts * (1.0 - (1.0 - 1.0 / experts) ** pairs)


def _model(rows, keys, layers, experts=32, heads=0):
    """Bytes and flops of `rows` rows through the layers, `heads` of them through lm_head."""
    expert = _fp4(2 * INTER, HID) + _fp4(HID, INTER) + 2 * (2 * INTER + HID)
    dense = 2.0 * (QKV * HID + HID * HQ * HD + experts * HID)
    by = layers * (dense + _used(rows * TOP_K, experts) * expert + rows * keys * 2 * HKV * HD * 2)
    fl = 2.0 * rows * layers * (QKV * HID + HID * HQ * HD + experts * HID + 3.0 * TOP_K * INTER * HID
                                + 2.0 * keys * HQ * HD)
    if heads:
        by += 2.0 * VOCAB * HID + 4.0 * heads * VOCAB
        fl += 2.0 * heads * VOCAB * HID
    return by, fl


def work(case):
    kind = case["kind"]
    if kind == "turn":
        B, n, steps = case["batch"], (case["lo"] + case["hi"]) / 2.0, case["steps"]
        by, fl = _model(B * n, 0.5 * n, 24, heads=B)
        b1, f1 = _model(B, n + 0.5 * steps, 24, heads=B)
        # the prompt's keys are written and read once by its own pass
        by -= 24 * B * n * (0.5 * n - 1) * 2 * HKV * HD * 2
        return dict(bytes=by + steps * b1, flops=fl + steps * f1)
    if kind == "score":
        b1, f1 = _model(case["batch"], 0.5 * case["tokens"], case["layers"], heads=case["batch"])
        return dict(bytes=case["tokens"] * b1, flops=case["tokens"] * f1)
    if kind == "moe_layer":
        B, E = case["batch"], case["experts"]
        by = E * HID * 2 + _used(B * TOP_K, E) * (_fp4(2 * INTER, HID) + _fp4(HID, INTER)
                                                  + 2 * (2 * INTER + HID)) + 3 * B * HID * 2
        fl = 2.0 * B * (E * HID + 3.0 * TOP_K * INTER * HID)
        return dict(bytes=case["layers"] * by, flops=case["layers"] * fl)
    if kind == "moe_prompt":
        M, E = case["rows"], case["experts"]
        by = _used(M * TOP_K, E) * (_fp4(2 * INTER, HID) + _fp4(HID, INTER)
                                    + 2 * (2 * INTER + HID)) + M * (3 * HID * 2 + TOP_K * 8)
        return dict(bytes=by, flops=2.0 * M * 3.0 * TOP_K * INTER * HID)
    if kind == "attn_step":
        T, B = case["cache"], case["batch"]
        keys = min(T if B == 1 else 0.75 * T, case["window"] or T)
        return dict(bytes=B * (keys * 2 * HKV * HD * 2 + 2 * HQ * HD * 2),
                    flops=4.0 * B * keys * HQ * HD)
    if kind == "attn_prompt":
        M, W = case["rows"], case["window"] or case["rows"]
        pairs = sum(min(t + 1, W) for t in range(M))
        return dict(bytes=M * (2 * HQ * HD + 2 * HKV * HD) * 2, flops=4.0 * pairs * HQ * HD)
    if kind == "proj_prompt":
        N, K = (QKV, HID) if case["which"] == "qkv" else (HID, HQ * HD)
        M = case["rows"]
        by = 2.0 * (N * K + M * K + M * N * (2 if case["which"] == "o" else 1))
        return dict(bytes=by, flops=2.0 * M * N * K)
    N, K, B = case["n"], case["k"], case["batch"]
    return dict(bytes=_fp4(N, K) + 2 * N + 2 * B * (K + N), flops=2.0 * B * N * K)


# ---------------------------------------------------------------------------
# how far another correct implementation may be off
# ---------------------------------------------------------------------------
def tolerance(case):
    kind = case["kind"]
    if kind == "turn":
        # the exact modes promise the same bits whatever the batch or the pass
        return "exact"
    if kind == "score":
        # matrix against exact steps of the same inputs: rel 0.0064 - 0.0076,
        # max 0.05 - 0.1 where no near-tied expert changes place (batches of
        # 16, 40 and 64, both instruction forms)
        return dict(rel=2.8e-2, max=0.6)
    if kind == "moe_prompt":
        # two roundings to bf16 on the way: 2.6e-3 off the 64-bit result
        return dict(rel=3e-3, max=2e-2)
    # one rounding to bf16: 1.7e-3 off the 64-bit result
    return dict(rel=2e-3, max=1.6e-2)


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]


def _dequant(codes, scales, N, K):
    """[N][K/2] code bytes and [N][K/32] E8M0 scales as float64 [N][K]."""
    table = torch.tensor(_E2M1, dtype=torch.float64, device=codes.device)
    c = codes.view(N, K // 2).to(torch.int64)
    w = torch.stack([table[c & 15], table[c >> 4]], dim=2).reshape(N, K // 32, 32)
    s = torch.pow(torch.tensor(2.0, dtype=torch.float64, device=codes.device),
                  scales.view(N, K // 32, 1).to(torch.float64) - 127.0)
    return (w * s).reshape(N, K)


def _experts(x, idx, score, w, E):
    """sum_s score[t][s] expert_{idx[t][s]}(x[t]) in float64."""
    out = torch.zeros_like(x)
    guc, gus = w["guc"].view(E, -1), w["gus"].view(E, -1)
    dnc, dns = w["dnc"].view(E, -1), w["dns"].view(E, -1)
    for e in torch.unique(idx).tolist():
        t, slot = torch.nonzero(idx == e, as_tuple=True)
        y = x[t] @ _dequant(guc[e], gus[e], 2 * INTER, HID).T + w["gub"][e].double()
        gate = y[:, 0::2].clamp(max=LIMIT)
        up = y[:, 1::2].clamp(min=-LIMIT, max=LIMIT)
        a = (up + 1.0) * gate * torch.sigmoid(ALPHA * gate)
        y = a @ _dequant(dnc[e], dns[e], HID, INTER).T + w["dnb"][e].double()
        out.index_add_(0, t, y * score[t, slot].double()[:, None])
    return out


def _attend(q, k, v, sinks, mask):
    """q [h][r][d], k / v [h][t][d], mask [r][t] of the keys a row sees."""
    sc = (q @ k.transpose(1, 2)) / math.sqrt(HD)
    sc = sc.masked_fill(~mask[None], -math.inf)
    sink = sinks.double()[:, None, None].expand(-1, sc.shape[1], 1)
    p = torch.softmax(torch.cat([sc, sink], dim=2), dim=2)[:, :, :-1]
    return p @ v


def exact(case, seed):
    kind = case["kind"]
    if kind in ("turn", "score"):
        return None  # a whole model in 64 bits takes minutes
    s = prepare(case, seed)
    if kind == "moe_layer":
        outs = []
        for w in s["layers"]:
            x = w["x"].double()
            lg = x @ w["rw"].double().T + w["rb"].double()
            v, i = torch.topk(lg, TOP_K, dim=1)
            p = torch.softmax(v, dim=1)
            outs.append(dict(out=w["h"].double() + _experts(x, i, p, w, case["experts"]),
                             idx=None, score=p))
        return outs
    if kind == "moe_prompt":
        return s["h"].double() + _experts(s["x"].double(), s["idx"].long(), s["score"], s,
                                          case["experts"])
    if kind == "attn_step":
        rows = []
        for b, p in enumerate(_positions(case, seed)):
            lo = max(0, p + 1 - case["window"]) if case["window"] else 0
            k = s["k"][b, :, lo:p + 1].double().repeat_interleave(HQ // HKV, dim=0)
            v = s["v"][b, :, lo:p + 1].double().repeat_interleave(HQ // HKV, dim=0)
            q = s["q"][b].view(HQ, 1, HD).double()
            mask = torch.ones((1, p + 1 - lo), dtype=torch.bool, device="cuda")
            rows.append(_attend(q, k, v, s["sinks"], mask).reshape(HQ * HD))
        return torch.stack(rows)
    if kind == "attn_prompt":
        M = case["rows"]
        t = torch.arange(M, device="cuda")
        mask = t[None, :] <= t[:, None]
        if case["window"]:
            mask &= t[None, :] > t[:, None] - case["window"]
        out = torch.empty((M, HQ, HD), dtype=torch.float64, device="cuda")
        g = HQ // HKV
        for j in range(HKV):
            out[:, j * g:(j + 1) * g] = _attend(
                s["q"][:, j * g:(j + 1) * g].double().permute(1, 0, 2).contiguous(),
                s["k"][j].double().expand(g, -1, -1).contiguous(),
                s["v"][j].double().expand(g, -1, -1).contiguous(),
                s["sinks"][j * g:(j + 1) * g], mask).permute(1, 0, 2)
        return out.reshape(M, HQ * HD)
    if kind == "proj_prompt":
        y = s["a"].double() @ s["w"].double().T + s["b"].double()
        return s["c"].double() + y if case["which"] == "o" else y
    return s["x"].double() @ _dequant(s["codes"], s["scales"], case["n"], case["k"]).T \
        + s["b"].double()
