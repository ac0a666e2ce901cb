"""GPU checks of the batched prefill: matrix-core GEMMs, grouped MXFP4 expert
GEMMs and the tiled causal sink attention, then the whole prompt pass.

The matrix cores accumulate in their own order, so unlike the decode kernels
these are not bit-identical to the canonical oracle.  The bars:
  - GEMM: within one bf16 rounding of the fp64 product plus fp32-accumulation
    slack (2^-17 of the sum of |terms|), per element;
  - experts and attention: the fp32 results of the canonical oracle within a
    stated relative bound (one bf16 rounding of the intermediate activations
    can differ, and the fast exp of the prefill attention);
  - whole prompt, up to the full 20b width at four layers: north_star's 2e-2
    relative bound on the logits against the exact stepwise path, and the
    same first token wherever the stepwise top-2 margin exceeds that bound;
    at all 24 layers the rounding differences grow with depth in a
    random-init model, and that case has a bar of its own (below).
"""
import sys

import numpy as np
import pytest

import neonengine_amd as ne
from tests.gpu_util import bf16_err_ok, empty_dev, fix_routing, to_dev, to_host, torch_cuda

pytestmark = pytest.mark.gpu

def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


# (67, 48, 96): K not a multiple of the 64-deep K step (zero-filled tail)
@pytest.mark.parametrize("M,N,K", [(2047, 5120, 2880), (300, 2880, 4096), (5, 32, 2880),
                                   (129, 200, 64), (67, 48, 96)])
def test_gemm_bf16(orc, M, N, K):
    A = orc.fill_bf16(0, 31, M * K, 0.0, 1.0)
    W = orc.fill_bf16(0, 32, N * K, 0.0, 0.02)
    bias = orc.fill_bf16(0, 33, N, 0.0, 0.02)
    say(f"gemm_bf16 M={M} N={N} K={K}")
    C = empty_dev((M, N), np.uint16)
    ne.gemm_bf16(to_dev(A), to_dev(W), to_dev(bias), C, M, N, K)
    got = to_host(C)
    Af = orc.bf16_to_f32(A).reshape(M, K).astype(np.float64)
    Wf = orc.bf16_to_f32(W).reshape(N, K).astype(np.float64)
    bf = orc.bf16_to_f32(bias).astype(np.float64)
    ref = Af @ Wf.T + bf
    abs_sum = np.abs(Af) @ np.abs(Wf).T + np.abs(bf)
    ok, ratio = bf16_err_ok(got, ref, abs_sum)
    say(f"  worst error / bound = {ratio.max():.3f}")
    assert ok.all()


def test_gemm_bf16_residual(orc):
    M, N, K = 70, 2880, 4096
    A = orc.fill_bf16(1, 34, M * K, 0.0, 1.0)
    W = orc.fill_bf16(1, 35, N * K, 0.0, 0.02)
    res = orc.fill_bf16(1, 36, M * N, 0.0, 5.0)
    C = to_dev(res)
    ne.gemm_bf16(to_dev(A), to_dev(W), None, C, M, N, K, accumulate=True)
    got = to_host(C).reshape(M, N)
    # y = bf16(res + bf16(dot)): compare against the exact dot rounded the same way
    Af = orc.bf16_to_f32(A).reshape(M, K).astype(np.float64)
    Wf = orc.bf16_to_f32(W).reshape(N, K).astype(np.float64)
    dot = Af @ Wf.T
    ref = orc.bf16_to_f32(res).reshape(M, N).astype(np.float64) + dot
    abs_sum = np.abs(Af) @ np.abs(Wf).T
    bound = 2.0 ** -7 * np.abs(ref) + 2.0 ** -8 * np.abs(dot) + 2.0 ** -17 * abs_sum + 1e-30
    err = np.abs(orc.bf16_to_f32(got).astype(np.float64) - ref)
    say(f"gemm residual: worst error / bound = {(err / bound).max():.3f}")
    assert (err <= bound).all()


def moe_weights(orc, E, H, I, seed):
    return dict(
        rw=orc.fill_bf16(seed, 52, E * H, 0.0, 0.02),
        rb=orc.fill_bf16(seed, 53, E, 0.0, 0.02),
        guc=orc.fill_bytes(seed, 54, E * 2 * I * H // 2),
        gus=orc.fill_scales(seed, 55, E * 2 * I * H // 32, 119, 6),
        gub=orc.fill_bf16(seed, 56, E * 2 * I, 0.0, 0.02),
        dnc=orc.fill_bytes(seed, 57, E * H * I // 2),
        dns=orc.fill_scales(seed, 58, E * H * I // 32, 119, 6),
        dnb=orc.fill_bf16(seed, 59, E * H, 0.0, 0.02),
    )


# (29, 8, 288, 352, 2): H and I not multiples of the 64-deep K step
@pytest.mark.parametrize("M,E,H,I,k", [(300, 32, 2880, 2880, 4), (37, 8, 256, 512, 2),
                                       (29, 8, 288, 352, 2)])
def test_moe_prefill_vs_oracle(orc, M, E, H, I, k):
    """Rows grouped by expert into MXFP4 matrix-core GEMMs vs the canonical
    per-row MoE (experts and weights from the oracle's router)."""
    d = moe_weights(orc, E, H, I, seed=2)
    x = orc.fill_bf16(2, 51, M * H, 0.0, 1.0)
    ref, ridx, rsc = orc.moe_layer(x, d["rw"], d["rb"], d["guc"], d["gus"], d["gub"], d["dnc"],
                                   d["dns"], d["dnb"], E, H, I, k)
    say(f"moe_prefill M={M} E={E} H={H} I={I} k={k}")
    h = to_dev(np.zeros((M, H), np.uint16))  # residual 0: h becomes bf16(moe)
    dv = {n: to_dev(v) for n, v in d.items()}
    ne.moe_prefill(to_dev(x), to_dev(ridx), to_dev(rsc), dv["guc"], dv["gus"], dv["gub"],
                   dv["dnc"], dv["dns"], dv["dnb"], h, M, E, H, I, k)
    got = orc.bf16_to_f32(to_host(h)).astype(np.float64)
    r = orc.bf16_to_f32(ref).astype(np.float64)
    err = np.abs(got - r)
    rel = err.max() / np.abs(r).max()
    same = (to_host(h) == ref).mean()
    say(f"  max error / max|ref| = {rel:.3e}, median |err| / rms = "
        f"{np.median(err) / np.sqrt((r ** 2).mean()):.3e}, bit-equal fraction {same:.3f}")
    assert rel < 2e-2
    assert np.median(err) <= 2.0 ** -8 * np.sqrt((r ** 2).mean())


def test_moe_prefill_drops_out_of_range_ids(orc):
    """Ids outside [0, E) given to neon_moe_prefill: those pairs join no
    expert group, add 0 in the combine, and neon_device_check reports
    NEON_EINVAL; the other pairs match the oracle with the slots dropped."""
    M, E, H, I, k = 37, 8, 256, 512, 2
    d = moe_weights(orc, E, H, I, seed=4)
    x = orc.fill_bf16(4, 51, M * H, 0.0, 1.0)
    _, ridx, rsc = orc.moe_layer(x, d["rw"], d["rb"], d["guc"], d["gus"], d["gub"], d["dnc"],
                                 d["dns"], d["dnb"], E, H, I, k)
    ridx = ridx.copy()
    ridx[3, 0], ridx[20, 1], ridx[36, 0] = E, -7, 1000
    want = orc.moe_experts(x, ridx, rsc, d["guc"], d["gus"], d["gub"], d["dnc"], d["dns"],
                           d["dnb"], E, H, I, k)
    h = to_dev(np.zeros((M, H), np.uint16))
    dv = {n: to_dev(v) for n, v in d.items()}
    ne.device_check()
    ne.moe_prefill(to_dev(x), to_dev(ridx), to_dev(rsc), dv["guc"], dv["gus"], dv["gub"],
                   dv["dnc"], dv["dns"], dv["dnb"], h, M, E, H, I, k)
    with pytest.raises(ne.NeonError) as e:
        ne.device_check()
    assert e.value.status == ne.NEON_EINVAL
    got = orc.bf16_to_f32(to_host(h)).astype(np.float64)
    r = orc.bf16_to_f32(want).astype(np.float64)
    rel = np.abs(got - r).max() / np.abs(r).max()
    say(f"moe_prefill with dropped ids: max error / max|ref| = {rel:.3e}")
    assert rel < 2e-2


@pytest.mark.parametrize("H,I", [(32, 96), (128, 224), (288, 320), (256, 544)])
def test_moe_prefill_tile_edges(orc, H, I):
    """The FP4 GEMM tiles where they can go wrong: experts of 0 to 129 rows
    (32-row blocks of a 128-row tile that are full, partly full or skipped) and
    K of 1 to 9 steps of 64 (whole and half last steps; every remainder of the
    4 steps in flight).  The bars of test_moe_prefill_vs_oracle."""
    E, k = 8, 1
    counts = [0, 1, 31, 32, 33, 64, 97, 129]
    M = sum(counts)
    d = moe_weights(orc, E, H, I, seed=7)
    x = orc.fill_bf16(7, 51, M * H, 0.0, 1.0)
    idx = np.repeat(np.arange(E, dtype=np.int32), counts).reshape(M, 1)
    idx = np.ascontiguousarray(idx[np.random.default_rng(7).permutation(M)])
    score = np.ones((M, 1), np.float32)
    want = orc.moe_experts(x, idx, score, d["guc"], d["gus"], d["gub"], d["dnc"], d["dns"],
                           d["dnb"], E, H, I, k)
    h = to_dev(np.zeros((M, H), np.uint16))
    dv = {n: to_dev(v) for n, v in d.items()}
    ne.moe_prefill(to_dev(x), to_dev(idx), to_dev(score), dv["guc"], dv["gus"], dv["gub"],
                   dv["dnc"], dv["dns"], dv["dnb"], h, M, E, H, I, k)
    got = orc.bf16_to_f32(to_host(h)).astype(np.float64).reshape(M, H)
    r = orc.bf16_to_f32(want).astype(np.float64).reshape(M, H)
    err = np.abs(got - r)
    say(f"moe_prefill H={H} I={I}: max error / max|ref| = {err.max() / np.abs(r).max():.3e}")
    assert err.max() < 2e-2 * np.abs(r).max()
    assert np.median(err) <= 2.0 ** -8 * np.sqrt((r ** 2).mean())


@pytest.mark.parametrize("gate,up", [(6.0, 7.0), (2.0 ** -9, 0.0)])
def test_moe_prefill_every_scale_and_code(orc, gate, up):
    """Every E8M0 scale (0, 1, 254 and the NaN 255 among them) times every E2M1
    code at every place of a 32-value block, through the bf16 form's
    dequantisation: expert e's activation is A at column e and 0 elsewhere (x is
    0, the gate bias one-hot), its down row h holds the code of h / 256 at that
    column and the scale h % 256, so out[e][h] is bf16(A W).  The products are
    exact in fp32 where they are normal (8 + 2 bits); gate 6 lifts the
    subnormal weights above 2^-126, gate 2^-9 keeps the largest finite."""
    H, I, E = 4096, 32, 32
    M = E
    cols, rows = np.arange(I), np.arange(H)
    guc = np.zeros((E, 2 * I, H // 2), np.uint8)
    gus = np.full((E, 2 * I, H // 32), 127, np.uint8)
    gub = np.zeros((E, 2 * I), np.float32)
    gub[cols, 2 * cols] = gate
    gub[:, 1::2] = up
    dnc = np.zeros((E, H, I // 2), np.uint8)
    for e in range(E):
        dnc[e, :, e // 2] = (rows // 256) << (4 * (e & 1))
    dns = np.broadcast_to((rows % 256).astype(np.uint8)[None, :, None], (E, H, 1))
    h = to_dev(np.zeros((M, H), np.uint16))
    say(f"moe_prefill scales x codes, gate {gate}")
    ne.moe_prefill(to_dev(np.zeros((M, H), np.uint16)), to_dev(cols.astype(np.int32).reshape(M, 1)),
                   to_dev(np.ones((M, 1), np.float32)), to_dev(guc), to_dev(gus),
                   to_dev(orc.f32_to_bf16(gub)), to_dev(dnc), to_dev(dns),
                   to_dev(np.zeros((E, H), np.uint16)), h, M, E, H, I, 1)
    got = orc.bf16_to_f32(to_host(h)).reshape(M, H).astype(np.float64)
    e2m1 = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6], np.float64)
    val = np.concatenate([e2m1, -e2m1])[rows // 256]
    w = np.ldexp(val, rows % 256 - 127)                     # exact in float64
    w[np.abs(w) > 3.4e38] = np.copysign(np.inf, w[np.abs(w) > 3.4e38])  # 2^128 and more
    w[rows % 256 == 255] = np.nan
    A = got[0, 2 * 256 + 127]                               # the weight 1.0
    assert np.isfinite(A) and A > 0 and (got[:, 2 * 256 + 127] == A).all()
    with np.errstate(over="ignore", invalid="ignore"):
        want = orc.bf16_to_f32(orc.f32_to_bf16((A * w).astype(np.float32))).astype(np.float64)
    small = (np.abs(A * w) > 0) & (np.abs(A * w) < 2.0 ** -126)  # subnormal results: not claimed
    ok = (got == want[None, :]) | (np.isnan(got) & np.isnan(want)[None, :]) | small[None, :]
    bad = np.argwhere(~ok)
    assert len(bad) == 0, [(int(e), int(r) // 256, int(r) % 256, got[e, r], want[r])
                           for e, r in bad[:8]]
    if gate > 1:
        assert not small.any()


@pytest.mark.parametrize("window", [0, 64])
def test_attn_prefill_vs_oracle(orc, window):
    M, Hq, Hkv, D, T = 200, 8, 2, 64, 256
    q = orc.fill_bf16(4, 61, M * Hq * D, 0.0, 1.0)
    kc = orc.fill_bf16(4, 62, Hkv * T * D, 0.0, 1.0)
    vc = orc.fill_bf16(4, 63, Hkv * T * D, 0.0, 1.0)
    sinks = orc.fill_bf16(4, 64, Hq, 0.0, 1.0)
    say(f"attn_prefill M={M} Hq={Hq} Hkv={Hkv} window={window}")
    out = empty_dev((M, Hq * D), np.uint16)
    ne.attn_prefill(to_dev(q), to_dev(kc), to_dev(vc), to_dev(sinks), out, M, Hq, Hkv, D, T,
                    window)
    got = to_host(out)
    # every row is the decode attention of its own position over the same cache
    kcb = np.broadcast_to(kc.reshape(1, -1), (M, kc.size))
    vcb = np.broadcast_to(vc.reshape(1, -1), (M, vc.size))
    _, ref = orc.attn_decode(q, kcb, vcb, sinks, M, Hq, Hkv, D, T,
                             np.arange(M, dtype=np.int32), window)
    vmax = np.abs(orc.bf16_to_f32(vc)).max()
    ok, ratio = bf16_err_ok(got, ref, np.full(ref.shape, vmax), k_eps=2.0 ** -14)
    say(f"  worst error / bound = {ratio.max():.3f}")
    assert ok.all()


SMALL = dict(n_layers=4, hidden=512, n_heads=16, n_kv_heads=2, head_dim=64, n_experts=8,
             top_k=4, intermediate=512, vocab=4096, sliding_window=128, max_seq=512,
             max_batch=2)


def prompt_pass(cfg, seed, prompt, n_steps, mode, fixed_routing=False):
    eng = ne.Engine(cfg)
    eng.init_random(seed)
    if fixed_routing:
        fix_routing(eng, cfg)
    eng.set_prefill_mode(mode)
    eng.prefill(prompt)
    first = eng.read_logits()
    eng.decode(n_steps)
    toks = eng.read_tokens()[:, len(prompt[0]):]
    eng.close()
    return first, toks


def compare_modes(cfg, seed, prompt, n_steps, fixed_routing=False, bar=2e-2,
                  mode=ne.PREFILL_BATCHED, ref_mode=ne.PREFILL_STEPWISE):
    """A matrix-core prompt pass (`mode`) vs an exact one (`ref_mode`:
    stepwise or chunked, both bit-identical to the oracle)."""
    torch_cuda()
    say(f"prefill modes layers={cfg.n_layers} hidden={cfg.hidden} batch={len(prompt)} "
        f"prompt={len(prompt[0])} fixed_routing={fixed_routing} mode={mode} ref={ref_mode}")
    lg_s, tok_s = prompt_pass(cfg, seed, prompt, n_steps, ref_mode, fixed_routing)
    lg_b, tok_b = prompt_pass(cfg, seed, prompt, n_steps, mode, fixed_routing)
    rel = np.abs(lg_b - lg_s).max() / np.abs(lg_s).max()
    top2 = np.sort(lg_s, axis=1)[:, -2:]
    margin = (top2[:, 1] - top2[:, 0]) / np.abs(lg_s).max(axis=1)
    say(f"  logits rel max err {rel:.3e}; first-token top-2 margin (relative) {margin}")
    assert rel < bar
    for b in range(len(prompt)):
        if margin[b] > bar:  # a decisive first token must agree
            assert tok_b[b, 0] == tok_s[b, 0]
    agree = (tok_b == tok_s).all(axis=1)
    say(f"  greedy ids identical over {n_steps + 1} tokens per row: {agree}")
    return rel, agree


def test_small_model_batched_prefill():
    """Two rows, 150-token prompts: several 128-row GEMM tiles and the moving
    128-key sliding window inside the prompt."""
    cfg = ne.config_preset("gpt-oss-20b", **SMALL)
    prompt = [[(7 * i + 3) % 4096 for i in range(150)], [(11 * i + 5) % 4096 for i in range(150)]]
    compare_modes(cfg, 9, prompt, 16)


def test_small_model_batched_prefill_ring_wrap():
    """A 300-token prompt: the sliding layers' 256-row ring cache keeps only
    the last 256 prompt rows, and the prompt attention reads the staged rows."""
    cfg = ne.config_preset("gpt-oss-20b", **SMALL)
    prompt = [[(13 * i + 1) % 4096 for i in range(300)], [(5 * i + 2) % 4096 for i in range(300)]]
    compare_modes(cfg, 4, prompt, 16)


def test_gpt_oss_20b_batched_prefill():
    """Full 20b width (2880 hidden, 64 / 8 heads, 32 experts, vocab 201088),
    four layers (two sliding, two full), 300-token prompt past the 256-row
    ring, free routing: north_star's 2e-2 bar."""
    cfg = ne.config_preset("gpt-oss-20b", max_seq=512, n_layers=4)
    prompt = [[(1009 * i + 17) % 201088 for i in range(300)]]
    compare_modes(cfg, 0, prompt, 16)


def test_gpt_oss_20b_batched_prefill_full_depth():
    """All 24 layers.  The matrix cores round in another order, so single
    bf16 outputs differ by one unit now and then, and a random-init model
    amplifies such differences with depth: measured with the routing fixed
    (router weights 0, distinct biases), the logits differ by 4.9e-3, 1.4e-2,
    2.5e-2 and 6.7e-2 (relative) at 2, 6, 12 and 24 layers.  With free routing
    some rows' 4th and 5th router logits also lie within rounding of each
    other, so the modes pick different experts (0.52 at 12 layers).  The bar
    is twice what a change of summation order alone does to this model at 24
    layers with the routing fixed: the CPU oracle in its fp64-accumulation
    order differs from its canonical fp32 order by up to 6.6e-2
    (tests/golden/conditioning.npz), so 0.13; the exact prompt modes stay
    the default."""
    import os
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "conditioning.npz")
    with np.load(path, allow_pickle=False) as z:
        bar = 2 * float(z["fixed_24"].max())
    cfg = ne.config_preset("gpt-oss-20b", max_seq=512)
    prompt = [[(1009 * i + 17) % 201088 for i in range(300)]]
    rel, _ = compare_modes(cfg, 0, prompt, 16, fixed_routing=True, bar=bar)
    assert rel < bar


def conditioning_bar(key):
    import os
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "conditioning.npz")
    with np.load(path, allow_pickle=False) as z:
        return 2 * float(z[key].max())


@pytest.mark.parametrize("mode", [ne.PREFILL_BATCHED, ne.PREFILL_MX8])
def test_gpt_oss_20b_matrix_prefill_2048(mode):
    """The matrix-core prompt passes at the length the bench quotes them: the
    24-layer 20b model, a 2048-token prompt (32 key tiles per query tile in
    the prompt attention, ~8k (row, slot) pairs in the expert grouping, the
    XCD block order over many row tiles per expert), routing fixed, against
    the exact chunked pass: the first token's logits within twice the
    oracle's own reorder error at 24 layers."""
    bar = conditioning_bar("fixed_24")
    cfg = ne.config_preset("gpt-oss-20b", max_seq=2048 + 32)
    rng = np.random.default_rng(2048)
    prompt = [rng.integers(0, cfg.vocab, 2048).tolist()]
    rel, _ = compare_modes(cfg, 0, prompt, 8, fixed_routing=True, bar=bar, mode=mode,
                           ref_mode=ne.PREFILL_CHUNKED)
    assert rel < bar


@pytest.mark.parametrize("plen", [2048, 16384])
def test_gpt_oss_120b_mx8_prefill(plen):
    """Config 4: the gpt-oss-120b shape (36 layers, 128 experts), a 2048- and
    a 16384-token prompt in the MXFP8 matrix-core pass against the exact
    chunked pass, routing fixed: the first token's logits within twice the
    oracle's own reorder error at 36 layers; then 8 greedy steps decode on
    top of each."""
    bar = conditioning_bar("fixed_36")
    cfg = ne.config_preset("gpt-oss-120b", max_seq=plen + 16)
    rng = np.random.default_rng(plen)
    prompt = [rng.integers(0, cfg.vocab, plen).tolist()]
    rel, _ = compare_modes(cfg, 1, prompt, 8, fixed_routing=True, bar=bar, mode=ne.PREFILL_MX8,
                           ref_mode=ne.PREFILL_CHUNKED)
    assert rel < bar


def test_prefill_mode_validation():
    torch_cuda()
    cfg = ne.config_preset("gpt-oss-20b", **dict(SMALL, max_seq=16))
    eng = ne.Engine(cfg)
    with pytest.raises(ne.NeonError) as e:
        eng.set_prefill_mode(7)
    assert e.value.status == ne.NEON_EINVAL
    eng.set_prefill_mode(ne.PREFILL_BATCHED)
    eng.set_prefill_mode(ne.PREFILL_STEPWISE)
    eng.set_prefill_mode(ne.PREFILL_CHUNKED)
    eng.close()


# ---------------------------------------------------------------------------
# MXFP8 x MXFP4 expert GEMMs (NEON_PREFILL_MX8, v_mfma_scale_f32_32x32x64_f8f6f4)
# ---------------------------------------------------------------------------
def test_mx8_quant_bitexact(orc):
    """The device quantiser gives the oracle's bytes: both E4M3 terms and both
    scale bytes of every block, over rows spanning 2^-130 .. 2^120 with zero
    blocks, NaN and infinite elements, and blocks whose maximum's
    significand is above and below 1.75."""
    torch_cuda()
    rng = np.random.default_rng(11)
    rows, K = 257, 2880
    x = (rng.standard_normal((rows, K)) *
         np.exp2(rng.integers(-60, 60, (rows, 1)))).astype(np.float32)
    x[1, :64] = 0.0
    x[2, 5], x[2, 40], x[2, 77] = np.nan, np.inf, -np.inf
    x[3, :] *= np.float32(2.0 ** -70)
    x[4, :32] = np.float32(2.0 ** -130)       # bf16 subnormals
    x[5, :] = np.float32(2.0 ** 100) * rng.standard_normal(K).astype(np.float32)
    xb = orc.f32_to_bf16(x.ravel()).reshape(rows, K)
    want = orc.mx8_quant(xb)
    hi, lo = empty_dev((rows, K), np.uint8), empty_dev((rows, K), np.uint8)
    sh, sl = empty_dev((rows, K // 32), np.uint8), empty_dev((rows, K // 32), np.uint8)
    say(f"mx8_quant rows={rows} K={K}")
    ne.mx8_quant(to_dev(xb), rows, K, hi, lo, sh, sl)
    for name, g, w in zip(("hi", "lo", "s_hi", "s_lo"), (hi, lo, sh, sl), want):
        got = to_host(g)
        bad = np.argwhere(got != w)
        if len(bad):
            r, c = bad[0]
            say(f"  {name} differs at {r},{c}: gpu {got[r, c]:#x} oracle {w[r, c]:#x}")
        assert not len(bad), name


@pytest.mark.parametrize("M,E,H,I,k", [(300, 32, 2880, 2880, 4), (37, 8, 256, 512, 2)])
def test_moe_prefill_mx8_vs_oracle(orc, M, E, H, I, k):
    """neon_moe_prefill_mx8 against the canonical per-row MoE at the bars of
    the bf16 grouped form (2e-2 relative max, median within 2^-8 of the rms):
    the two-term MXFP8 inputs carry each bf16 block to within half a bf16
    unit of its maximum, so the errors stay of the bf16 form's size, which
    the test prints beside them."""
    d = moe_weights(orc, E, H, I, seed=2)
    x = orc.fill_bf16(2, 51, M * H, 0.0, 1.0)
    ref, ridx, rsc = orc.moe_layer(x, d["rw"], d["rb"], d["guc"], d["gus"], d["gub"], d["dnc"],
                                   d["dns"], d["dnb"], E, H, I, k)
    say(f"moe_prefill_mx8 M={M} E={E} H={H} I={I} k={k}")
    dv = {n: to_dev(v) for n, v in d.items()}
    r = orc.bf16_to_f32(ref).astype(np.float64)
    rms = np.sqrt((r ** 2).mean())
    out = {}
    for name, fn in (("bf16", ne.moe_prefill), ("mx8", ne.moe_prefill_mx8)):
        h = to_dev(np.zeros((M, H), np.uint16))
        fn(to_dev(x), to_dev(ridx), to_dev(rsc), dv["guc"], dv["gus"], dv["gub"],
           dv["dnc"], dv["dns"], dv["dnb"], h, M, E, H, I, k)
        err = np.abs(orc.bf16_to_f32(to_host(h)).astype(np.float64) - r)
        out[name] = (err.max() / np.abs(r).max(), np.median(err) / rms)
        say(f"  {name}: max error / max|ref| = {out[name][0]:.3e}, "
            f"median |err| / rms = {out[name][1]:.3e}")
    assert out["mx8"][0] < 2e-2
    assert out["mx8"][1] <= 2.0 ** -8


def test_small_model_mx8_prefill():
    cfg = ne.config_preset("gpt-oss-20b", **SMALL)
    prompt = [[(7 * i + 3) % 4096 for i in range(150)], [(11 * i + 5) % 4096 for i in range(150)]]
    compare_modes(cfg, 9, prompt, 16, mode=ne.PREFILL_MX8)


def test_gpt_oss_20b_mx8_prefill():
    """Full 20b width, four layers, 300-token prompt: the 2e-2 bar."""
    cfg = ne.config_preset("gpt-oss-20b", max_seq=512, n_layers=4)
    prompt = [[(1009 * i + 17) % 201088 for i in range(300)]]
    compare_modes(cfg, 0, prompt, 16, mode=ne.PREFILL_MX8)


def test_gpt_oss_20b_mx8_prefill_full_depth():
    """All 24 layers with the routing fixed: the conditioning bar of the
    batched pass (twice the oracle's own reorder error at 24 layers)."""
    import os
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "conditioning.npz")
    with np.load(path, allow_pickle=False) as z:
        bar = 2 * float(z["fixed_24"].max())
    cfg = ne.config_preset("gpt-oss-20b", max_seq=512)
    prompt = [[(1009 * i + 17) % 201088 for i in range(300)]]
    rel, _ = compare_modes(cfg, 0, prompt, 16, fixed_routing=True, bar=bar, mode=ne.PREFILL_MX8)
    assert rel < bar


def test_mx8_validation(orc):
    """The kernel-level MXFP8 expert FFN needs H and I multiples of 64 (the
    64-deep steps of the scaled instruction); the mode itself is accepted by
    every context (whose widths are multiples of 64)."""
    torch_cuda()
    M, E, H, I, k = 5, 4, 288, 352, 2
    d = moe_weights(orc, E, H, I, seed=3)
    dv = {n: to_dev(v) for n, v in d.items()}
    x = to_dev(orc.fill_bf16(3, 51, M * H, 0.0, 1.0))
    idx = to_dev(np.zeros((M, k), np.int32))
    sc = to_dev(np.full((M, k), 0.5, np.float32))
    h = to_dev(np.zeros((M, H), np.uint16))
    with pytest.raises(ne.NeonError) as e:
        ne.moe_prefill_mx8(x, idx, sc, dv["guc"], dv["gus"], dv["gub"], dv["dnc"], dv["dns"],
                           dv["dnb"], h, M, E, H, I, k)
    assert e.value.status == ne.NEON_EINVAL
    cfg = ne.config_preset("gpt-oss-20b", **dict(SMALL, max_seq=16))
    eng = ne.Engine(cfg)
    eng.set_prefill_mode(ne.PREFILL_MX8)
    eng.close()
