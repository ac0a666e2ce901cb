"""The exact experts and prompt passes on the fp32 matrix instructions: the
same bits as the one-row kernels, which the oracle tests pin."""
import pytest

import neonengine_amd as ne
from tests.gpu_util import torch_cuda

pytestmark = pytest.mark.gpu


def _experts(torch, B, E, H, I, k, seed, special):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def bf(*shape, std=1.0):
        return (std * torch.randn(shape, generator=g, device="cuda")).to(torch.bfloat16)

    def by(n, lo, hi):
        return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=torch.uint8)

    w = dict(guc=by(E * I * H, 0, 256), gus=by(E * 2 * I * H // 32, 117, 123), gub=bf(E, 2 * I),
             dnc=by(E * H * I // 2, 0, 256), dns=by(E * H * I // 32, 117, 123), dnb=bf(E, H))
    x, h = bf(B, H), bf(B, H)
    idx = torch.stack([torch.randperm(E, generator=g, device="cuda")[:k] for _ in range(B)])
    score = torch.softmax(torch.randn((B, k), generator=g, device="cuda"), dim=1)
    if special:  # NaN and extreme scales, an infinite and a subnormal input, a dropped slot
        w["gus"][5], w["gus"][77], w["dns"][9], w["dns"][40] = 255, 0, 255, 254
        x[0, 3], x[B - 1, H - 1], x[1, 0] = float("inf"), 1e-39, -0.0
        idx[B // 2, 0] = E + 3
    return w, x, h, idx.to(torch.int32).contiguous(), score.contiguous()


def _run(torch, w, x, h, idx, score, E, H, I, k):
    B = x.shape[0]
    out = torch.empty_like(h)
    act = torch.empty(B * k * I, dtype=torch.bfloat16, device="cuda")
    ne.moe_experts(x, idx, score, w["guc"], w["gus"], w["gub"], w["dnc"], w["dns"], w["dnb"], h,
                   out, act, B, E, H, I, k)
    return out


@pytest.mark.parametrize("B,E,H,I,k,special", [
    (2, 2, 32, 32, 2, False),       # one unit per row, one group
    (5, 3, 544, 96, 2, True),       # 17 units: a group of one; 3 units
    (12, 8, 1024, 2048, 4, False),  # whole groups of 16 units, 2 and 4 groups
    (16, 32, 2880, 2880, 4, True),  # the 20b shape
    (33, 16, 3104, 1056, 4, False), # 97 and 33 units: the first unit past 64, past 32
    (80, 4, 4096, 480, 4, True),    # 8 groups, 15 units; 20 quads of pairs per expert
    (320, 6, 64, 160, 4, False),    # the most pairs (1280)
    # matrix form, as above but with enough column blocks to take it
    (80, 256, 32, 32, 16, False),   # one unit per row; 256 experts, 1280 pairs
    (160, 128, 544, 96, 4, True),   # 17 and 3 units
    (46, 32, 4096, 480, 4, True),   # 8 groups, 15 units
    (20, 8, 96, 2080, 4, True),     # 65 units of I: 5 groups run as 6
    (16, 8, 320, 3104, 4, False),   # 97 units of I: 7 groups run as 8
    (12, 32, 2880, 2880, 4, False), # the fewest rows of the 20b shape
    (8, 8, 2880, 2880, 4, True),    # the fewest pairs: 32 of 40 column blocks
    # grouped form
    (9, 32, 2880, 2880, 4, True),
    (11, 32, 2880, 2880, 4, False),
    (10, 8, 4128, 2880, 4, True),   # rows of 129 units: past the matrix form's
    (16, 8, 2880, 4128, 4, False),
])
def test_experts_batch_bits(B, E, H, I, k, special):
    """Rows that share experts against the same rows one at a time: pair by pair,
    grouped on the vector units or on the matrix instructions, as the sizes say."""
    torch = torch_cuda()
    print(f"moe_experts B={B} E={E} H={H} I={I} k={k} special={special}", flush=True)
    w, x, h, idx, score = _experts(torch, B, E, H, I, k, 7 * B + E, special)
    got = _run(torch, w, x, h, idx, score, E, H, I, k)
    ref = torch.cat([_run(torch, w, x[b:b + 1], h[b:b + 1], idx[b:b + 1], score[b:b + 1], E, H, I, k)
                     for b in range(B)])
    if special:
        with pytest.raises(ne.NeonError):
            ne.device_check()
    same = (got.view(torch.int16) == ref.view(torch.int16)) | (got.isnan() & ref.isnan())
    assert bool(same.all()), int((~same).sum())


@pytest.mark.parametrize("B", [11, 12, 13, 16])
def test_experts_alike_bits(B):
    """Every row on the same four experts, on both sides of the line between the
    grouped and the matrix form."""
    torch = torch_cuda()
    E, H, I, k = 32, 2880, 2880, 4
    print(f"moe_experts alike B={B}", flush=True)
    w, x, h, idx, score = _experts(torch, B, E, H, I, k, B, False)
    idx = idx[:1].expand(B, k).contiguous()
    got = _run(torch, w, x, h, idx, score, E, H, I, k)
    ref = torch.cat([_run(torch, w, x[b:b + 1], h[b:b + 1], idx[b:b + 1], score[b:b + 1], E, H, I, k)
                     for b in range(B)])
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("B", [8, 9, 11, 12])
def test_engine_batch_rows_bits(B):
    """Decode steps of the 20b layer shape at the batches where the experts change
    form (pair by pair, grouped, matrix): each row's logits are those of the
    sequence decoding alone; half of the rows are alike."""
    torch_cuda()
    print(f"engine rows B={B}", flush=True)
    cfg = ne.config_preset("gpt-oss-20b", n_layers=2, vocab=2048, max_seq=64, max_batch=12)
    eng = ne.Engine(cfg)
    eng.init_random(9)
    prompts = [[(31 * i + 17 * (b // 2 if b % 4 < 2 else b) + 3) % 2048 for i in range(4)]
               for b in range(B)]
    eng.prefill(prompts)
    eng.decode(3)
    got = eng.read_logits()
    for b in range(0, B, 3):
        eng.prefill([prompts[b]])
        eng.decode(3)
        assert eng.read_logits()[0].tobytes() == got[b].tobytes(), b
    eng.close()


SMALL = dict(n_layers=2, hidden=512, n_heads=16, n_kv_heads=2, head_dim=64, n_experts=8, top_k=4,
             intermediate=512, vocab=1024, sliding_window=128, max_seq=768, max_batch=4)


@pytest.mark.parametrize("lens,over", [
    ([25], {}),                                    # 24 rows: passes of 16 and 8
    ([49], {}),                                    # 48 rows: the most by 16
    ([50], {}),                                    # 49 rows: the fewest of a wide pass
    ([145], {}),                                   # a second attention launch of 16 rows
    ([530], {}),                                   # a pass of 512 rows, then 17 by 16s; ring wraps
    ([562], {}),                                   # a pass of 512 rows, then a wide one of 49
    ([40, 3, 1, 90], {}),                          # several sequences in one pass
    ([200], dict(sliding_window=40)),              # ring of 64 rows: 24 rows per attention launch
    ([70], dict(hidden=192, intermediate=320)),    # 6 and 10 units: short rows, empty chains
    ([70], dict(hidden=2112, intermediate=2176, n_experts=4)),  # 66 and 68 units: second passes
    ([60], dict(n_experts=1, top_k=1, sliding_window=0)),       # one expert, every layer full
])
def test_prompt_passes_bits(lens, over):
    """Prompt rows many at a time against every token as a step of its own:
    the same logits after the prompt and after four more steps."""
    torch_cuda()
    print(f"prompt passes lens={lens} {over}", flush=True)
    cfg = ne.config_preset("gpt-oss-20b", **dict(SMALL, **over))
    prompts = [[(37 * i + 11 * b + 5) % 1024 for i in range(n)] for b, n in enumerate(lens)]
    got = []
    for mode in (ne.PREFILL_CHUNKED, ne.PREFILL_STEPWISE):
        eng = ne.Engine(cfg)
        eng.init_random(5)
        eng.set_prefill_mode(mode)
        eng.prefill(prompts)
        first = eng.read_logits()
        eng.decode(4)
        got.append((first, eng.read_logits(), eng.read_tokens()))
        eng.close()
    for a, b in zip(*got):
        assert a.tobytes() == b.tobytes()


@pytest.mark.parametrize("B,Hq,Hkv,T,window", [
    (64, 8, 8, 130, 0),    # one query head per kv head, one split of up to 3 chunks
    (72, 16, 8, 64, 0),    # two heads; one chunk
    (33, 16, 4, 700, 0),   # four heads, 11 splits of one chunk, most of them empty early on
    (5, 64, 8, 2200, 0),   # 32 splits of one or two chunks
    (20, 64, 8, 300, 77),  # windows that start inside a chunk
    # the matrix form with fewer heads per kv head than columns are made for
    (64, 8, 8, 700, 0),    # one head, 11 splits
    (128, 16, 8, 64, 0),   # two heads, one split of one chunk
    (48, 16, 4, 700, 0),   # four heads, 11 splits
    (36, 16, 4, 200, 130), # four heads, one split, windows of up to 3 chunks
    (16, 16, 4, 3000, 0),  # four heads, 32 splits of one or two chunks
])
def test_attention_batch_bits(B, Hq, Hkv, T, window):
    """Batches large enough for the matrix form against one row at a time, with
    positions at the ends of chunks and rows past them that hold NaN."""
    torch = torch_cuda()
    print(f"attention B={B} Hq={Hq} Hkv={Hkv} T={T} window={window}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B + T)

    def bf(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)

    q, k, v, sinks = bf(B, Hq * 64), bf(B, Hkv, T, 64), bf(B, Hkv, T, 64), bf(Hq)
    ends = [0, 1, 62, 63, 64, 65, 127, 128, T - 1, T // 2]
    pos = [min(ends[b % len(ends)] + 64 * (b // len(ends)), T - 1) for b in range(B)]
    for b, p in enumerate(pos):
        k[b, :, p + 1:], v[b, :, p + 1:] = float("nan"), float("nan")
    v[1, 0, 0, 5], k[2, 0, 0, 7] = float("inf"), float("nan")
    pt = torch.tensor(pos, dtype=torch.int32, device="cuda")

    def run(lo, hi):
        out = torch.empty((hi - lo, Hq * 64), dtype=torch.bfloat16, device="cuda")
        ne.attn_decode(q[lo:hi], k[lo:hi], v[lo:hi], sinks, pt[lo:hi].contiguous(), out, hi - lo,
                       Hq, Hkv, 64, T, window)
        return out

    got, ref = run(0, B), torch.cat([run(b, b + 1) for b in range(B)])
    same = (got.view(torch.int16) == ref.view(torch.int16)) | (got.isnan() & ref.isnan())
    assert bool(same.all()), int((~same).sum())


@pytest.mark.parametrize("V,T,p", [(1, 1.0, 0.9), (1000, 0.7, 0.9), (66560, 1.3, 0.999),
                                   (70001, 0.5, 1.0), (201088, 0.8, 0.95)])
def test_sampling_rows_alike(V, T, p):
    """A batch draws the same ids twice, its first row (the draw's key holds the
    row) the id that it draws alone, and equal logits (every value at the
    threshold) stay in range."""
    torch = torch_cuda()
    print(f"sampling V={V} T={T} top_p={p}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(V)
    lg = 3 * torch.randn((3, V), generator=g, device="cuda")
    lg[2] = 0.25
    pos = torch.tensor([5, 6, 7], dtype=torch.int32, device="cuda")
    out, again = torch.empty_like(pos), torch.empty_like(pos)
    ne.sample_logits(lg, 3, V, T, p, 11, pos, out)
    ne.sample_logits(lg, 3, V, T, p, 11, pos, again)
    assert out.tolist() == again.tolist() and all(0 <= i < V for i in out.tolist())
    one = torch.empty(1, dtype=torch.int32, device="cuda")
    ne.sample_logits(lg[:1].contiguous(), 1, V, T, p, 11, pos[:1].contiguous(), one)
    assert one.item() == out[0].item()
