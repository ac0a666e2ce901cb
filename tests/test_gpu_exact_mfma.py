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
])
def test_experts_batch_bits(B, E, H, I, k, special):
    """Rows that share experts against the same rows one at a time."""
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
