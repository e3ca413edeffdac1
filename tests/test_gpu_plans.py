"""The forward's key-split workgroups and head-dim instances at the sizes where they can go wrong:
ends of 32-key halves, 64-key tiles and query blocks, groups without a tile, head dims at the edges
of the compiled ones (needs a GPU).

Reference: float32 attention from the same 16-bit values.  With u the unit roundoff of the type
(2^-8 bf16, 2^-11 fp16), the probabilities, their sum and the output are each rounded once:
|dO| <= 3 u max|V|.  The LSE is float32 throughout: scores of magnitude up to 2^6 carry about
sqrt(D) roundings of 2^-24, below 1e-4.
"""
import math

import pytest
import torch

import custom_flash_attn

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}

# The kernel each (B, H, Nq, Nk, causal) reaches on 256 CUs (checked in test_plan_cpu.py).
NARROW_PLANS = {  # head dims up to 64
    "kGroups4": [                  # 2 row waves x 4 key groups
        (1, 1, 1025, 1025, True),  # one row past a block
        (1, 2, 33, 1100, False),   # unmasked, a ragged last tile
        (1, 1, 1300, 1090, True),  # rows past the last key
        (1, 256, 5, 1100, False),
    ],
    "kPairs": [                    # 2 x 2: a causal call's first block has one tile, its second group none
        (1, 100, 200, 200, True),
        (1, 60, 321, 500, True),
        (1, 21, 1153, 1153, True),
    ],
    "kGroups2": [                  # 4 x 2
        (1, 150, 127, 1056, False),
        (1, 20, 2049, 2049, True),
    ],
    "kHalves": [                   # 32-row blocks, 4 key waves
        (1, 130, 1, 1, True),      # one row, one key
        (1, 131, 65, 65, True),
        (1, 40, 97, 130, False),
        (1, 25, 700, 700, True),   # more than one round
    ],
    "kWhole": [
        (1, 256, 65, 1, True),
        (1, 130, 100, 100, True),
        (1, 200, 96, 96, True),
        (2, 65, 127, 127, True),
        (1, 60, 640, 640, True),
        (1, 44, 641, 641, True),
    ],
}
WIDE_PLANS = {  # head dims past 64
    "kHalves": [
        (1, 3, 130, 130, True),
        (1, 70, 65, 65, True),
        (1, 200, 3, 705, False),
    ],
    "kPairs": [
        (1, 20, 703, 703, True),
        (1, 180, 34, 300, False),
        (1, 150, 64, 993, False),
    ],
    "kGroups2": [
        (1, 35, 700, 700, True),
        (1, 200, 100, 705, False),
        (1, 20, 2049, 2049, True),
    ],
    "kWhole": [
        (1, 180, 34, 34, True),
        (1, 140, 33, 65, True),
        (1, 192, 65, 33, True),
        (1, 25, 600, 97, True),
        (1, 130, 200, 130, False),
    ],
}
NARROW = [s for shapes in NARROW_PLANS.values() for s in shapes]
WIDE = [s for shapes in WIDE_PLANS.values() for s in shapes]


def _reference(q, k, v, causal):
    if q.dtype != torch.float64:
        q, k, v = q.float(), k.float(), v.float()
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        s.masked_fill_(torch.ones(s.shape[-2:], dtype=torch.bool, device=DEV).triu(1), -math.inf)
    return torch.matmul(torch.softmax(s, -1), v), torch.logsumexp(s, -1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("D", [8, 32, 40, 64, 72, 96, 104, 128])
def test_every_plan_and_head_dim(D, dtype):
    for B, H, Nq, Nk, causal in (NARROW if D <= 64 else WIDE):
        print(f"D={D} {dtype} B={B} H={H} Nq={Nq} Nk={Nk} causal={causal}", flush=True)
        g = torch.Generator(device=DEV).manual_seed(Nq * 7 + Nk + D)
        q, k, v = (torch.randn((B, n, H, D), device=DEV, generator=g).to(dtype).transpose(1, 2)
                   for n in (Nq, Nk, Nk))
        q = q * 2
        buf = torch.full((B, Nq, H, D + 8), 1000.0, dtype=dtype, device=DEV)
        o, lse = custom_flash_attn.attention(q, k, v, out=buf[..., :D].transpose(1, 2), causal=causal,
                                             return_lse=True)
        o_ref, lse_ref = _reference(q, k, v, causal)
        assert (o.float() - o_ref).abs().max().item() <= 3 * U[dtype] * v.abs().max().item()
        assert (lse - lse_ref).abs().max().item() <= 1e-4
        assert torch.equal(buf[..., D:], torch.full_like(buf[..., D:], 1000.0))
        # Without the LSE, and from contiguous copies: the same arithmetic, bit for bit.
        assert torch.equal(custom_flash_attn.attention(q, k, v, causal=causal), o)
        c = custom_flash_attn.attention(q.contiguous(), k.contiguous(), v.contiguous(), causal=causal)
        assert torch.equal(c, o)


@pytest.mark.parametrize("B,H,N", [(1, 4, 1500), (2, 16, 777), (1, 25, 2048)])
def test_key_groups_merge_extreme_rows(B, H, N):
    """Rows whose keys differ by hundreds between groups (one group's weight is 0), rows of equal
    scores, and in the first head values near the largest that O is finite for (max|V| < 2^62): the
    float32 partials and their merge keep the relative accuracy of ordinary ones."""
    g = torch.Generator(device=DEV).manual_seed(N)
    q, k, v = (torch.randn((B, H, N, 64), device=DEV, generator=g).to(torch.bfloat16) for _ in range(3))
    q[:, :, ::3] = 0
    k[:, :, 64:96] *= 40
    v[:, 0] *= 2.0 ** 55
    o, lse = custom_flash_attn.forward_lse(q, k, v)
    o_ref, lse_ref = _reference(q, k, v, True)
    for part in (slice(0, 1), slice(1, None)):
        err = (o[:, part].float() - o_ref[:, part]).abs().max().item()
        assert err <= 3 * U[torch.bfloat16] * v[:, part].abs().max().item()
    assert ((lse - lse_ref).abs() <= 1e-4 + 1e-5 * lse_ref.abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kind", ["rising", "falling", "zigzag halves", "zigzag tiles"])
def test_offset_moves_inside_key_groups(kind, dtype):
    """Scores that climb past the offset's margin in every half, fall, or alternate by +-40 between a
    group's halves or between the groups, at shapes of each key-group kernel.  Against float64.  Scores of
    magnitude up to `span` are rounded to 2^-24 of it by each of the D / 16 accumulating MFMAs of the dot
    product and four times after it (times the scale, less the offset, plus log2 of the sum, times ln 2),
    so the LSE, and each probability relatively, is off by up to (D / 16 + 4) span 2^-24."""
    for D, plans in ((64, NARROW_PLANS), (128, WIDE_PLANS)):
        for plan, group in plans.items():
            for B, H, Nq, Nk, causal in (group if "Groups" in plan or plan == "kPairs" else ()):
                print(f"{kind} D={D} {dtype} {plan} H={H} Nq={Nq} Nk={Nk} causal={causal}", flush=True)
                g = torch.Generator(device=DEV).manual_seed(Nq + Nk + D)
                q, k, v = (torch.randn((B, H, n, D), device=DEV, generator=g) for n in (Nq, Nk, Nk))
                j = torch.arange(Nk, device=DEV)
                rise = 0.75 * (j if kind == "rising" else Nk - j)
                sign = 1.0 - 2.0 * ((j // (32 if kind == "zigzag halves" else 64)) % 2)
                q, k = 0.1 * q, 0.1 * k
                q[..., 0] = 8.0
                k[..., 0] += (rise if kind in ("rising", "falling") else 40.0 * sign) * math.sqrt(D) / 8
                q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
                o, lse = custom_flash_attn.attention(q, k, v, causal=causal, return_lse=True)
                assert torch.equal(custom_flash_attn.attention(q, k, v, causal=causal), o)
                pick = sorted({0, H // 2, H - 1})
                o_ref, lse_ref = _reference(*(t[:, pick].double() for t in (q, k, v)), causal)
                span = lse_ref.abs().max().item() + 40
                rounding = (D / 16 + 4) * span * 2.0 ** -24
                err = (o[:, pick].double() - o_ref).abs().max().item()
                assert err <= (3 * U[dtype] + 2 * rounding) * v[:, pick].abs().max().item()
                assert (lse[:, pick] - lse_ref).abs().max().item() <= 1e-4 + rounding


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("D", [64, 128])
def test_first_scores_of_minus_infinity(D, dtype):
    """Keys of infinite magnitude and opposite sign score -inf and drop out of a row, also where they
    are all a wave's or a key group's first half or tile holds.  A row of nothing else is NaN."""
    for B, H, Nq, Nk, causal in (NARROW if D == 64 else WIDE):
        if Nk < 600:
            continue
        for width, period in ((32, 64), (64, 256), (256, Nk)):  # first halves, first tiles, the first four tiles
            print(f"D={D} {dtype} H={H} Nq={Nq} Nk={Nk} causal={causal} {width} of {period}", flush=True)
            g = torch.Generator(device=DEV).manual_seed(Nq + Nk + period)
            q, k, v = (torch.randn((B, H, n, D), device=DEV, generator=g).to(dtype) for n in (Nq, Nk, Nk))
            q[..., 0] = -1
            k[:, :, torch.arange(Nk, device=DEV) % period < width, 0] = math.inf
            o, lse = custom_flash_attn.attention(q, k, v, causal=causal, return_lse=True)
            assert torch.equal(custom_flash_attn.attention(q, k, v, causal=causal).isnan(), o.isnan())
            o_ref, lse_ref = _reference(q, k, v, causal)
            seen = lse_ref > -math.inf
            assert torch.equal(seen, ~o.isnan().any(-1)) and torch.equal(seen, ~o.isnan().all(-1))
            assert (o.float() - o_ref)[seen].abs().max().item() <= 3 * U[dtype] * v.abs().max().item()
            assert (lse - lse_ref)[seen].abs().max().item() <= 1e-4
            assert (lse[~seen] == -math.inf).all()
