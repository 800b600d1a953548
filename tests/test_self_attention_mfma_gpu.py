"""The matrix-core kernels of llaisysSelfAttention (head dims 64 and 128) at the
edges of their tiles, stages and key splits, against a float64 statement of
test/ops/self_attention.py:11-28, and the calls that keep the general kernel."""
import math

import pytest
import torch

import llaisys_amd as L
from utils import to_llaisys, to_torch

pytestmark = pytest.mark.gpu

TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def exact(q, k, v, scale):
    """Each query over the keys it may see, in float64."""
    Lq, nh, _ = q.shape
    S, nkvh = k.shape[:2]
    q, k, v = q.double(), k.double(), v.double()
    out = torch.empty(Lq, nh, v.shape[2], dtype=torch.float64, device=q.device)
    for i in range(Lq):
        n = i + S - Lq + 1
        for h in range(nh):
            kh = h // (nh // nkvh)
            p = torch.softmax(k[:n, kh] @ q[i, h] * scale, 0)
            out[i, h] = (p[:, None] * v[:n, kh]).sum(0)
    return out


def inputs(Lq, S, nh, nkvh, d, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + 31 * Lq + S)
    return [torch.randn(s, generator=g, device="cuda").to(dtype)
            for s in ((Lq, nh, d), (S, nkvh, d), (S, nkvh, d))]


def run(q, k, v, scale):
    out = to_llaisys(torch.full((q.shape[0], q.shape[1], v.shape[2]), float("nan"), dtype=q.dtype, device="cuda"))
    L.Ops.self_attention(out, to_llaisys(q), to_llaisys(k), to_llaisys(v), scale)
    return to_torch(out)


def check(got, want, v, dtype):
    """The output's own rounding (half an ulp), and 32-bit sums over values of
    max |v|: weights to 2^-17 (hi + lo halves of bf16) with room for the sums."""
    half_ulp = {torch.float32: 2.0**-24, torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}[dtype]
    slack = (2.0**-17 if dtype == torch.float32 else 2.0**-14) * float(v.float().abs().max())
    assert torch.all((got.double() - want).abs() <= half_ulp * want.abs() + slack)


# Columns = queries x heads per kv head: tiles of 16 to 128 columns with a
# remainder of one or all but one, stages of 64 to 256 keys likewise.
@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("Lq,S,nh,nkvh,d", [
    (1, 1, 12, 2, 128),       # one key
    (1, 33, 4, 4, 64),        # one column a tile
    (1, 257, 16, 1, 128),     # a full tile, a stage and a key
    (1, 1025, 12, 2, 128),    # five stages: the key splits begin
    (1, 5000, 8, 2, 64),      # the most splits
    (17, 17, 1, 1, 64),       # one column past a tile, no earlier keys
    (31, 300, 2, 1, 128),
    (43, 129, 12, 2, 128),    # 258 columns
    (350, 350, 12, 2, 128),   # tiles of 32 columns
])
def test_edges(Lq, S, nh, nkvh, d, dtype):
    q, k, v = inputs(Lq, S, nh, nkvh, d, TYPES[dtype])
    scale = 1 / math.sqrt(d)
    check(run(q, k, v, scale), exact(q, k, v, scale), v, TYPES[dtype])


def exact_head(q, k, v, h, scale):
    """Head h of every query, in float64."""
    Lq, S, kh = q.shape[0], k.shape[0], h // (q.shape[1] // k.shape[1])
    see = torch.arange(S, device="cuda")[None] <= torch.arange(Lq, device="cuda")[:, None] + S - Lq
    w = (q[:, h].double() @ k[:, kh].double().t().contiguous() * scale).masked_fill(~see, -math.inf)
    return torch.softmax(w, -1) @ v[:, kh].double().contiguous()


# The wide tiles need thousands of columns: 8622 take tiles of 64, 18000 of
# 128 (both with a remainder). A few heads of the result against float64.
WIDE = [(1437, 1500, 12, 2), (1500, 1501, 48, 4), (3000, 3131, 12, 2)]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("Lq,S,nh,nkvh", WIDE)
def test_wide_tiles(Lq, S, nh, nkvh, d, dtype):
    q, k, v = inputs(Lq, S, nh, nkvh, d, TYPES[dtype])
    scale = 1 / math.sqrt(d)
    got = run(q, k, v, scale)
    for h in (0, nh // 2, nh - 1):
        check(got[:, h], exact_head(q, k, v, h, scale), v, TYPES[dtype])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("Lq,S,nh,nkvh", WIDE[:2])
def test_wide_tiles_non_finite(Lq, S, nh, nkvh, d, dtype):
    q, k, v = inputs(Lq, S, nh, nkvh, d, TYPES[dtype])
    kb, vb = k.clone(), v.clone()
    kb[-2:], vb[-2:] = math.nan, math.nan  # only the last two queries see these
    vb[700, :, 9] = math.inf               # and only queries from there on this one
    got = run(q, kb, vb, 0.1)
    sees = torch.arange(Lq - 2, device="cuda") + S - Lq >= 700
    for h in (0, nh - 1):
        want = exact_head(q, k, v, h, 0.1)[:-2]
        assert torch.isnan(got[-2:, h]).all()
        assert (got[:-2, h, 9][sees] == math.inf).all()
        want[:, 9] = torch.where(sees, 0.0, want[:, 9])
        mine = got[:-2, h].clone()
        mine[:, 9] = torch.where(sees, torch.zeros_like(mine[:, 9]), mine[:, 9])
        check(mine, want, v, TYPES[dtype])


# Values of 2^118, whose sums with the lazy max's weights (up to
# 2^8) would leave f32's range: their average does not.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("Lq,S", [(1, 300), (350, 350), (1437, 1500)])
def test_huge_finite_values(Lq, S, dtype):
    q, k, v = inputs(Lq, S, 12, 2, 128, TYPES[dtype])
    k = k * torch.linspace(0.5, 3, S, device="cuda", dtype=k.dtype)[:, None, None]
    v = (1.0 + 0.01 * v.float().clamp(-3, 3)).mul(2.0**118).to(TYPES[dtype])
    got = run(q, k, v, 0.1)
    for h in (0, 7):
        check(got[:, h].float() / 2.0**118, exact_head(q, k, v, h, 0.1) / 2.0**118, v.float() / 2.0**118, TYPES[dtype])


# f32 sums are cut into short chains: 2-norm of the error at most 5 roundings
# of 2^-24 (measured 2.1e-7 to 2.5e-7; one running sum per score and per output
# gives 4.2e-7 to 5.2e-7 here).
@pytest.mark.parametrize("Lq,S,d", [(1, 513, 128), (1, 2000, 128), (64, 1000, 128), (512, 1536, 128), (512, 1536, 64)])
def test_f32_error(Lq, S, d):
    q, k, v = inputs(Lq, S, 12, 2, d, torch.float32)
    scale = 1 / math.sqrt(d)
    got = run(q, k, v, scale)
    want = torch.stack([exact_head(q, k, v, h, scale) for h in range(12)], 1)
    assert float((got.double() - want).norm() / want.norm()) < 5 * 2.0**-24


def test_scores_that_grow_and_large_scale():
    # every stage raises the running max by far more than the lazy bound
    q, k, v = inputs(20, 700, 12, 2, 128, torch.float32)
    k = k * torch.linspace(0.1, 6, 700, device="cuda")[:, None, None]
    check(run(q, k, v, 0.5), exact(q, k, v, 0.5), v, torch.float32)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("Lq,S", [(40, 40), (3, 1500), (350, 350)])
def test_values_past_a_query_do_not_reach_it(Lq, S, dtype):
    q, k, v = inputs(Lq, S, 12, 2, 128, TYPES[dtype])
    for bad in (math.nan, math.inf):
        kb, vb = k.clone(), v.clone()
        kb[-2:], vb[-2:] = bad, bad
        got, clean = run(q, kb, vb, 0.1), exact(q, k, v, 0.1)
        check(got[:-2], clean[:-2], v, TYPES[dtype])
        assert torch.isnan(got[-1]).all()


# One key takes nearly all the weight and has a small value; 4000 others have
# 2^-gap of its weight each and values of 30000. Nothing of the sum may be lost
# to the range of the 16-bit type: dim 0 is their sum, dim 1 the large weight's
# own value. (S = 4001; L = 40 also runs tiles of more columns.)
@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("gap", [14.0, 17.5, 26.5, 34.0, 45.0, 70.0])
@pytest.mark.parametrize("Lq,d", [(1, 64), (40, 128)])
def test_small_weights_of_large_values(Lq, d, gap, dtype):
    t = TYPES[dtype]
    q = torch.zeros(Lq, 12, d, device="cuda", dtype=t)
    k, v = torch.zeros(4000 + Lq, 2, d, device="cuda", dtype=t), torch.zeros(4000 + Lq, 2, d, device="cuda", dtype=t)
    q[..., 0], k[1000, :, 0] = 8.0, gap / 8
    v[..., 0], v[1000, :, 0], v[1000, :, 1] = 30000.0, 0.0, 1.0
    scale = float(math.log(2.0))  # scores in powers of two
    got, want = run(q, k, v, scale), exact(q, k, v, scale)
    half_ulp = {torch.float32: 2.0**-24, torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}[t]
    # weights to 2^-16 of their own size; gap ulps of the exponent (|s| 2^-24, twice); f16's least step
    rel = half_ulp + (2.0**-16 if t != torch.float32 else 2.0**-18) + gap * 2.0**-23
    assert torch.all((got.double() - want).abs() <= rel * want.abs() + (2.0**-25 if t == torch.float16 else 0.0))


def test_infinite_value_that_is_seen():
    q, k, v = inputs(9, 300, 12, 2, 128, torch.bfloat16)
    v[5, 0, 7] = math.inf
    v[6, 1, 9] = -math.inf
    got = run(q, k, v, 0.05)
    assert (got[:, :6, 7] == math.inf).all() and (got[:, 6:, 9] == -math.inf).all()
    got[:, :6, 7], got[:, 6:, 9] = 0, 0
    assert torch.isfinite(got).all()


@pytest.mark.parametrize("scale", [-0.1, 0.0])
def test_scales_of_the_general_kernel(scale):
    q, k, v = inputs(7, 90, 12, 2, 128, torch.float32)
    check(run(q, k, v, scale), exact(q, k, v, scale), v, torch.float32)


def test_operands_off_alignment():
    # one element into a larger buffer: contiguous, not 16 B aligned
    q, k, v = inputs(5, 70, 4, 2, 64, torch.bfloat16)

    def off(t):
        flat = to_llaisys(torch.cat([torch.zeros(1, dtype=t.dtype, device="cuda"), t.flatten()]))
        return flat.slice(0, 1, t.numel() + 1).view(*t.shape)

    for which in range(3):
        ts = [off(t) if i == which else to_llaisys(t) for i, t in enumerate((q, k, v))]
        out = to_llaisys(torch.zeros_like(q))
        L.Ops.self_attention(out, *ts, 0.125)
        check(to_torch(out), exact(q, k, v, 0.125), v, torch.bfloat16)
