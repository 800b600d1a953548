"""llaisysLinear where the tiled GEMM's k is cut in numbers that do not divide
it, and with the three-stage rings of the 128 x 256 tiles at few k tiles,
against float64."""
import pytest
import torch

import llaisys_amd as L
from utils import to_llaisys, to_torch

pytestmark = pytest.mark.gpu

TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("M,N,K", [
    (40, 256, 1544),    # 25 k tiles of 64, the last of 8
    (130, 1536, 2824),  # 45 k tiles in several uneven parts
    (257, 1000, 4104),
    (777, 1536, 3080),  # 16-bit: 128 x 128 tiles, three parts
    (300, 8968, 64),    # one k tile, fewer than the ring's stages
    (300, 8968, 136),   # two and a piece
    (200, 17928, 264),  # 128 x 256 or 256 x 128 tiles
])
def test_uneven_k(M, N, K, dtype):
    t = TYPES[dtype]
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").to(t)
    w = torch.randn(N, K, generator=g, device="cuda").to(t)
    b = torch.randn(N, generator=g, device="cuda").to(t)
    y = to_llaisys(torch.full((M, N), float("nan"), dtype=t, device="cuda"))
    L.Ops.linear(y, to_llaisys(x), to_llaisys(w), to_llaisys(b))
    want = x.double() @ w.double().t() + b.double()
    half = {"f32": 2.0**-24, "f16": 2.0**-11, "bf16": 2.0**-8}[dtype]  # half an ulp of the result
    # 32-bit sums of K products in any order, each addition 2^-24 of a partial sum
    terms = x.double().abs() @ w.double().abs().t() + 1
    assert torch.all((to_torch(y).double() - want).abs() <= half * want.abs() + 2.0**-24 * (K / 8 + 16) * terms)
