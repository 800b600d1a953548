"""llaisysLinear with few rows (the kernel that streams W once) at the edges of
its row groups, segments and dispatch, against float64."""
import pytest
import torch

import llaisys_amd as L
from utils import to_llaisys, to_torch

pytestmark = pytest.mark.gpu

TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def check(M, N, K, dtype, bias=True, off=0):
    g = torch.Generator(device="cuda").manual_seed(M * 7919 + N * 31 + K)
    t = TYPES[dtype]
    x = torch.randn(M, K, generator=g, device="cuda").to(t)
    w = torch.randn(N, K, generator=g, device="cuda").to(t)
    b = torch.randn(N, generator=g, device="cuda").to(t) if bias else None
    y = to_llaisys(torch.full((M, N), float("nan"), dtype=t, device="cuda"))
    lx = to_llaisys(x)
    if off:  # contiguous, but not on a 16 B boundary
        lx = to_llaisys(torch.cat([x.new_zeros(off), x.flatten()])).slice(0, off, off + x.numel()).view(M, K)
    L.Ops.linear(y, lx, to_llaisys(w), to_llaisys(b) if bias else None)
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    # the type's half ulp, and 32-bit sums of K products in any order: each
    # addition rounds to 2^-24 of a partial sum below sum |x w|
    half = {"f32": 2.0**-24, "f16": 2.0**-11, "bf16": 2.0**-8}[dtype]
    terms = x.double().abs() @ w.double().abs().t() + 1
    assert torch.all((to_torch(y).double() - want).abs() <= half * want.abs() + 2.0**-24 * (K / 8 + 16) * terms)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("N,K", [(1, 8), (7, 72), (250, 1000), (1537, 1536)])
def test_rows_and_widths(M, N, K, dtype):
    check(M, N, K, dtype, bias=M % 2 == 1)


# both sides of the dispatch's lines, and a long K
@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("M,N,K", [(1, 4099, 8960), (3, 64, 16384), (8, 4096, 1024), (8, 4097, 1024), (16, 2048, 2048),
                                   (16, 2056, 2048), (16, 128, 4096), (16, 128, 4104), (32, 4096, 1024), (32, 4096, 1032),
                                   (2, 4104, 1016), (2, 4104, 1024), (4, 4096, 4088), (4, 4096, 4096), (4, 2056, 504),
                                   (4, 2056, 512), (8, 70, 8192), (8, 70, 8200), (16, 70, 3072), (16, 70, 3080),
                                   (32, 70, 2048), (32, 70, 2056)])
def test_around_the_dispatch(M, N, K, dtype):
    check(M, N, K, dtype)


def test_a_single_piece_of_k():
    check(3, 5, 8, "f32", bias=False)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_unaligned_rows_keep_the_tiles(dtype):
    check(2, 300, 512, dtype, off=1)


def test_what_lies_in_other_rows_stays_there():
    # rows of X and W that share an MFMA with others: a NaN reaches only its own outputs
    x = torch.ones(2, 512, device="cuda")
    w = torch.ones(9, 512, device="cuda")
    x[1, 300] = float("nan")
    w[5, 7] = float("inf")
    y = to_llaisys(torch.zeros(2, 9, device="cuda"))
    L.Ops.linear(y, to_llaisys(x), to_llaisys(w), None)
    got = to_torch(y)
    assert torch.isnan(got[1]).all() and got[0, 5] == float("inf")
    assert (got[0, [0, 1, 2, 3, 4, 6, 7, 8]] == 512).all()
