"""llaisysLinear in 32 bits: the error of its sums against float64."""
import pytest
import torch

import llaisys_amd as L
from utils import to_llaisys, to_torch

pytestmark = pytest.mark.gpu


# Random products: sums of 128 k at a time (or less), then of those, round about
# sqrt(32 + K / 128) times half an ulp of a partial sum. Measured 2.0e-7 to
# 4.0e-7 of the result's 2-norm; one running sum per split of K gives 3.6e-7 at
# 16 x 2048 x 1536, 5.7e-7 at 16 x 1000 x 4000 and 9.8e-7 at 400 x 1536 x 8960.
@pytest.mark.parametrize("M,N,K,most", [
    (9, 2048, 1536, 2.6e-7), (16, 256, 1536, 2.6e-7), (16, 300, 3000, 3.6e-7),  # few rows
    (17, 300, 1540, 2.6e-7), (100, 520, 132, 2.2e-7),                           # k tiles with a remainder
    (400, 1536, 8960, 6.0e-7), (1024, 1536, 1536, 3.0e-7), (300, 1000, 4000, 4.1e-7),
])
def test_error(M, N, K, most):
    g = torch.Generator(device="cuda").manual_seed(K + M)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    y = to_llaisys(torch.zeros(M, N, device="cuda"))
    L.Ops.linear(y, to_llaisys(x), to_llaisys(w), None)
    want = x.double() @ w.double().t()
    assert float((to_torch(y).double() - want).norm() / want.norm()) < most
