"""add, swiglu, rms_norm and rope where their 16 B pieces begin and end: sizes
around whole pieces, rows of one piece to past a wave's registers, operands off
16 B boundaries. Bit for bit where one rounding of one formula gives the result."""
import pytest
import torch

import llaisys_amd as L
from utils import to_llaisys, to_torch

pytestmark = pytest.mark.gpu

TYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def rnd(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda").to(TYPES[dtype])


def at_offset(t, off):
    flat = to_llaisys(torch.cat([t.new_zeros(off), t.flatten(), t.new_zeros(3)]))
    return flat.slice(0, off, off + t.numel()).view(*t.shape)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("n", [1, 3, 4, 7, 8, 9, 2047, 2048, 2049, 100003])
@pytest.mark.parametrize("off", [0, 1])
def test_add_and_swiglu(n, off, dtype):
    a, b = rnd((n,), dtype, 1), rnd((n,), dtype, 2)
    out = at_offset(torch.zeros_like(a), off)
    L.Ops.add(out, at_offset(a, off), to_llaisys(b))
    assert torch.equal(to_torch(out), (a.float() + b.float()).to(a.dtype))
    L.Ops.swiglu(out, to_llaisys(a), at_offset(b, off))
    want = b.double() * a.double() / (1 + torch.exp(-a.double()))
    ulp = {"f32": 2.0**-20, "f16": 2.0**-10, "bf16": 2.0**-7}[dtype]  # exp, division, the rounding
    torch.testing.assert_close(to_torch(out).double(), want, rtol=ulp, atol=1e-7)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("rows,d", [(1, 1), (3, 7), (5, 8), (2, 520), (9, 1536), (4, 2048), (3, 2052), (2, 4096),
                                    (2, 4104), (1, 10000), (1025, 8), (1027, 7),
                                    (1026, 520), (1030, 1536), (1025, 2052), (1026, 4096), (1025, 4104),
                                    # a wave per row from 2049 rows, long rows from 3073
                                    (2048, 8), (2049, 8), (2050, 520), (2051, 1536), (2049, 1024), (3072, 4096),
                                    (3073, 2052), (3074, 4096), (3073, 4104)])
@pytest.mark.parametrize("off", [0, 1])
def test_rms_norm(rows, d, off, dtype):
    x, w = rnd((rows, d), dtype, 3), rnd((d,), dtype, 4)
    out = to_llaisys(torch.zeros_like(x))
    L.Ops.rms_norm(out, at_offset(x, off), to_llaisys(w), 1e-6)
    x, w = x.double(), w.double()
    want = x * w * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)
    ulp = {"f32": 2.0**-19, "f16": 2.0**-10, "bf16": 2.0**-7}[dtype]  # sums of d squares, rsqrt, the rounding
    torch.testing.assert_close(to_torch(out).double(), want, rtol=ulp, atol=1e-7)


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("tokens,heads,d", [(1, 1, 2), (3, 5, 12), (7, 12, 128), (2, 40, 64), (2, 1, 1024), (2, 2, 1040),
                                            # around a wave of elements, and shared angles with ragged halves
                                            (4, 2, 64), (4, 2, 80), (3, 3, 44), (7, 12, 36), (2, 2, 1024), (3, 1, 128)])
@pytest.mark.parametrize("off", [0, 1])
def test_rope(tokens, heads, d, off, dtype):
    x = rnd((tokens, heads, d), dtype, 5)
    pos = torch.arange(tokens, device="cuda", dtype=torch.int64) * 17
    out = to_llaisys(torch.zeros_like(x))
    L.Ops.rope(out, at_offset(x, off), to_llaisys(pos), 10000.0)
    # the angle in 32 bits, as the formula is stated; pow's error (a few ulp) times the angle remains
    j = 2.0 * torch.arange(d // 2, dtype=torch.float32, device="cuda") / d
    phi = (pos.float()[:, None] / torch.pow(torch.tensor(10000.0, device="cuda"), j)).double()[:, None]
    a, b = x.double()[..., : d // 2], x.double()[..., d // 2:]
    want = torch.cat([a * phi.cos() - b * phi.sin(), b * phi.cos() + a * phi.sin()], -1)
    ulp = {"f32": 2.0**-22, "f16": 2.0**-11, "bf16": 2.0**-8}[dtype]
    size = x.double().abs().max()
    assert ((to_torch(out).double() - want).abs() <= 2 * ulp * size + 2.0**-21 * float(pos.max()) * size).all()
