"""Paged decode attention at the edges of its routes: block tables up to 44
(64, from 128 units) pages (one workgroup per sequence and kv head) against wider ones (stream-K),
and few sequences cut into few, many, the most and too many record slots."""
import numpy as np
import pytest
import torch

import llaisys_amd as L
import oracle
from paged_cases import make_case, queries
from utils import from_bits, to_llaisys, to_torch

pytestmark = pytest.mark.gpu

SCALE = 1.0 / 128**0.5


def run(case, q, dtype, fn=L.Ops.paged_attention, fill=0.0, ctx=None):
    kp, vp = case.device_pools()
    table, lens = case.device_meta()
    out = to_llaisys(torch.full((case.B, case.nh, 128), fill, dtype=dtype, device="cuda"))
    fn(out, to_llaisys(from_bits(q)), kp, vp, table, lens if ctx is None else to_llaisys(torch.from_numpy(ctx)), SCALE)
    return to_torch(out).float().cpu().numpy()


def check(case, fn=L.Ops.paged_attention):
    q = queries(5, case.B, case.nh)
    ref = oracle.paged_attention(q, case.k_log, case.v_log, case.table, case.ctx, SCALE, nthreads=8)
    # weights to 2^-17 and 32-bit sums; bf16 also rounds its output (2^-9 of values up to ~4)
    assert np.max(np.abs(run(case, q, torch.float32, fn) - ref)) <= 1e-4 * np.max(np.abs(ref))
    assert np.max(np.abs(run(case, q, torch.bfloat16, fn) - ref)) <= 2e-2
    assert L.device_error_flags() == 0


# Pairs of pages per unit (32 tokens each) against slices of 1 to 64 pairs and
# 8 or 32 slots: 25 pairs over slices of 3, 31 x 3 pairs, 31 x 4 and one more,
# the longest that 32 slots hold (31 x 64 pairs) and past it.
@pytest.mark.parametrize("tokens", [785, 31 * 3 * 32, 31 * 4 * 32, 31 * 4 * 32 + 1, 31 * 64 * 32, 33 * 64 * 32 - 5])
@pytest.mark.parametrize("fn", [L.Ops.paged_attention, L.Ops.paged_attention_no_alloc], ids=["slots", "no_alloc"])
def test_one_long_sequence(tokens, fn):
    check(make_case(tokens, np.array([tokens], np.int32)), fn)


# 2-norm of the error. bf16: the result's own rounding (1.65e-3 for values spread
# over their exponents) and a tenth for the weights' two parts; with one part
# 2.0e-3 to 2.4e-3. f32: sums in 32 bits (about 2^-21); with two parts 1.7e-6 and more.
@pytest.mark.parametrize("lens", [[700], [300], [4000], [200, 450, 700], [100] * 40 + [800] * 30])
def test_weights_do_not_show(lens):
    case = make_case(8, np.array(lens, np.int32))
    q = queries(5, case.B, case.nh)
    ref = np.empty(q.shape)  # in 64 bits (the oracle's own 32-bit sums are off by 1.3e-6 at 4000 tokens)
    for b, n in enumerate(lens):
        k, v = (from_bits(log[case.table[b, :(n + 15) // 16]].swapaxes(1, 2).reshape(-1, case.nkvh, 128)[:n]).double().cpu()
                for log in (case.k_log, case.v_log))
        for h in range(case.nh):
            w = torch.softmax(k[:, h // 6] @ from_bits(q[b, h]).double().cpu() * SCALE, 0)
            ref[b, h] = (w @ v[:, h // 6]).numpy()
    for dtype, most in ((torch.bfloat16, 1.8e-3), (torch.float32, 2.0**-20)):
        assert np.linalg.norm(run(case, q, dtype) - ref) < most * np.linalg.norm(ref), dtype


def test_a_long_sequence_among_short_ones():
    check(make_case(3, np.array([3, 900, 17, 20000, 33, 1, 64, 2500], np.int32)))


def test_more_units_than_many_slots_serve():
    ctx = oracle.randint(4, 257, 1, 300).astype(np.int32)
    ctx[100] = 9000  # cut finer than 8 slots
    check(make_case(6, ctx))


@pytest.mark.parametrize("batch", [7, 65])
@pytest.mark.parametrize("width", [43, 44, 45, 47, 48, 49, 64, 65])
@pytest.mark.parametrize("fn", [L.Ops.paged_attention, L.Ops.paged_attention_no_alloc], ids=["", "no_alloc"])
def test_table_widths_around_the_line(width, batch, fn):
    lens = np.array([16 * width, 1, 31, 16 * width - 15, 32, 33, 500] + [9] * (batch - 7), np.int32)
    case = make_case(width, lens, nh=8, nkvh=2)
    assert case.table.shape[1] == width
    check(case, fn)


@pytest.mark.parametrize("width", [20, 60])
def test_invalid_lengths_leave_their_rows_alone(width):
    case = make_case(9, np.array([16 * width, 40, 7], np.int32))
    q = queries(5, 3, 12)
    lens = np.array([16 * width, 16 * width + 1, 0], np.int32)
    got = run(case, q, torch.bfloat16, fill=3.0, ctx=lens)
    assert L.device_error_flags() == 2
    assert (got[1:] == 3.0).all() and not (got[0] == 3.0).all()
