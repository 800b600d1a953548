"""Varlen paged attention where the persistent kernel chooses its split size:
batches whose choice is the finest, in between and the coarsest, the lines of
the rule, and calls of different choices one after the other."""
import numpy as np
import pytest
import torch

import llaisys_amd as L
import oracle
from paged_cases import make_case, queries
from utils import from_bits, to_llaisys, to_torch

pytestmark = pytest.mark.gpu

SCALE = 1.0 / 128**0.5

# (new tokens, contexts) per sequence
BATCHES = {
    "one_prompt": ([520], [530]),                      # 34 pages: its queries alone show a long context
    "finest": ([64], [1100]),                          # 69 pages: one sequence
    "prompts": ([750, 20, 810], [750, 700, 1100]),
    "between": ([540, 540, 540], [1900, 560, 1700]),
    "decode_beside": ([1030, 1], [1100, 1500]),
    "decode_binds": ([1030, 1], [1100, 3600]),         # the decode's length keeps the splits longer
    "many_queries": ([700] * 3, [700, 1200, 1300]),
    # and some that keep splits of 64 pages
    "short_prompt": ([500], [530]),
    "few_queries": ([350, 20, 610], [350, 700, 610]),
    "with_decodes": ([40, 1, 1, 200, 1], [900, 3, 1500, 200, 64]),
    "short_tables": ([200, 7], [500, 512]),
}


def run(name, dtype):
    lq, ctx = BATCHES[name]
    case = make_case(len(name), np.array(ctx, np.int32))
    cu = np.concatenate([[0], np.cumsum(lq)]).astype(np.int32)
    q = queries(9, int(cu[-1]), 12)
    kp, vp = case.device_pools()
    table, lens = case.device_meta()
    out = to_llaisys(torch.full((int(cu[-1]), 12, 128), float("nan"), dtype=dtype, device="cuda"))
    L.Ops.paged_attention_varlen(out, to_llaisys(from_bits(q)), kp, vp, table, to_llaisys(torch.from_numpy(cu)), lens,
                                 SCALE)
    assert L.device_error_flags() == 0
    return case, q, cu, to_torch(out).float().cpu().numpy()


@pytest.mark.parametrize("name", list(BATCHES))
def test_against_the_oracle(name):
    case, q, cu, got32 = run(name, torch.float32)
    ref = oracle.paged_attention(q, case.k_log, case.v_log, case.table, case.ctx, SCALE, cu_q=cu, nthreads=8)
    # fp32: weights to 2^-17; bf16: weights, records and the output each rounded to 2^-9
    assert np.max(np.abs(got32 - ref)) <= 1e-4 * np.max(np.abs(ref))
    assert np.max(np.abs(run(name, torch.bfloat16)[3] - ref)) <= 2e-2


@pytest.mark.parametrize("name", ["finest", "between", "decode_beside"])
def test_without_the_queue(name, monkeypatch):
    # one workgroup per grid slot: splits of 64 pages for every batch
    monkeypatch.setenv("LLAISYS_PREFILL_QUEUE", "0")
    case, q, cu, got32 = run(name, torch.float32)
    ref = oracle.paged_attention(q, case.k_log, case.v_log, case.table, case.ctx, SCALE, cu_q=cu, nthreads=8)
    assert np.max(np.abs(got32 - ref)) <= 1e-4 * np.max(np.abs(ref))


def test_choices_in_turn_leave_nothing_behind():
    first = {n: run(n, torch.bfloat16)[3] for n in BATCHES}
    for n in reversed(list(BATCHES)):
        assert np.array_equal(run(n, torch.bfloat16)[3], first[n])
