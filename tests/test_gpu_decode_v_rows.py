"""GPU: which rows of a page's V a lane holds depends on the head dim and the pool's format. Sequences of 1 to
33 tokens with the step's own, so that the new token takes every place of a page, in both schedules, every format and both
head dims: the pool as the append alone leaves it, each row as float64 arithmetic gives it. Slots past the end of a
sequence hold NaN (codes: the largest there are)."""

import pytest
import torch

from llama_lite_npu_amd import ops, workloads
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = list(range(1, 34))


@pytest.mark.parametrize("schedule", [0, 1, 4])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_the_new_token_at_every_place_of_a_page(fmt, head_dim, schedule):
    hq, hkv = 6, 2
    print(f"V rows: {fmt} pool, heads of {head_dim}, schedule {schedule}", flush=True)
    case = workloads.make_decode_case("rows", 85, [n - 1 for n in LENS], hq, hkv, device=DEV, head_dim=head_dim)
    pool, scales, dtype = case.kv_pool.clone(), None, torch.float16
    if fmt != "f16":
        dtype = torch.uint8 if fmt == "fp8" else torch.int8
        scales = torch.tensor([0.031, 0.043, 0.027, 0.039], device=DEV)
        slots = torch.arange(pool.shape[0], dtype=torch.int32, device=DEV)
        pool = torch.empty(case.kv_pool.shape, dtype=dtype, device=DEV)
        ops.kv_append_quantised(case.kv_pool[:, :hkv], case.kv_pool[:, hkv:], slots, pool, scales)
    used = torch.zeros(pool.shape[0], dtype=torch.bool, device=DEV)
    for b, n in enumerate(LENS):
        for t in range(n - 1):
            used[int(case.block_table[b, t // 16]) * 16 + t % 16] = True
    pool[~used] = float("nan") if fmt == "f16" else 0x7e if fmt == "fp8" else 127
    want = pool.clone()
    if fmt == "f16":
        ops.kv_append(case.k_new, case.v_new, case.slot_mapping, want)
    else:
        ops.kv_append_quantised(case.k_new, case.v_new, case.slot_mapping, want, scales)
    plan = ops.DecodePlan(case.block_table, case.seq_lens, hq, hkv, case.num_pages, chunks=7, kv_dtype=dtype,
                          token_bytes=2 * hkv * head_dim * dtype.itemsize)
    plan.set_schedule(schedule)
    out = ops.decode_step(case.q, pool, plan, case.k_new, case.v_new, case.softmax_scale, kv_scales=scales)
    torch.cuda.synchronize()
    words = torch.int16 if fmt == "f16" else torch.uint8
    assert torch.equal(pool.view(words), want.view(words))
    rows = want.double() if fmt != "fp8" else want.view(torch.float8_e4m3fn).double()
    full = (rows if scales is None else rows * scales.double()[None, :, None]).cpu()
    q = case.q.double().cpu()
    ref = torch.empty_like(q)
    for b, n in enumerate(LENS):
        at = torch.tensor([int(case.block_table[b, t // 16]) * 16 + t % 16 for t in range(n)])
        for h in range(hq):
            p = torch.softmax(full[at, h // 3] @ q[b, h] * case.softmax_scale, 0)
            ref[b, h] = p @ full[at, hkv + h // 3]
    assert_attention_close(out, ref.numpy(), f"{fmt} {head_dim} schedule {schedule}")


RAGGED = [700, 1, -1, 16, 333, 17, -1, 1024, 96, 15]        # tokens before the step's own; -1: an empty row
FULL = [319, 303, 318, 190, 319, -1, 304, 317, 311, 288]    # ... that all but fill a table of 20 pages


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("lens,per_chunk", [(FULL, n) for n in (1, 2, 3, 4, 5, 7, 11)] + [(RAGGED, n) for n in (5, 13, 17, 40)])
def test_codes_of_64_with_two_and_four_pages_in_flight(fmt, lens, per_chunk):
    """Four from 13 pages a chunk by the block table's width on. Chunks of up to ``per_chunk`` pages, cut anywhere in the
    sequences, with a table of their own width, which the full one keeps at two, and with one wide enough for four.
    The pages are attended one after the other in both: the same bits, and close to float64."""
    hq, hkv, d = 6, 2, 64
    print(f"pages in flight: {fmt}, {per_chunk} pages a chunk, up to {max(lens)} tokens", flush=True)
    case = workloads.make_decode_case("flight", 86, [max(n, 0) for n in lens], hq, hkv, device=DEV, head_dim=d)
    dtype = torch.uint8 if fmt == "fp8" else torch.int8
    scales = torch.tensor([0.031, 0.043, 0.027, 0.039], device=DEV)
    slots = torch.arange(case.kv_pool.shape[0], dtype=torch.int32, device=DEV)
    pool = torch.empty(case.kv_pool.shape, dtype=dtype, device=DEV)
    ops.kv_append_quantised(case.kv_pool[:, :hkv], case.kv_pool[:, hkv:], slots, pool, scales)
    seq = torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=DEV)
    pages = sum(-(-(n + 1) // 16) for n in lens)
    chunks = -(-pages // per_chunk)
    width = case.block_table.shape[1]
    widths = [width, max(width, -(-13 * chunks // len(lens)))]
    assert len(lens) * widths[1] >= 13 * chunks                     # four pages in flight
    if lens is FULL:
        assert len(lens) * widths[0] < 13 * chunks                  # two
    outs, pools = [], []
    for w in widths:
        table = torch.zeros((len(lens), w), dtype=torch.int32, device=DEV)
        table[:, :width] = case.block_table
        plan = ops.DecodePlan(table, seq, hq, hkv, case.num_pages, chunks=chunks, kv_dtype=dtype, token_bytes=4 * d)
        assert plan.schedule == 0
        mine = pool.clone()
        outs.append(ops.decode_step(case.q, mine, plan, case.k_new, case.v_new, case.softmax_scale, kv_scales=scales))
        pools.append(mine)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(pools[0].view(torch.uint8), pools[1].view(torch.uint8))
    rows = pools[0].double() if fmt == "int8" else pools[0].view(torch.float8_e4m3fn).double()
    full = (rows * scales.double()[None, :, None]).cpu()
    q = case.q.double().cpu()
    ref = torch.zeros_like(q)
    for b, n in enumerate(lens):
        if n < 0:
            continue
        at = torch.tensor([int(case.block_table[b, t // 16]) * 16 + t % 16 for t in range(n + 1)])
        for h in range(hq):
            p = torch.softmax(full[at, h // 3] @ q[b, h] * case.softmax_scale, 0)
            ref[b, h] = p @ full[at, hkv + h // 3]
    assert_attention_close(outs[0], ref.numpy(), f"{fmt} {per_chunk}")
