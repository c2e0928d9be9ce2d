"""GPU: the splits schedule reads a block-table row through a window of 64 entries per wavefront and
its merge requests every partial row a head could have. Rows of just under, exactly and just over
one and two windows, in one to sixteen splits, beside sequences of one page and of none, against the
oracle; unwritten partial rows hold NaN."""

import pytest
import torch

from llama_lite_npu_amd import ops, workloads
from oracle import c_oracle
from tests.parity import assert_attention_close, to_np16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("splits", [1, 2, 4, 16])
@pytest.mark.parametrize("pages", [3, 63, 64, 65, 127, 129, 193])
@pytest.mark.parametrize("hq,hkv", [(16, 8), (40, 8)])
def test_rows_around_the_window(hq, hkv, pages, splits):
    lens = [16 * pages - 3, 0, 5, 16 * (pages - 2), 16 * pages - 1]   # tokens before the step's own
    print(f"row window: heads {hq}/{hkv} pages {pages} splits {splits}", flush=True)
    case = workloads.make_decode_case("window", 77, lens, hq, hkv, device=DEV)
    plan = ops.DecodePlan(case.block_table, case.seq_lens, hq, hkv, case.num_pages)
    plan.set_schedule(splits)
    if plan.split_workspace is not None:
        plan.split_workspace.fill_(float("nan"))
    pool = case.kv_pool.clone()
    out = ops.decode_step(case.q, pool, plan, case.k_new, case.v_new, case.softmax_scale)
    want = case.kv_pool.clone()
    ops.kv_append(case.k_new, case.v_new, case.slot_mapping, want)
    torch.cuda.synchronize()
    assert torch.equal(pool.view(torch.int16), want.view(torch.int16))
    ref = c_oracle.paged_decode(to_np16(case.q), to_np16(pool), case.block_table.cpu().numpy(),
                                case.seq_lens.cpu().numpy(), case.softmax_scale)
    assert_attention_close(out, ref, f"pages {pages} splits {splits}")


@pytest.mark.parametrize("splits", [0, 1, 4])
def test_rows_that_end_with_their_table(splits):
    """Views of some columns of a wider table, the last row's included: as the copied table."""
    print(f"table views, {splits} splits", flush=True)
    for lens in ([300, 40, 200], [150]):
        case = workloads.make_decode_case("views", 78, lens, 16, 8, device=DEV)
        b, width = case.block_table.shape
        wide = torch.full((b, width + 1500), case.num_pages - 1, dtype=torch.int32, device=DEV)
        wide[:, 1500:] = case.block_table
        outs = []
        for table in (case.block_table, wide[:, 1500:]):
            plan = ops.DecodePlan(table, case.seq_lens, 16, 8, case.num_pages)
            plan.set_schedule(splits)
            plan.refresh()
            outs.append(ops.decode_step(case.q, case.kv_pool.clone(), plan, case.k_new, case.v_new, case.softmax_scale))
            out = torch.empty_like(case.q)
            if splits > 0:
                outs.append(ops.paged_decode_static(case.q, case.kv_pool, table, case.seq_lens, out, splits, 1))
        torch.cuda.synchronize()
        half = len(outs) // 2
        assert all(torch.equal(a, b) for a, b in zip(outs[:half], outs[half:]))


@pytest.mark.parametrize("batch,hq,hkv", [(16, 64, 8), (17, 64, 8), (33, 32, 4)])
@pytest.mark.parametrize("splits", [16, 17])
def test_merge_on_either_side_of_its_rule(batch, hq, hkv, splits):
    """16 rows a head are requested before the length up to 8 MiB of them (16 x 64 heads); more rows, and
    more splits, after it: the same fold in fp32, so the sequences both batches hold agree to a step of
    the output's fp16."""
    print(f"merge: {batch} sequences, {hq}/{hkv} heads, {splits} splits", flush=True)
    lens = [30, 0, 4000, 700, 17, 255, 256, 257, 1, 2000, 33, 48] * 3
    case = workloads.make_decode_case("merge", 79, lens[:batch], hq, hkv, device=DEV)
    outs = []
    for rows in (slice(0, 12), slice(0, batch)):
        plan = ops.DecodePlan(case.block_table[rows].contiguous(), case.seq_lens[rows].contiguous(), hq, hkv,
                              case.num_pages)
        plan.set_schedule(splits)
        plan.split_workspace.fill_(float("nan"))
        outs.append(ops.decode_step(case.q[rows], case.kv_pool.clone(), plan, case.k_new[rows], case.v_new[rows],
                                    case.softmax_scale))
    torch.cuda.synchronize()
    few, many = outs[0].float(), outs[1][:12].float()
    assert bool(((few - many).abs() <= 2.0 ** -10 * few.abs() + 2.0 ** -24).all())
    pool = case.kv_pool.clone()
    ops.kv_append(case.k_new, case.v_new, case.slot_mapping, pool)
    ref = c_oracle.paged_decode(to_np16(case.q), to_np16(pool), case.block_table.cpu().numpy(),
                                case.seq_lens.cpu().numpy(), case.softmax_scale)
    assert_attention_close(outs[1], ref, f"{batch} sequences, {splits} splits")
