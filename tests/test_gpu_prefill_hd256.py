"""Prefill at head dim 256 on the tiled kernel, against the fp32 oracle."""

import pytest
import torch

from llama_lite_npu_amd import ops, workloads
from oracle import c_oracle, cpu_ref, fp8, int8
from tests.parity import assert_attention_close, to_np16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
D = 256


def _oracle(case, pool):
    return c_oracle.paged_prefill(to_np16(case.q), pool, case.block_table.cpu().numpy(), case.cu_q_lens.cpu().numpy(),
                                  case.context_lens.cpu().numpy(), case.softmax_scale, page_size=case.page_size)


@pytest.mark.parametrize("hq,hkv,lens,ctx,page_size", [
    (16, 4, [700, 333, 1, 16, 63, 64, 65, 129], None, 16),   # tiles below the diagonal, tile and block edges
    (8, 8, [130, 257], [0, 511], 32),                        # no grouping: 128 query rows per workgroup
    (14, 2, [200, 31], None, 64),                            # 7 heads per kv head: an idle column tile
    (24, 2, [90, 17], [900, 64], 16),                        # 12: two workgroups per kv head, long history
])
def test_tiled_prefill_256(hq, hkv, lens, ctx, page_size):
    """Paged = packed bit for bit, repeats bit for bit, and an output whose rows are not 16-byte
    aligned (the general kernel) agrees. Probabilities reach the second product within 2^-23 of
    themselves or 2^-34 of the row's largest, so what is left against the oracle is the output's own rounding: 2^-11 of the value, and fp32 noise."""
    print(f"prefill 256 {hq}/{hkv} {lens} ctx {ctx} page_size {page_size}", flush=True)
    case = workloads.make_prefill_case("p256", 5200 + hq, lens, hq, hkv, context_lens=ctx, device=DEV,
                                       page_size=page_size, head_dim=D)
    ops.kv_append(case.k, case.v, case.slot_mapping, case.kv_pool)
    args = (case.q, case.kv_pool, case.block_table, case.cu_q_lens, case.context_lens if ctx is not None else None,
            case.max_q_len, case.softmax_scale)
    outs = [ops.paged_prefill(*args, page_size=page_size) for _ in range(3)]
    wide = torch.zeros((case.q.shape[0], hq * D + 4), dtype=torch.float16, device=DEV)
    general = ops.paged_prefill(*args, out=wide[:, :hq * D].unflatten(1, (hq, D)), page_size=page_size)
    torch.cuda.synchronize()
    ref = torch.from_numpy(_oracle(case, to_np16(case.kv_pool)))
    assert_attention_close(outs[0], ref.numpy(), "paged prefill 256")
    assert bool(((outs[0].float().cpu() - ref).abs() <= 2.0 ** -11 * ref.abs() + 2e-5).all())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert_attention_close(general, ref.numpy(), "general kernel")
    assert bool((wide[:, hq * D:] == 0).all())
    if ctx is None:
        packed = ops.varlen_prefill(case.q, case.k, case.v, case.cu_q_lens[:-1], case.seq_lens, case.max_q_len,
                                    case.softmax_scale)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], packed)


@pytest.mark.parametrize("hq,hkv", [(1, 1), (6, 2), (8, 2), (8, 1)])
def test_row_blocks_of_every_fill_256(hq, hkv):
    """One column tile per wavefront: blocks of 128, 32 and 16 rows, filled from one row to all, and a
    prompt whose rows end a tile of keys early, on it and behind it. Bound as above."""
    lens = [1, 15, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 193]
    print(f"prefill 256 {hq}/{hkv}, every fill of a block", flush=True)
    case = workloads.make_prefill_case("p256", 5250 + hq + hkv, lens, hq, hkv, device=DEV, head_dim=D)
    ops.kv_append(case.k, case.v, case.slot_mapping, case.kv_pool)
    out = ops.paged_prefill(case.q, case.kv_pool, case.block_table, case.cu_q_lens, None, case.max_q_len,
                            case.softmax_scale)
    torch.cuda.synchronize()
    ref = torch.from_numpy(_oracle(case, to_np16(case.kv_pool)))
    assert bool(((out.float().cpu() - ref).abs() <= 2.0 ** -11 * ref.abs() + 2e-5).all())


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("lens,ctx,page_size", [([200, 1, 64], [300, 47, 0], 16), ([129], [640], 64)])
def test_tiled_chunk_prefill_256_of_codes(fmt, lens, ctx, page_size):
    print(f"prefill 256 over {fmt} {lens} ctx {ctx} page_size {page_size}", flush=True)
    hq, hkv = 16, 4
    case = workloads.make_prefill_case("p256", 5300 + sum(lens), lens, hq, hkv, context_lens=ctx, device=DEV,
                                       page_size=page_size, head_dim=D)
    oracle, dtype = (fp8, torch.uint8) if fmt == "fp8" else (int8, torch.int8)
    scales = torch.linspace(0.03, 0.05, 2 * hkv, device=DEV)
    pool = torch.zeros(case.kv_pool.shape, dtype=dtype, device=DEV)
    every = torch.arange(pool.shape[0], dtype=torch.int32, device=DEV)
    ops.kv_append_quantised(case.kv_pool[:, :hkv], case.kv_pool[:, hkv:], every, pool, scales)
    ops.kv_append_quantised(case.k, case.v, case.slot_mapping, pool, scales)
    out = ops.paged_prefill(case.q, pool, case.block_table, case.cu_q_lens, case.context_lens, case.max_q_len,
                            case.softmax_scale, page_size=page_size, kv_scales=scales)
    torch.cuda.synchronize()
    values = oracle.dequantize_pool(pool.cpu().numpy(), scales.cpu().numpy())
    ref = cpu_ref.paged_prefill_ref(case.q.cpu(), torch.from_numpy(values), case.block_table.cpu(),
                                    case.cu_q_lens.cpu(), case.context_lens.cpu(), case.softmax_scale,
                                    page_size=page_size)
    assert_attention_close(out, ref.numpy(), f"chunk prefill 256 over {fmt}")
