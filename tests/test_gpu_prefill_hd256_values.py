"""256-wide prefill over scales and values that the matrix pipeline is not made for, against float64:
what it cannot serve goes to fp32 arithmetic, with the results that arithmetic gives."""

import pytest
import torch

from llama_lite_npu_amd import ops, workloads
from oracle import cpu_ref, fp8, int8
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
D = 256


def _case(seed, lens, hq, hkv, ctx=None, page_size=16):
    case = workloads.make_prefill_case("v256", seed, lens, hq, hkv, context_lens=ctx, device=DEV, page_size=page_size,
                                       head_dim=D)
    ops.kv_append(case.k, case.v, case.slot_mapping, case.kv_pool)
    return case


def _reference(case, scale, values=None):
    pool = case.kv_pool.cpu() if values is None else values
    return cpu_ref.paged_prefill_ref(case.q.cpu(), pool, case.block_table.cpu(), case.cu_q_lens.cpu(),
                                     case.context_lens.cpu(), scale, page_size=case.page_size, dtype=torch.float64)


def _paged(case, scale, pool=None, **kw):
    return ops.paged_prefill(case.q, case.kv_pool if pool is None else pool, case.block_table, case.cu_q_lens,
                             case.context_lens, case.max_q_len, scale, page_size=case.page_size, **kw)


def _packed(case, scale):
    return ops.varlen_prefill(case.q, case.k, case.v, case.cu_q_lens[:-1], case.seq_lens, case.max_q_len, scale)


@pytest.mark.parametrize("scale", [0.0, -0.0625, 1e-38])
def test_any_softmax_scale(scale):
    """0 and (nearly) 0: uniform weights; below 0: the smallest product weighs most."""
    print(f"prefill 256, softmax scale {scale}", flush=True)
    case = _case(61, [130, 1, 70], 16, 4)
    paged, packed = _paged(case, scale), _packed(case, scale)
    torch.cuda.synchronize()
    ref = _reference(case, scale).numpy()
    assert_attention_close(paged, ref, f"paged, scale {scale}")
    assert_attention_close(packed, ref, f"packed, scale {scale}")


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("hq,lens,ctx,page_size", [(16, [70, 1, 33], [130, 0, 64], 32), (28, [20], [47], 16)])
def test_any_k_scale(fmt, hq, lens, ctx, page_size):
    """Pools of codes whose K scales are ordinary, 0, negative and next to nothing, side by side."""
    print(f"prefill 256 over {fmt}, {hq} heads, K scales of every kind", flush=True)
    case = _case(62, lens, hq, 4, ctx, page_size)
    gen = torch.Generator().manual_seed(5)
    codes = torch.randint(-80, 81, case.kv_pool.shape, generator=gen, dtype=torch.int8)
    oracle = int8
    if fmt == "fp8":
        oracle, codes = fp8, codes.view(torch.uint8) & 0xBF        # |value| < 2
    scales = torch.tensor([0.04, 0.0, -0.03, 1e-36, 0.03, 0.04, 0.05, 0.06])
    out = _paged(case, 0.0625, codes.to(DEV), kv_scales=scales.to(DEV))
    torch.cuda.synchronize()
    values = torch.from_numpy(oracle.dequantize_pool(codes.numpy(), scales.numpy()))
    assert_attention_close(out, _reference(case, 0.0625, values).numpy(), f"K scales over {fmt}")
