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


def _plant(case, key, element, value, which):
    """The packed row `key` gets `value` in one element of kv head 1 (k or v), in the pool as well."""
    (case.k if which == "k" else case.v)[key, 1, element] = value
    ops.kv_append(case.k, case.v, case.slot_mapping, case.kv_pool)


def _rows_with_values(out, ref, key, element, want, group):
    """`out` is `ref`, but for the rows from `key` on of the heads of kv head 1: `want` in `element`."""
    ref = ref.clone()
    ref[key:, group:2 * group, element] = want
    got = out.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    fine = torch.isfinite(ref)
    assert torch.equal(got[~fine & ~torch.isnan(ref)], ref[~fine & ~torch.isnan(ref)])
    assert_attention_close(torch.where(fine, got, 0.0), torch.where(fine, ref, 0.0).numpy(), "finite part")


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("hq,length,key", [(16, 200, 40), (16, 200, 130), (8, 190, 0), (28, 70, 69), (4, 150, 127),
                                               (16, 161, 3), (8, 169, 168)])
def test_an_infinite_value_reaches_the_rows_that_see_it(hq, length, key, value):
    """V of one key, one element: rows from that key on get it (a weight is above 0 at these scores), no
    earlier row and no other element does, wherever the key stands in its tile."""
    print(f"prefill 256, {value} in V of key {key} of {length}, {hq} heads", flush=True)
    case = _case(63, [length], hq, 4)
    ref = _reference(case, 0.0625)
    _plant(case, key, 77, value, "v")
    for out in (_paged(case, 0.0625), _packed(case, 0.0625)):
        torch.cuda.synchronize()
        _rows_with_values(out, ref, key, 77, value, hq // 4)


def test_a_value_that_is_not_a_number_in_a_pool_of_codes():
    case = _case(64, [90], 16, 4, [100])
    gen = torch.Generator().manual_seed(5)
    codes = torch.randint(-128, 128, case.kv_pool.shape, generator=gen, dtype=torch.int16).to(torch.uint8) & 0xBF
    scales = torch.full((8,), 0.5)
    ref = _reference(case, 0.0625, torch.from_numpy(fp8.dequantize_pool(codes.numpy(), scales.numpy())))
    slot = int(case.slot_mapping[50])
    codes[slot, 4 + 1, 33] = 0x7F                                   # V of the chunk's row 50, kv head 1
    out = _paged(case, 0.0625, codes.to(DEV), kv_scales=scales.to(DEV))
    torch.cuda.synchronize()
    _rows_with_values(out, ref, 50, 33, float("nan"), 4)


def test_an_infinite_key_and_query():
    """A score of -inf takes the key out of the row, one of +inf (or a query that is not a number) makes
    the row not a number; rows beside it in the tile stay as they are."""
    case = _case(65, [150], 16, 4)
    case.q[90, 5, 3] = float("nan")
    case.q[:, 4:8, 20] = case.q[:, 4:8, 20].abs().clamp(min=0.25) * -1
    case.q[100, 6, 20] = 0.5
    _plant(case, 30, 20, float("inf"), "k")
    ref = _reference(case, 0.0625)                                  # softmax of -inf is 0, of +inf NaN
    assert int(torch.isnan(ref).any(-1).sum()) == 2
    for out in (_paged(case, 0.0625), _packed(case, 0.0625)):
        torch.cuda.synchronize()
        got = out.double().cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(ref)) and not bool(torch.isinf(got).any())
        assert_attention_close(got.nan_to_num(0.0), ref.nan_to_num(0.0).numpy(), "rows beside it")


@pytest.mark.parametrize("first", [True, False], ids=["likeliest first", "likeliest last"])
@pytest.mark.parametrize("below,history", [(14.4, 3000), (22.4, 12000), (24.4, 20000)])
def test_many_unlikely_keys_behind_one_of_no_value(below, history, first):
    """One key `below` powers of two likelier than each of the history's others, of value 0 in half of the
    elements: there the row is the sum over the others, so their probabilities must keep their bits.

    Bound: fp16's rounding of the output, 2^-11 of it; probabilities that are off by 2^-34 of the
    likeliest's, all to one side, times the largest value; fp32 sums over steps of 32 keys, one
    rounding (2^-24 of the sum) each, and as much again for scores and exponentials."""
    print(f"prefill 256, {history} keys {below} powers of two below one, first {first}", flush=True)
    case = _case(66, [20], 8, 2, [history])
    gen = torch.Generator().manual_seed(7)
    n = history + 20
    slots = (case.block_table[0].long().cpu()[torch.arange(n) // 16] * 16 + torch.arange(n) % 16)
    k, v = torch.zeros((n, 2, D)), 20 + torch.randn((n, 2, D), generator=gen)
    log2e = 1.4426950408889634
    k[:, :, 0] = -(below + torch.rand((n, 2), generator=gen) * 0.4 - 0.2) / log2e
    at = 0 if first else history - 1
    k[at, :, 0], v[at, :, :D // 2] = 0.0, 0.0
    pool = case.kv_pool.cpu()
    pool[slots] = torch.cat([k, v], 1).half()
    case.kv_pool.copy_(pool)
    case.q[:] = 0.0
    case.q[:, :, 0] = 16.0
    out = _paged(case, 0.0625)
    torch.cuda.synchronize()
    ref = _reference(case, 0.0625)
    bound = (2.0 ** -11 + 2 * (n / 32) * 2.0 ** -24) * ref.abs() + n * 2.0 ** -34 * float(v.max())
    off = (out.double().cpu() - ref).abs()
    print(f"  largest error {float((off / ref.abs()).max()):.2e} of the value", flush=True)
    assert bool((off <= bound).all()), float((off / bound).max())


def _spiked(case, at):
    """Key `at` of sequence 0 scores about 2^40 above the others for every query head that follows it."""
    case.q[:, :, :4] = 4.0
    case.k[at, :, :4] = 28.0
    ops.kv_append(case.k, case.v, case.slot_mapping, case.kv_pool)


@pytest.mark.parametrize("fmt", ["f16", "packed", "fp8", "int8"])
@pytest.mark.parametrize("hq,lens,ctx,page_size,at", [(16, [150, 1, 33], [70, 0, 5], 16, 90), (28, [40], [47], 32, 3)])
def test_general_kernel_in_every_form(fmt, hq, lens, ctx, page_size, at):
    """Outputs whose rows are not 16-byte aligned stay with the general kernel: every source of keys, one
    key that takes the whole weight, nothing written beside the rows."""
    if fmt == "packed":
        ctx = None
    print(f"prefill 256, general kernel, {fmt}, {hq} heads, {lens}", flush=True)
    case = _case(67, lens, hq, 4, ctx, page_size)
    _spiked(case, at)
    wide = torch.zeros((case.q.shape[0], hq * D + 4), dtype=torch.float16, device=DEV)
    out = wide[:, :hq * D].unflatten(1, (hq, D))
    values = None
    if fmt == "packed":
        ops.varlen_prefill(case.q, case.k, case.v, case.cu_q_lens[:-1], case.seq_lens, case.max_q_len, 0.0625, out=out)
    elif fmt == "f16":
        _paged(case, 0.0625, out=out)
    else:
        scales = torch.tensor([28.0 / 100] * 4 + [0.04] * 4)
        pool = torch.zeros(case.kv_pool.shape, dtype=torch.uint8 if fmt == "fp8" else torch.int8, device=DEV)
        every = torch.arange(pool.shape[0], dtype=torch.int32, device=DEV)
        ops.kv_append_quantised(case.kv_pool[:, :4], case.kv_pool[:, 4:], every, pool, scales.to(DEV))
        _paged(case, 0.0625, pool, out=out, kv_scales=scales.to(DEV))
        values = torch.from_numpy((fp8 if fmt == "fp8" else int8).dequantize_pool(pool.cpu().numpy(), scales.numpy()))
    torch.cuda.synchronize()
    assert_attention_close(out, _reference(case, 0.0625, values).numpy(), f"general kernel, {fmt}")
    assert bool((wide[:, hq * D:] == 0).all())
