"""GPU: the native prefill call takes launches that are cut along their keys, workspace included: the bits of the
wrapper's own way, for chunks on both sides of the rule, every pool format, heads of 64 and 128, two streams, and a library
status as it is."""

import pytest
import torch

from llama_lite_npu_amd import _lib, ops
from tests.test_native_calls import _NoCalls

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _chunk(fmt, d, rows, history, batch=1, hq=8, hkv=2):
    gen = torch.Generator(device=DEV).manual_seed(d + rows + history)
    pages = -(-(history + rows) // 16)
    pool = torch.randn((batch * pages * 16, 2 * hkv, d), generator=gen, device=DEV, dtype=torch.float16)
    scales = None
    if fmt != "f16":
        scales = torch.full((2 * hkv,), 0.03, device=DEV)
        codes = torch.empty(pool.shape, device=DEV, dtype=torch.int8 if fmt == "int8" else torch.uint8)
        ops.kv_append_quantised(pool[:, :hkv], pool[:, hkv:], torch.arange(pool.shape[0], dtype=torch.int32, device=DEV), codes,
                                scales)
        pool = codes
    table = torch.randperm(batch * pages, generator=gen, device=DEV).to(torch.int32).view(batch, pages)
    return dict(q=torch.randn((batch * rows, hq, d), generator=gen, device=DEV, dtype=torch.float16), kv_pool=pool,
                block_table=table, cu_q_lens=torch.arange(0, batch * rows + 1, rows, dtype=torch.int32, device=DEV),
                context_lens=torch.full((batch,), history, dtype=torch.int32, device=DEV), max_q_len=rows,
                softmax_scale=d ** -0.5, page_size=16, kv_scales=scales, max_kv_len=history + rows)


@pytest.mark.parametrize("rows,history,batch", [(1, 1000, 1), (16, 200, 1), (37, 3001, 1), (64, 5000, 2), (300, 90, 1)])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_cut_launches_as_the_wrapper_makes_them(fmt, d, rows, history, batch, monkeypatch):
    print(f"native key slices: {fmt}, heads of {d}, {batch} x {rows} rows over {history}", flush=True)
    c = _chunk(fmt, d, rows, history, batch)
    slices = _lib.load().litekv_paged_prefill_key_slices(batch, 8, 2, d, rows, history + rows)
    assert (slices > 1) == (history >= 1000)
    calls = _lib.calls()
    taken = calls.paged_prefill(c["q"], c["kv_pool"], c["block_table"], c["cu_q_lens"], c["context_lens"], rows,
                                c["softmax_scale"], 16, c["kv_scales"], history + rows, ops._stream())
    native = ops.paged_prefill(**c)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        beside = ops.paged_prefill(**c)
    torch.cuda.current_stream().wait_stream(side)
    monkeypatch.setattr(_lib, "calls", lambda: _NoCalls)
    plain = ops.paged_prefill(**c)
    torch.cuda.synchronize()
    assert isinstance(taken, torch.Tensor)
    assert all(torch.equal(x, plain) for x in (taken, native, beside))


def test_a_status_of_a_cut_launch_comes_back():
    print("native key slices: status", flush=True)
    c = _chunk("f16", 128, 16, 2000)
    q = torch.zeros(c["q"].numel() + 1, device=DEV, dtype=torch.float16)[1:].view_as(c["q"])     # misaligned
    status = _lib.calls().paged_prefill(q, c["kv_pool"], c["block_table"], c["cu_q_lens"], c["context_lens"], 16, 0.1, 16, None,
                                        2016, ops._stream())
    assert type(status) is int and status == 1
    with pytest.raises(_lib.LiteKVError, match="align"):
        _lib.check(status)
