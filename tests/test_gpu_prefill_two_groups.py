"""GPU: a prefill of at most as many workgroups as compute units whose longest row sees many keys (as the
caller says) is attended by two groups of wavefronts per block, each over half of its key tiles; one of at
most half as many workgroups with one column tile per wavefront. Blocks of one tile (the first group has none) up to odd
and even numbers of them, ragged last blocks and tiles, every pool format, both head dims, paged and
packed, in a batch (two groups) and sequence by sequence (one column tile): against float64 arithmetic."""

import pytest
import torch

from llama_lite_npu_amd import ops
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# (rows of the chunk, keys cached before it): the tiles of a block go from 1 to 12
SHAPES = [(1, 0), (70, 0), (17, 47), (16, 48), (64, 64), (33, 95), (1, 127), (129, 128), (130, 250), (5, 700), (150, 511)]


def _reference(q, k, v, ctx, scale):
    q, k, v = q.double().cpu(), k.double().cpu(), v.double().cpu()
    group = q.shape[1] // k.shape[1]
    visible = torch.arange(k.shape[0])[None, :] <= ctx + torch.arange(q.shape[0])[:, None]
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // group].T * scale).masked_fill(~visible, float("-inf"))
        out[:, h] = torch.softmax(s, 1) @ v[:, h // group]
    return out


@pytest.mark.parametrize("hq,hkv", [(8, 1), (4, 2), (3, 3), (10, 1)])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_two_groups(fmt, head_dim, hq, hkv):
    print(f"two key groups: {fmt} pool, {hq}/{hkv} heads of {head_dim}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(5)
    rows = [r for r, _ in SHAPES]
    ctx = [c for _, c in SHAPES]
    pages = [-(-(r + c) // 16) for r, c in SHAPES]
    perm = torch.randperm(sum(pages), generator=gen, device=DEV).to(torch.int32)
    width = max(pages)
    table = torch.zeros((len(SHAPES), width), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    kv = torch.randn((sum(pages) * 16, 2 * hkv, head_dim), generator=gen, dtype=torch.float16, device=DEV)
    pool, scales, values = kv, None, kv
    if fmt != "f16":
        scales = torch.full((2 * hkv,), 0.035, device=DEV)
        pool = torch.empty(kv.shape, dtype=torch.uint8 if fmt == "fp8" else torch.int8, device=DEV)
        slots = torch.arange(kv.shape[0], dtype=torch.int32, device=DEV)
        ops.kv_append_quantised(kv[:, :hkv], kv[:, hkv:], slots, pool, scales)
        values = (pool if fmt == "int8" else pool.view(torch.float8_e4m3fn)).double() * 0.035
    q = torch.randn((sum(rows), hq, head_dim), generator=gen, dtype=torch.float16, device=DEV)
    scale = head_dim ** -0.5
    one = torch.empty_like(q)
    first = 0
    for b, (r, c) in enumerate(SHAPES):
        part = slice(first, first + r)
        ops.paged_prefill(q[part], pool, table[b:b + 1], torch.tensor([0, r], dtype=torch.int32, device=DEV),
                          torch.tensor([c], dtype=torch.int32, device=DEV), r, scale, out=one[part], kv_scales=scales,
                          key_slices=1)
        first += r
    # the batch, as often as makes it more than half as many workgroups as there are compute units
    splits = -(-(hq // hkv) // 8)
    block_rows = 16 * (8 // -(-(hq // hkv) // splits))
    wgs = hkv * splits * -(-max(rows) // block_rows) * len(rows)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    copies = cus // 2 // wgs + 1
    assert cus < 2 * wgs * copies <= 2 * cus
    cu = torch.tensor([0] + rows * copies, dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV)
    batch = ops.paged_prefill(q.repeat(copies, 1, 1), pool, table.repeat(copies, 1), cu,
                              torch.tensor(ctx * copies, dtype=torch.int32, device=DEV), max(rows), scale, kv_scales=scales,
                              key_slices=1, max_kv_len=4096)      # (the form goes by the bound, not by the lengths)
    torch.cuda.synchronize()
    for out in batch.split(sum(rows)):
        assert torch.equal(out, batch[:sum(rows)])
    first = 0
    for b, (r, c) in enumerate(SHAPES):
        slot = torch.cat([table[b, t // 16, None].long() * 16 + t % 16 for t in range(r + c)])
        ref = _reference(q[first:first + r], values[slot, :hkv], values[slot, hkv:], c, scale).numpy()
        assert_attention_close(batch[first:first + r], ref, f"two groups, rows {r} ctx {c}")
        assert_attention_close(one[first:first + r], ref, f"one column tile, rows {r} ctx {c}")
        first += r


@pytest.mark.parametrize("head_dim", [64, 128])
def test_two_groups_over_packed_rows(head_dim):
    print(f"two key groups, packed, heads of {head_dim}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(6)
    lens, hq, hkv = [513, 1, 64, 65, 130], 6, 2
    q, k, v = (torch.randn((sum(lens), h, head_dim), generator=gen, dtype=torch.float16, device=DEV) for h in (hq, hkv, hkv))
    starts = torch.tensor([0] + lens[:-1], dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV)
    out = ops.varlen_prefill(q, k, v, starts, torch.tensor(lens, dtype=torch.int32, device=DEV), max(lens))
    torch.cuda.synchronize()
    first = 0
    for n in lens:
        s = slice(first, first + n)
        assert_attention_close(out[s], _reference(q[s], k[s], v[s], 0, head_dim ** -0.5).numpy(), f"length {n}")
        first += n


@pytest.mark.parametrize("fmt,head_dim,rows,batch,keys,told", [
    ("f16", 128, 60, 8, 64, True), ("f16", 128, 60, 8, 9 * 64, True),       # few keys
    ("f16", 128, 16, 30, 23 * 64, True),                                    # one block a sequence
    ("f16", 64, 100, 7, 9 * 64, True), ("fp8", 128, 60, 8, 3 * 64, True), ("int8", 64, 100, 7, 3 * 64, True),
    ("f16", 128, 60, 8, 20 * 64, False), ("fp8", 64, 100, 7, 20 * 64, False),   # the caller does not say
])
def test_few_keys_in_a_wide_table_are_attended_by_one_group(fmt, head_dim, rows, batch, keys, told):
    """A launch of more workgroups than compute units has one group a block: the same bits."""
    print(f"one key group: {fmt} pool, heads of {head_dim}, {batch} x {rows} rows, {keys} keys, told {told}", flush=True)
    hq, hkv = (64, 8) if head_dim == 128 else (32, 8)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    wgs = hkv * batch * -(-rows // (128 * hkv // hq))
    assert cus < 2 * wgs <= 2 * cus
    gen = torch.Generator(device=DEV).manual_seed(9)
    pages = keys // 16
    pool = torch.randn((batch * keys, 2 * hkv, head_dim), generator=gen, dtype=torch.float16, device=DEV)
    scales = None
    if fmt != "f16":
        scales = torch.full((2 * hkv,), 0.035, device=DEV)
        codes = torch.empty(pool.shape, dtype=torch.uint8 if fmt == "fp8" else torch.int8, device=DEV)
        slots = torch.arange(batch * keys, dtype=torch.int32, device=DEV)
        ops.kv_append_quantised(pool[:, :hkv], pool[:, hkv:], slots, codes, scales)
        pool = codes
    table = torch.zeros((batch, 2048), dtype=torch.int32, device=DEV)
    table[:, :pages] = torch.randperm(batch * pages, generator=gen, device=DEV).to(torch.int32).view(batch, pages)
    q = torch.randn((batch * rows, hq, head_dim), generator=gen, dtype=torch.float16, device=DEV)

    def run(copies):
        cu = torch.arange(0, (batch * copies + 1) * rows, rows, dtype=torch.int32, device=DEV)
        ctx = torch.full((batch * copies,), keys - rows, dtype=torch.int32, device=DEV)
        return ops.paged_prefill(q.repeat(copies, 1, 1), pool, table.repeat(copies, 1), cu, ctx, rows, head_dim ** -0.5,
                                 kv_scales=scales, key_slices=1, max_kv_len=keys if told else None)

    few, many = run(1), run(cus // wgs + 1)
    torch.cuda.synchronize()
    assert torch.equal(few, many[:few.shape[0]])
