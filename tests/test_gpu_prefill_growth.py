"""GPU: key tiles below the diagonal are attended two to an iteration, and one whose scores outgrow the running
maximum is redone, after which the loop may stand at an odd or an even tile. Scores that jump in every set of tiles up to
the diagonal, in either half of a tile, over 2 to 9 tiles, all head dims, as float64 arithmetic gives them; the same jumps in
every form the loop is compiled into: two groups of wavefronts and key slices, whose tiles are counted from their own first one,
packed prompts, and the keys of a shared prefix in a decode step."""

import pytest
import torch

from llama_lite_npu_amd import ops
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
JUMPS = [(), (1,), (2,), (1, 2), (2, 3), (1, 3), (2, 4), (1, 2, 3, 4), (3, 4, 5), (5,), (6,), (7,)]


def _inputs(sets, rows, history, hq, hkv, d, fmt, bases=(0,)):
    """q [n, rows, Hq, D], and the keys and values of each sequence as its pool holds them ([n, tokens, 2 Hkv, D] with whole
    pages) and in float64: scores that jump in tiles ``base + tile`` for every tile of the sequence's set."""
    gen = torch.Generator().manual_seed(d + history)
    total = history + rows
    pages = -(-total // 16)
    n = len(sets)
    q0 = torch.randn(hq // 2, d, generator=gen)
    q0 = (q0 / q0.norm(dim=1, keepdim=True)).mean(0)
    q0 = q0 / q0.norm() * d ** 0.5
    q = (q0 + 0.05 * torch.randn(n, rows, hq, d, generator=gen)).half()
    k = 0.3 * torch.randn(n, pages * 16, hkv, d, generator=gen)
    v = torch.randn(n, pages * 16, hkv, d, generator=gen)
    for b, jumps in enumerate(sets):
        for base in bases:
            for step, tile in enumerate(jumps):         # each some 2^10 times as likely as what came before
                at = 64 * (base + tile) + (40 if (b + step) % 2 else 9)
                if at < total:
                    k[b, at] = 7.0 * (step + 1) * q0 / d ** 0.5
    return (q, *_stored(torch.cat([k, v], 2), fmt))


def _stored(rows, fmt):
    """Rows [..., 2 Hkv, D] as a pool holds them, what they stand for in float64, and the scales."""
    if fmt == "f16":
        return rows.half(), rows.half().double(), None
    hkv = rows.shape[-2] // 2
    scales = torch.tensor([0.05] * hkv + [0.04] * hkv)
    codes = rows / scales[:, None]
    if fmt == "int8":
        codes = codes.round().clamp(-127, 127).to(torch.int8)
        values = codes.double()
    else:
        codes = codes.to(torch.float8_e4m3fn)
        values = codes.double()
        codes = codes.view(torch.uint8)
    return codes, values * scales.double()[:, None], scales.to(DEV)


def _check(out, q, full, history, what):
    """out, q: [n, rows, Hq, D]; row r sees the first history + r + 1 tokens of ``full``."""
    n, rows, hq, d = q.shape
    hkv, total = full.shape[2] // 2, history + rows
    seen = torch.arange(total)[None, :] <= history + torch.arange(rows)[:, None]
    qd = q.double()
    for h in range(hq):
        kv = h // (hq // hkv)
        s = torch.matmul(qd[:, :, h], full[:, :total, kv].transpose(1, 2).contiguous()) * d ** -0.5
        p = torch.softmax(s.masked_fill(~seen, -torch.inf), -1)
        ref = torch.matmul(p, full[:, :total, hkv + kv])
        assert_attention_close(out[:, :, h], ref.numpy(), f"{what} head {h}")


def _paged(q, pool, scales, history, copies, **options):
    n, rows, hq, d = q.shape
    pages = pool.shape[1] // 16
    table = torch.arange(n * pages, dtype=torch.int32).view(n, pages).repeat(copies, 1).to(DEV)
    out = ops.paged_prefill(q.repeat(copies, 1, 1, 1).view(-1, hq, d).to(DEV), pool.reshape(-1, pool.shape[2], d).to(DEV), table,
                            torch.arange(0, n * copies * rows + 1, rows, dtype=torch.int32, device=DEV),
                            torch.full((n * copies,), history, dtype=torch.int32, device=DEV), rows, d ** -0.5,
                            kv_scales=scales, max_kv_len=history + rows, **options)
    torch.cuda.synchronize()
    out = out.view(copies, n, rows, hq, d)
    assert bool((out == out[:1]).all())
    return out[0]


@pytest.mark.parametrize("wide", [False, True])         # many workgroups, or few with 64 columns each
@pytest.mark.parametrize("history", [64, 130, 191, 192, 256, 320, 511])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("fmt", ["f16", "int8"])
def test_jumps(fmt, d, history, wide):
    copies = 60 if wide else 1
    print(f"jumps: {fmt}, heads of {d}, {history} cached, {copies} x", flush=True)
    q, pool, full, scales = _inputs(JUMPS, 33, history, 4, 2, d, fmt)
    _check(_paged(q, pool, scales, history, copies), q, full, history, f"{fmt} {d} {history}")


@pytest.mark.parametrize("history", [1563, 1630])       # 25 tiles: groups of 13 and 12; 26: 13 each
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_jumps_in_two_groups(fmt, d, history):
    """192 workgroups of at least 24 tiles: two groups of wavefronts a block (where a workgroup has a compute unit)."""
    print(f"jumps in two groups: {fmt}, heads of {d}, {history} cached", flush=True)
    q, pool, full, scales = _inputs(JUMPS, 33, history, 4, 2, d, fmt, bases=(0, 13))
    _check(_paged(q, pool, scales, history, 8), q, full, history, f"{fmt} {d} {history}")


@pytest.mark.parametrize("copies", [1, 8])              # 64 and 128 columns a workgroup
@pytest.mark.parametrize("history", [1563, 1630])       # 24 and 25 tiles below the diagonal: slices of 8; of 9, 9 and 8
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_jumps_in_key_slices(fmt, d, history, copies):
    print(f"jumps in key slices: {fmt}, heads of {d}, {history} cached, {copies} x", flush=True)
    per = -(-((history + 1) // 64) // 3)
    q, pool, full, scales = _inputs(JUMPS, 33, history, 4, 2, d, fmt, bases=(0, per, 2 * per))
    _check(_paged(q, pool, scales, history, copies, key_slices=3), q, full, history, f"{fmt} {d} {history} {copies}")


@pytest.mark.parametrize("sets,copies", [(JUMPS[3:9], 1), (JUMPS, 1), (JUMPS, 2)])      # one column tile, two groups, neither
@pytest.mark.parametrize("d", [64, 128, 256])
def test_jumps_in_packed_prompts(d, sets, copies):
    rows, hq, hkv, n = 609, 4, 2, len(sets)
    print(f"jumps in packed prompts: heads of {d}, {n} x {copies}", flush=True)
    q, _, full, _ = _inputs(sets, rows, 0, hq, hkv, d, "f16")
    kv = full[:, :rows].half().repeat(copies, 1, 1, 1).view(-1, 2 * hkv, d).to(DEV)
    starts = torch.arange(0, n * copies * rows, rows, dtype=torch.int32, device=DEV)
    out = ops.varlen_prefill(q.repeat(copies, 1, 1, 1).view(-1, hq, d).to(DEV), kv[:, :hkv], kv[:, hkv:], starts,
                             torch.full_like(starts, rows), rows, d ** -0.5)
    torch.cuda.synchronize()
    out = out.view(copies, n, rows, hq, d)
    assert bool((out == out[:1]).all())
    _check(out[0], q, full, 0, f"packed {d} {n} x {copies}")


@pytest.mark.parametrize("sets", [JUMPS, JUMPS[0::3], JUMPS[1::3], JUMPS[2::3]])        # 384 columns: eight wavefronts; 128: four
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_jumps_behind_a_shared_prefix(fmt, d, sets):
    """A wavefront's 32 columns are four sequences of eight heads, with a set of tiles of their own; the prefix is cut into
    8 slices of 9 tiles, each with the same jumps. A sequence's q finds a large score in the tiles of its set alone."""
    hq, tiles, slices, own = 8, 9, 8, 5
    print(f"jumps behind a shared prefix: {fmt}, heads of {d}, {len(sets)} sets", flush=True)
    n, prefix = 4 * len(sets), 64 * tiles * slices
    gen = torch.Generator().manual_seed(d + n)
    rows = torch.randn(prefix + 16 * n, 2, d, generator=gen)
    rows[:, 0] *= 0.3
    q = 0.05 * torch.randn(n, hq, d, generator=gen)
    for tile in range(1, 8):
        for s in range(slices):
            at = 64 * (tiles * s + tile) + (40 if (s + tile) % 2 else 9)
            rows[at, 0] = 0.0
            rows[at, 0, tile] = 6.0
        for b in range(n):
            if tile in sets[b // 4]:
                q[b, :, tile] += 7.0 * (1 + sets[b // 4].index(tile)) * d ** 0.5 / 6.0
    q = q.half()
    pool, full, scales = _stored(rows, fmt)
    shared = prefix // 16
    table = torch.cat([torch.arange(shared).expand(n, -1), shared + torch.arange(n)[:, None]], 1).to(torch.int32).to(DEV)
    lens = torch.full((n,), prefix + own, dtype=torch.int32, device=DEV)
    pool = pool.to(DEV)
    plan = ops.DecodePlan(table, lens, hq, 1, pool.shape[0] // 16, shared_pages=shared, kv_dtype=pool.dtype,
                          token_bytes=2 * d * pool.element_size())
    out = ops.decode_step(q.to(DEV), pool, plan, softmax_scale=d ** -0.5, kv_scales=scales)
    torch.cuda.synchronize()
    seen = torch.cat([torch.arange(prefix).expand(n, -1), prefix + 16 * torch.arange(n)[:, None] + torch.arange(own)], 1)
    mine = full[seen]
    p = torch.softmax(torch.matmul(q.double(), mine[:, :, 0].transpose(1, 2).contiguous()) * d ** -0.5, -1)
    assert_attention_close(out, torch.matmul(p, mine[:, :, 1]).numpy(), f"prefix {fmt} {d}")
