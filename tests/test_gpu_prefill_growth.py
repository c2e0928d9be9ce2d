"""GPU: key tiles below the diagonal are attended two to an iteration, and one whose scores outgrow the running
maximum is redone, after which the loop may stand at an odd or an even tile. Scores that jump in every set of tiles up to
the diagonal, in either half of a tile, over 2 to 9 tiles, all head dims, as float64 arithmetic gives them."""

import pytest
import torch

from llama_lite_npu_amd import ops
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
JUMPS = [(), (1,), (2,), (1, 2), (2, 3), (1, 3), (2, 4), (1, 2, 3, 4), (3, 4, 5), (5,), (6,), (7,)]


@pytest.mark.parametrize("wide", [False, True])         # many workgroups, or few with 64 columns each
@pytest.mark.parametrize("history", [64, 130, 191, 192, 256, 320, 511])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("fmt", ["f16", "int8"])
def test_jumps(fmt, d, history, wide):
    rows, hq, hkv = 33, 4, 2
    copies = 60 if wide else 1
    print(f"jumps: {fmt}, heads of {d}, {history} cached, {copies} x", flush=True)
    gen = torch.Generator().manual_seed(d + history)
    total = history + rows
    pages = -(-total // 16)
    n = len(JUMPS)
    q0 = torch.randn(hq // 2, d, generator=gen)
    q0 = (q0 / q0.norm(dim=1, keepdim=True)).mean(0)
    q0 = q0 / q0.norm() * d ** 0.5
    q = (q0 + 0.05 * torch.randn(n, rows, hq, d, generator=gen)).half()
    k = 0.3 * torch.randn(n, pages * 16, hkv, d, generator=gen)
    v = torch.randn(n, pages * 16, hkv, d, generator=gen)
    for b, jumps in enumerate(JUMPS):
        for step, tile in enumerate(jumps):             # each some 2^10 times as likely as what came before
            at = 64 * tile + (40 if (b + step) % 2 else 9)
            if at < total:
                k[b, at] = 7.0 * (step + 1) * q0 / d ** 0.5
    scales = None
    if fmt == "f16":
        pool = torch.cat([k, v], 2).half()
        full = pool.double()
    else:
        scales = torch.tensor([0.05] * hkv + [0.04] * hkv)
        full = torch.cat([k, v], 2) / scales[None, None, :, None]
        pool = full.round().clamp(-127, 127).to(torch.int8)
        full = pool.double() * scales.double()[None, None, :, None]
        scales = scales.to(DEV)
    table = torch.arange(n * pages, dtype=torch.int32).view(n, pages).repeat(copies, 1).to(DEV)
    out = ops.paged_prefill(q.repeat(copies, 1, 1, 1).view(-1, hq, d).to(DEV), pool.view(-1, 2 * hkv, d).to(DEV), table,
                            torch.arange(0, n * copies * rows + 1, rows, dtype=torch.int32, device=DEV),
                            torch.full((n * copies,), history, dtype=torch.int32, device=DEV), rows, d ** -0.5,
                            kv_scales=scales, max_kv_len=total)
    torch.cuda.synchronize()
    out = out.view(copies, n, rows, hq, d)
    assert bool((out == out[:1]).all())
    seen = torch.arange(total)[None, :] <= history + torch.arange(rows)[:, None]
    qd = q.double()
    for h in range(hq):
        s = torch.matmul(qd[:, :, h], full[:, :total, h // 2].transpose(1, 2).contiguous()) * d ** -0.5
        p = torch.softmax(s.masked_fill(~seen, -torch.inf), -1)
        ref = torch.matmul(p, full[:, :total, hkv + h // 2])
        assert_attention_close(out[0, :, :, h], ref.numpy(), f"{fmt} {d} {history} head {h}")
