"""GPU: the splits schedule attends two pages per step, with one step's or two steps' pages in flight
by the number of the launch's wavefronts. Lengths on both sides of a page, of a pair and of two, in
splits of odd and even page counts, every pool format and both head dims: each sequence as float64
arithmetic gives it, and the same bits in a small launch and in a large one. Slots past the end of
a sequence hold NaN (codes: the largest there are)."""

import pytest
import torch

from llama_lite_npu_amd import ops, workloads
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# tokens with the step's own: 1 to 9 pages, the last with one token, all but one, all
LENS = [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 80, 81, 96, 112, 128, 129, 144]


def _decoded(pool, fmt, scales, hkv):
    if fmt == "f16":
        return pool.double()
    rows = pool.double() if fmt == "int8" else pool.view(torch.float8_e4m3fn).double()
    return rows * scales.double()[None, :, None]


@pytest.mark.parametrize("splits", [1, 2, 4])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("fmt", ["f16", "fp8", "int8"])
def test_pairs_of_pages(fmt, head_dim, splits):
    hq, hkv = 6, 2
    print(f"page pairs: {fmt} pool, heads of {head_dim}, {splits} splits", flush=True)
    case = workloads.make_decode_case("pairs", 83, [n - 1 for n in LENS], hq, hkv, device=DEV, head_dim=head_dim)
    slots = torch.arange(case.kv_pool.shape[0], dtype=torch.int32, device=DEV)
    scales = None
    pool = case.kv_pool.clone()
    if fmt != "f16":
        scales = torch.tensor([0.031, 0.043, 0.027, 0.039], device=DEV)
        pool = torch.empty(case.kv_pool.shape, dtype=torch.uint8 if fmt == "fp8" else torch.int8, device=DEV)
        ops.kv_append_quantised(case.kv_pool[:, :hkv], case.kv_pool[:, hkv:], slots, pool, scales)
    used = torch.zeros(pool.shape[0], dtype=torch.bool, device=DEV)
    for b, n in enumerate(LENS):
        for t in range(n - 1):
            used[int(case.block_table[b, t // 16]) * 16 + t % 16] = True
    pool[~used] = float("nan") if fmt == "f16" else 0x7e if fmt == "fp8" else 127
    ws_floats = len(LENS) * hq * splits * (head_dim + 1)

    def run(copies):
        seq, table = case.seq_lens.repeat(copies), case.block_table.repeat(copies, 1).contiguous()
        kn, vn = case.k_new.repeat(copies, 1, 1), case.v_new.repeat(copies, 1, 1)
        mine = pool.clone()     # (every copy of a sequence appends the same row to the same slot)
        ws = torch.full((ws_floats * copies,), float("nan"), device=DEV)
        out = ops.paged_decode(case.q.repeat(copies, 1, 1), mine, table, seq, case.softmax_scale, max_splits=splits,
                               min_pages_per_split=1, workspace=ws, k_new=kn, v_new=vn, kv_scales=scales)
        separate = ops.paged_decode(case.q.repeat(copies, 1, 1), mine, table, seq, case.softmax_scale, max_splits=splits,
                                    min_pages_per_split=1, workspace=ws, kv_scales=scales)
        torch.cuda.synchronize()
        assert torch.equal(out, separate)
        return out, mine

    out, pool_after = run(1)                                    # 19 * 2 * splits wavefronts
    many, _ = run(-(-1100 // (len(LENS) * hkv * splits)))       # over 1024
    for rows in many.split(len(LENS)):
        assert torch.equal(rows, out)
    full = _decoded(pool_after, fmt, scales, hkv).cpu()
    q = case.q.double().cpu()
    ref = torch.empty_like(q)
    for b, n in enumerate(LENS):
        at = torch.tensor([int(case.block_table[b, t // 16]) * 16 + t % 16 for t in range(n)])
        k, v = full[at, :hkv], full[at, hkv:]
        for h in range(hq):
            p = torch.softmax(k[:, h // 3] @ q[b, h] * case.softmax_scale, 0)
            ref[b, h] = p @ v[:, h // 3]
    assert_attention_close(out, ref.numpy(), f"{fmt} {head_dim} {splits}")
