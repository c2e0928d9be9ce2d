"""Several small device arrays copied in one launch (ops.copy_tensors over litekv_copy_segments)."""

import pytest
import torch

from llama_lite_npu_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("count,batch,width", [
    (1, 1, 1), (7, 32, 257), (8, 3, 1023), (9, 5, 1025),     # one launch holds 8 arrays, a block 1024 words
    (2, 128, 2048),
])
def test_copy_tensors(count, batch, width):
    """Every array arrives, nothing beside it changes: contiguous 64-bit and 32-bit rows, and a table
    narrower than the one it goes into."""
    print(f"copy {count} arrays, table {batch} x {width}", flush=True)
    gen = torch.Generator().manual_seed(count)
    table = torch.randint(-2**31, 2**31 - 1, (batch, width), dtype=torch.int32, generator=gen).to(DEV)
    wide = torch.full((batch, width + 3), 7, dtype=torch.int32, device=DEV)
    pairs, want = [(wide[:, :width], table)], []
    for i in range(count - 1):
        src = torch.randint(-2**62, 2**62, (batch, 1), generator=gen).to(torch.int64 if i % 2 else torch.int32).to(DEV)
        pairs.append((torch.zeros_like(src), src))
    ops.copy_tensors(pairs)
    torch.cuda.synchronize()
    assert all(torch.equal(dst, src) for dst, src in pairs)
    assert bool((wide[:, width:] == 7).all())


def test_copies_of_another_kind_still_happen():
    """Other types, host sources, broadcast rows, odd byte counts: as dst.copy_(src)."""
    f = torch.arange(5, dtype=torch.float32, device=DEV)
    pairs = [(torch.zeros(5, dtype=torch.int64, device=DEV), f), (torch.zeros(3, device=DEV), torch.ones(3)),
             (torch.zeros((2, 4), dtype=torch.int32, device=DEV), torch.arange(4, dtype=torch.int32, device=DEV).expand(2, 4)),
             (torch.zeros(3, dtype=torch.uint8, device=DEV), torch.ones(3, dtype=torch.uint8, device=DEV)),
             (torch.zeros((4, 2), dtype=torch.int32, device=DEV), torch.arange(8, dtype=torch.int32, device=DEV).view(2, 4).t())]
    ops.copy_tensors(pairs)
    torch.cuda.synchronize()
    for dst, src in pairs:
        assert torch.equal(dst.cpu(), src.to(dst.dtype).cpu())
    with pytest.raises(_lib.LiteKVError, match="count"):
        _lib.check(_lib.load().litekv_copy_segments(None, 9, None))
