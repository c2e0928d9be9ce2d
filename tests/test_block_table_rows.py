"""Block tables as the decode kernels take them: they read rows to the end of their stride."""

import pytest
import torch

from llama_lite_npu_amd.ops import _table_rows

WIDE = torch.arange(6 * 20, dtype=torch.int32).view(6, 20)


@pytest.mark.parametrize("table", [
    WIDE, WIDE[:, :7], WIDE[:, 13:], WIDE[2:4, 5:9], WIDE[5:, 17:], WIDE[5:6], WIDE[4:, 19:], WIDE[1:2, 3:8],
    WIDE[:, 3:].contiguous(), WIDE[::2, 15:], WIDE[:0],
], ids=str)
def test_every_row_ends_within_the_storage(table):
    rows, stride = _table_rows(table)
    assert torch.equal(rows, table) and stride >= table.shape[1]
    assert rows.storage_offset() + rows.shape[0] * stride <= rows.untyped_storage().nbytes() // 4
    for b in range(table.shape[0]):        # row b as a kernel sees it
        flat = torch.as_strided(rows, (stride,), (1,), rows.storage_offset() + b * stride)
        assert torch.equal(flat[:table.shape[1]], table[b])


def test_tables_that_are_whole_are_not_copied():
    for table in (WIDE, WIDE[1:4], WIDE[3:4], WIDE[:, :7]):
        assert _table_rows(table)[0] is table
