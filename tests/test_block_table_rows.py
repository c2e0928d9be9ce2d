"""Block tables as the decode kernels take them: they read rows to the end of their stride."""

import subprocess
from pathlib import Path

import pytest
import torch

from llama_lite_npu_amd import build
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


def test_a_prefill_reads_no_entry_outside_its_row(tmp_path):
    """prefill_tile.h's entry of a page, compiled for the host: pages a sequence has, pages past the row, and the
    pages in front of it that a sequence without a key asks for."""
    csrc = Path(build.CSRC)
    source = tmp_path / "entry.hip"
    source.write_text('#include <cstdio>\n#include "head_dim.h"\n#include "prefill_tile.h"\n'
                      "int main() {\n  int p, s, n;\n  while (scanf(\"%d %d %d\", &p, &s, &n) == 3)\n"
                      "    printf(\"%u\\n\", litekv::LITEKV_HD_NS::prefill_tile::table_entry(p, s, n));\n}\n")
    subprocess.run([build._hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-Wno-inline-asm", f"-I{csrc}",
                    str(source), "-o", str(tmp_path / "entry")], check=True, capture_output=True)
    pages = [0, 1, 2, 3, 4, 7, 8, 63, 64, 1000, 2 ** 27 - 1, 2 ** 31 - 1, -1, -2, -3, -4, -5, -64, -1000, -2 ** 27, -2 ** 31]
    asked = [(p, shift, stride) for p in pages for shift in (0, 1, 2, 3) for stride in (1, 2, 5, 16, 2 ** 20)]
    out = subprocess.run([str(tmp_path / "entry")], input="\n".join("%d %d %d" % a for a in asked), text=True, check=True,
                         capture_output=True).stdout.split()
    for (page, shift, stride), entry in zip(asked, map(int, out), strict=True):
        assert entry == (min(page >> shift, stride - 1) if page >= 0 else stride - 1), (page, shift, stride)
