"""Into how many slices the library cuts a paged prefill along its keys (no GPU: without one the rule counts
256 compute units). Measured on an MI355X, us: 32/8 heads of 64, 8 to 64 rows over 1000 tokens 12.1 to 12.7 uncut,
8.6 to 10.6 in 8 slices; 64/8 heads of 128, 128 rows over 2048 tokens 30 uncut, 25 in 4."""

import pytest
import torch

from llama_lite_npu_amd import _lib

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the rule counts the device's compute units")


def _slices(*shape):
    return int(_lib.load().litekv_paged_prefill_key_slices(*shape))


@pytest.mark.parametrize("batch,rows", [(1, 8), (1, 16), (1, 64), (2, 8), (2, 16), (4, 8)])
def test_few_rows_of_narrow_heads_over_a_thousand_tokens_are_cut(batch, rows):
    assert _slices(batch, 32, 8, 64, rows, 1000 + rows) >= 6


@pytest.mark.parametrize("rows", [8, 64, 128, 512])
@pytest.mark.parametrize("head_dim", [64, 128])
def test_few_keys_are_not(head_dim, rows):
    for keys in (rows, 200 + rows):
        assert _slices(1, 32, 8, head_dim, rows, keys) == 1


def test_chunks_over_long_histories():
    assert _slices(1, 64, 8, 128, 128, 32768) == 8 and _slices(1, 64, 8, 128, 128, 2048 + 128) == 4
    assert _slices(1, 64, 8, 128, 512, 2048 + 512) == 1 and _slices(4, 64, 8, 128, 512, 32768) == 1
    assert _slices(1, 32, 8, 64, 256, 16384) >= 2
