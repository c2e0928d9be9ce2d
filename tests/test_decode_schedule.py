"""Host rule that picks the decode schedule of a step (no GPU): the qualitative behaviour the
measurements behind its constants showed, at the sizes the benchmark configurations name.
0 = balanced, 1 = one wavefront per (sequence, kv head), 4 / 8 / 16 = splits per sequence + merge."""

import pytest
import torch

from llama_lite_npu_amd.ops import SPLIT_COUNTS, decode_schedule, decode_schedule_estimates, pool_head_dim
from llama_lite_npu_amd import _lib, ops

TOK = 4096  # K + V bytes of a token: 8 kv heads, fp16


def pages(n):
    return (n + 15) // 16


def uniform(batch, tokens, **kw):
    return decode_schedule(batch, 8, pages(tokens), batch * pages(tokens), TOK, **kw)


def test_many_short_sequences_take_one_wavefront_each():
    for batch in (32, 64, 128, 256, 1024):
        assert uniform(batch, 64) == 1
    assert uniform(128, 256) == 1
    assert uniform(8, 40) == 1


def test_small_batches_take_several_splits_per_sequence():
    # measured: 1 to 8 sequences of 256 to 1024 tokens run 1.2 to 1.5 times faster in 8 or 16 splits
    for batch in (1, 2, 4, 8):
        for tokens in (256, 1024):
            assert uniform(batch, tokens) in (8, 16), (batch, tokens)
    assert uniform(8, 2048) in (8, 16)
    # from a few thousand tokens on, a step of few rows merges its long rows over several workgroups
    # and the balanced cut is the faster one again
    assert uniform(1, 4096) == 0 and uniform(2, 8192) == 0 and uniform(4, 8192) == 0
    c1 = [38, 129, 512, 1001]
    assert decode_schedule(4, 8, max(map(pages, c1)), sum(map(pages, c1)), TOK, heads_per_kv_head=2) in (8, 16)


def test_long_or_large_batches_stay_balanced():
    assert uniform(8, 16384) == 0 and uniform(16, 8192) == 0 and uniform(128, 2048) == 0
    assert uniform(1, 32768) == 0                             # one long sequence: the balanced cut
    # one long sequence among many short ones: the chain of its pages decides
    assert decode_schedule(128, 8, pages(8192), 127 * pages(64) + pages(8192), TOK) == 0
    # large batches of a few hundred tokens are bound by bytes, which the balanced cut streams faster
    assert uniform(1024, 512) == 0
    assert decode_schedule(32, 8, pages(4097), 32 * pages(2200), TOK) == 0             # C2
    assert decode_schedule(128, 4, pages(32769), 128 * pages(20000), TOK // 2) == 0    # C5


def test_the_choice_moves_one_way_with_the_longest_sequence():
    # one wavefront, then (small batches) several splits, then balanced: apart from a few pages
    # around a boundary (pages per split and per chunk are whole numbers) the choice never moves back
    for batch in (1, 4, 16, 64, 256):
        picks = [decode_schedule(batch, 8, mp, batch * mp, TOK) for mp in range(1, 2200)]
        order = [0 if p == 1 else 2 if p == 0 else 1 for p in picks]
        assert picks[0] == 1 and picks[-1] == 0
        backwards = [i for i in range(1, len(order)) if order[i] < order[i - 1]]
        assert len(backwards) <= 4, (batch, backwards)
        for i in backwards:                      # and it is back within 32 pages
            assert max(order[i:i + 32]) >= order[i - 1]


def test_degenerate_inputs():
    assert decode_schedule(0, 8, 0, 0, TOK) == 0 and decode_schedule(4, 8, 0, 0, TOK) == 0
    estimates = decode_schedule_estimates(4, 8, 10, 30, TOK)
    assert set(estimates) == {0, 1} | set(SPLIT_COUNTS) and all(t > 0 for t in estimates.values())


def test_splits_are_bounded_by_the_wavefronts_of_the_launch():
    for batch in (1, 2, 4, 8, 16, 32, 64, 128, 256, 1024):
        for tokens in (16, 64, 256, 1024, 4096, 16384):
            pick = uniform(batch, tokens)
            assert pick in (0, 1) + SPLIT_COUNTS
            assert pick <= 1 or batch * pick * 8 <= 2048
            wide = uniform(batch, tokens, heads_per_kv_head=32)     # two wavefronts per kv head
            assert wide <= 1 or batch * wide * 8 * 2 <= 2048


def test_wide_head_groups_lean_away_from_the_balanced_schedule():
    # 16 query heads per kv head slow the balanced schedule only: some steps leave it, none joins it
    moved = 0
    for batch in (8, 16, 64, 128):
        for mp in range(1, 400):
            narrow = decode_schedule(batch, 8, mp, batch * mp, TOK)
            wide = decode_schedule(batch, 8, mp, batch * mp, TOK, heads_per_kv_head=16)
            assert narrow != 0 or wide in (0, 1) + SPLIT_COUNTS
            assert wide != 0 or narrow == 0
            moved += narrow == 0 and wide != 0
    assert moved > 0


def test_the_schedule_in_use_keeps_an_advantage():
    changed = kept = 0
    for batch in (1, 4, 8, 16, 32):
        for mp in range(1, 700, 3):
            free = decode_schedule(batch, 8, mp, batch * mp, TOK)
            for current in (0, 1, 4, 8, 16):
                sticky = decode_schedule(batch, 8, mp, batch * mp, TOK, current=current, hysteresis=1.1)
                assert sticky in (free, current)             # hysteresis only ever keeps the current one
                kept += sticky == current != free
                changed += sticky != current
    assert kept > 0 and changed > 0
    # and a schedule that is not a candidate for the step (too many wavefronts) is not kept
    assert decode_schedule(512, 8, 4, 2048, TOK, current=16, hysteresis=2.0) in (0, 1)


def test_page_size_does_not_change_the_choice_for_the_same_tokens():
    for batch, tokens in ((2, 1024), (8, 512), (64, 256), (16, 16384)):
        picks = {decode_schedule(batch, 8, tokens // ps, batch * tokens // ps, TOK, page_size=ps)
                 for ps in (16, 64, 256)}
        assert len(picks) == 1, (batch, tokens, picks)


@pytest.mark.parametrize("batch,hkv,group,head_dim,code_bytes,longest,mean,want", [
    (128, 4, 8, 128, 1, 32464, 19636, 0),    # int8, 428 us per layer against 571 in 4 splits
    (42, 4, 8, 128, 1, 23920, 16034, 0),     # int8, 126 against 198 in 8 splits
    (12, 8, 4, 64, 2, 2909, 1573, 0),        # rows of 64: 16 us against 18 in 16 splits
    (12, 8, 2, 128, 2, 512, 484, 8),         # 11.6 us against 14.8 balanced
    (1, 8, 2, 128, 2, 779, 779, 16),
])
def test_the_choice_knows_the_pool_format_the_head_dim_and_the_kv_heads(batch, hkv, group, head_dim, code_bytes,
                                                                        longest, mean, want):
    pick = decode_schedule(batch, hkv, pages(longest), batch * pages(mean), 2 * hkv * head_dim * code_bytes,
                           heads_per_kv_head=group, head_dim=head_dim)
    assert pick in ((8, 16) if want in (8, 16) else (want,))


@pytest.mark.parametrize("batch,hkv,group,head_dim,code_bytes,longest,rest,want", [
    # one long sequence among short ones, us measured per layer: {0: balanced, 1, 4, 8, 16: wavefronts per sequence}
    (128, 8, 8, 128, 2, 512, 32, (1, 4)),      # {0: 28.5, 1: 20.5, 4: 21.0}
    (128, 8, 8, 128, 1, 512, 32, (1, 4)),      # {0: 26.4, 1: 18.9, 4: 18.4}
    (128, 8, 8, 128, 1, 256, 16, (1,)),        # {0: 16.4, 1: 11.9, 4: 17.5}
    (16, 8, 8, 128, 1, 2048, 128, (8, 16)),    # {0: 19.4, 1: 56.5, 4: 21.0, 8: 15.6, 16: 14.0}
    (32, 4, 8, 128, 1, 2048, 128, (8, 16)),    # {0: 18.9, 1: 67.9, 4: 23.9, 8: 17.2, 16: 14.4}
    (64, 4, 8, 128, 1, 1024, 64, (8, 16)),     # {0: 18.1, 1: 36.4, 4: 17.2, 8: 13.9, 16: 16.2}
    (256, 4, 8, 128, 2, 512, 32, (1, 4)),      # {0: 27.3, 1: 21.0, 4: 21.2}
    (128, 8, 4, 64, 2, 256, 16, (1, 4)),       # {0: 13.4, 1: 10.4, 4: 11.6}
    # equal lengths
    (64, 8, 8, 128, 1, 512, 512, (1, 4)),      # {0: 25.8, 1: 20.6, 4: 21.2, 8: 26.8}
    (2, 8, 8, 128, 1, 64, 64, (1,)),           # {0: 9.9, 1: 6.2, 4: 7.1, 8: 7.8, 16: 7.9}
])
def test_steps_whose_choice_cost_a_quarter(batch, hkv, group, head_dim, code_bytes, longest, rest, want):
    total = pages(longest + 1) + (batch - 1) * pages(rest + 1)
    pick = decode_schedule(batch, hkv, pages(longest + 1), total, 2 * hkv * head_dim * code_bytes,
                           heads_per_kv_head=group, head_dim=head_dim)
    assert pick in want


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("batch,tokens", [(1, 300), (24, 128), (4, 80), (12, 2900), (64, 512), (128, 64)])
def test_flash_decoding_asks_for_the_width_it_is_given(monkeypatch, batch, tokens, d):
    """Rows of 64 fp16 elements have the bytes of 128 codes: the wrapper says which it has."""
    from llama_lite_npu_amd import kernels

    hq, hkv = 32, 8
    taken = []
    monkeypatch.setattr(ops, "paged_decode", lambda *a, **kw: taken.append(kw.get("num_splits", 0)))
    pool = torch.zeros((16, 2 * hkv, d), dtype=torch.float16)
    kernels.flash_decoding(torch.zeros((batch, hq, d), dtype=torch.float16), pool[:, :hkv], pool[:, hkv:], 0.1,
                           torch.zeros((batch, tokens), dtype=torch.int32), torch.full((batch,), tokens), tokens)
    assert taken == [decode_schedule(batch, hkv, pages(tokens), batch * pages(tokens), 2 * hkv * d * 2,
                                     heads_per_kv_head=hq // hkv, head_dim=d)]


def test_a_plan_without_an_element_type_is_one_of_fp16():
    assert pool_head_dim(2 * 8 * 64 * 2, 8) == 64 and pool_head_dim(2 * 8 * 128 * 2, 8) == 128
    assert pool_head_dim(2 * 8 * 64 * 2, 8, torch.float16) == 64
    assert pool_head_dim(2 * 8 * 128, 8, torch.int8) == 128 and pool_head_dim(2 * 8 * 64, 8, torch.uint8) == 64
    assert pool_head_dim(2 * 4 * 256 * 2, 4) == 128                    # the rule's widths are 64 and 128


@pytest.mark.parametrize("hkv", [1, 2, 3, 4, 5, 8, 9, 16])
def test_the_rule_counts_the_chunks_a_launch_has(hkv):
    """Of 256 compute units, which is also what the library takes where it finds no device."""
    if not torch.cuda.is_available():
        assert ops._whole_device_chunks(hkv) == _lib.load().litekv_paged_decode_balanced_chunks(hkv)
    for group in (8, 16, 32, 64):              # slices of a kv head's query heads do not change the count
        shape = (16, hkv, 100, 1600, 4 * hkv * 128)
        same = decode_schedule_estimates(*shape, heads_per_kv_head=group, chunks=ops._whole_device_chunks(hkv))
        assert decode_schedule_estimates(*shape, heads_per_kv_head=group) == same
        few = decode_schedule_estimates(*shape, heads_per_kv_head=group, chunks=7)
        assert few[0] > same[0] and {k: v for k, v in few.items() if k} == {k: v for k, v in same.items() if k}


@pytest.mark.parametrize("hq,hkv,batch,tokens,want", [
    (32, 1, 8, 4000, (16,)),        # 18.8 us against 31.2 balanced (2048 chunks of 32 partial rows each)
    (32, 1, 16, 8000, (16,)),       # 31.3 against 48.0
    (32, 2, 128, 2000, (4, 8)),     # 50.5 and 56.1 against 62.8
    (64, 1, 2, 16000, (16,)),       # 46.8 against 55.2
    (32, 1, 1, 2000, (0, 16)),      # 11.9 balanced
])
def test_wide_groups_are_charged_for_their_partial_rows(hq, hkv, batch, tokens, want):
    pick = decode_schedule(batch, hkv, pages(tokens + 1), batch * pages(tokens + 1), 4 * hkv * 128,
                           heads_per_kv_head=hq // hkv)
    assert pick in want


def test_a_large_step_of_narrow_codes_stays_balanced():
    # 62 sequences of 1850 to 2799 tokens, 32/8 heads of 64 over int8: 43.7 us, 48.1 in 4 splits
    for longest, mean in ((2787, 2332), (5600, 4800)):
        assert decode_schedule(62, 8, pages(longest), 62 * pages(mean), 2 * 8 * 64, heads_per_kv_head=4, head_dim=64) == 0
