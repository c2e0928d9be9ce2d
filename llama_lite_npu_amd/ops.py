"""Block-table-native operators over liblitekv (PyTorch-ROCm tensors in, C ABI out).

PyTorch supplies device memory and the current stream; every byte of the path
is moved or computed by the HIP kernels behind include/litekv.h. All calls only
enqueue work on ``torch.cuda.current_stream()``.
"""

from __future__ import annotations

import ctypes
import math
from typing import Optional, Sequence

import torch

from . import _lib

PAGE_SIZE = 16
HEAD_DIM = 128


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _stream() -> int:
    """The current stream of the current device as the C ABI takes it (torch.cuda.current_stream() builds
    a Stream object around the same number, which takes longer than the rest of a wrapper's checks)."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


# The wrappers run once per layer and step: checks on their path are plain conditions, and the message
# of one is only put together when it fails.
def _need(cond: bool, msg: str) -> None:
    if not cond:
        raise ValueError(msg)


def _dev_half(name: str, t: torch.Tensor) -> None:
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU")
    if t.dtype is not torch.float16:
        raise ValueError(f"{name} must be float16, got {t.dtype}")


FP8_DTYPES = (torch.uint8, torch.float8_e4m3fn)
INT8_DTYPES = (torch.int8,)
_Q8_DTYPES = FP8_DTYPES + INT8_DTYPES


def _dev_pool(name: str, t: torch.Tensor) -> None:
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU")
    if t.dtype is not torch.float16 and t.dtype not in _Q8_DTYPES:
        raise ValueError(f"{name} must be float16, fp8 or int8, got {t.dtype}")


def is_fp8_pool(kv_pool: torch.Tensor) -> bool:
    """An fp8 pool holds one E4M3 code per element (a uint8 or float8_e4m3fn tensor)."""
    return kv_pool.dtype in FP8_DTYPES


def is_int8_pool(kv_pool: torch.Tensor) -> bool:
    """An int8 pool holds one signed 8-bit code per element (a torch.int8 tensor)."""
    return kv_pool.dtype in INT8_DTYPES


def is_quantised_pool(kv_pool: torch.Tensor) -> bool:
    """A pool of 8-bit codes (fp8 or int8) with one fp32 scale per kv head: value = code * scale."""
    return kv_pool.dtype in _Q8_DTYPES


def _q8_entry(lib, stem: str, kv_pool: torch.Tensor):
    """The library's entry point `stem` for the pool's 8-bit format (litekv_<stem>_fp8 / _int8)."""
    return getattr(lib, f"litekv_{stem}_{'int8' if is_int8_pool(kv_pool) else 'fp8'}")


def _dev_fp8_pool(kv_pool: torch.Tensor, scales: Optional[torch.Tensor], num_kv_heads: int) -> None:
    if not (kv_pool.is_cuda and kv_pool.dtype in _Q8_DTYPES):
        raise ValueError(f"kv_pool must be an fp8 (uint8 / float8_e4m3fn) or int8 GPU tensor, got {kv_pool.dtype}")
    if scales is None:
        raise ValueError("a pool of 8-bit codes needs its per-head scales")
    if not (scales.is_cuda and scales.dtype is torch.float32 and scales.is_contiguous()
            and scales.numel() == 2 * num_kv_heads):
        raise ValueError("scales must be float32 [2 * Hkv] on the GPU (K heads, then V heads)")


def _dev_i32(name: str, t: torch.Tensor) -> torch.Tensor:
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU")
    if t.dtype is not torch.int32:
        t = t.to(torch.int32)  # device-side cast, no host sync
    return t if t.is_contiguous() else t.contiguous()


def _table_rows(t: torch.Tensor) -> tuple:
    """(block table, entries per row) as the kernels take it: they may read a row to the end of its
    stride, whatever the lengths are, so no row may be said to reach past the tensor's storage. (The
    one row of a view counts as contiguous with any stride; a view of some columns of a wider table
    ends within its last row.)"""
    width, stride = t.shape[1], t.stride(0)
    if stride == width or t.shape[0] == 1:
        return t, max(1, width)
    if t.storage_offset() + t.shape[0] * stride > t.untyped_storage().nbytes() // t.element_size():
        return t.contiguous(), max(1, width)
    return t, stride


def _rows(name: str, t: torch.Tensor) -> int:
    """Token stride of a [T, H, D] tensor whose [H, D] block is contiguous."""
    shape, stride = t.shape, t.stride()
    if len(shape) != 3:
        raise ValueError(f"{name} must be [tokens, heads, head_dim]")
    if stride[2] != 1 or stride[1] != shape[2]:
        raise ValueError(f"{name}: [heads, head_dim] block must be contiguous")
    return stride[0] if shape[0] > 1 else max(stride[0], shape[1] * shape[2])


def pool_geometry(kv_pool: torch.Tensor, page_size: int = PAGE_SIZE):
    """(num_slots, num_kv_heads, head_dim, num_pages, page_bytes) of a [slots, 2*Hkv, D] pool."""
    shape = kv_pool.shape
    if len(shape) != 3 or not kv_pool.is_contiguous():
        raise ValueError("kv_pool must be contiguous [slots, 2*Hkv, D]")
    slots, two_h, d = shape
    if two_h % 2 != 0:
        raise ValueError("kv_pool dim 1 must be 2 * num_kv_heads")
    if slots % page_size != 0:
        raise ValueError("kv_pool slots must be a multiple of page_size")
    return slots, two_h // 2, d, slots // page_size, page_size * two_h * d * kv_pool.element_size()


def kv_append(k: torch.Tensor, v: torch.Tensor, slot_mapping: torch.Tensor, kv_pool: torch.Tensor) -> None:
    """kv_pool[slot_mapping[t]] = concat(k[t], v[t]) for every token t (bit exact, in place)."""
    _dev_half("k", k), _dev_half("v", v), _dev_half("kv_pool", kv_pool)
    slots, hkv, d, _, _ = pool_geometry(kv_pool, 1)
    if not (k.shape == v.shape):
        raise ValueError("k and v must have the same shape")
    if not (k.shape[1] == hkv and k.shape[2] == d):
        raise ValueError(f"k/v heads {tuple(k.shape[1:])} do not match pool ({hkv}, {d})")
    slot_mapping = _dev_i32("slot_mapping", slot_mapping)
    t = k.shape[0]
    if not (slot_mapping.numel() == t):
        raise ValueError("slot_mapping must hold one slot per token")
    lib = _lib.load()
    _lib.check(lib.litekv_kv_append(_ptr(k), _ptr(v), _rows("k", k), _rows("v", v), _ptr(slot_mapping),
                                    _ptr(kv_pool), t, hkv, d, slots, _stream()))


def kv_append_quantised(k: torch.Tensor, v: torch.Tensor, slot_mapping: torch.Tensor, kv_pool: torch.Tensor,
                        scales: torch.Tensor) -> None:
    """kv_pool[slot_mapping[t]] = code(concat(k[t], v[t]) / scale of the head) for every token t, in the
    pool's format (E4M3 for a uint8 / float8_e4m3fn pool, int8 for a torch.int8 pool);
    scales is float32 [2 * Hkv]: K-head scales, then V-head scales."""
    _dev_half("k", k), _dev_half("v", v)
    slots, hkv, d, _, _ = pool_geometry(kv_pool, 1)
    _dev_fp8_pool(kv_pool, scales, hkv)
    _need(k.shape == v.shape and k.shape[1] == hkv and k.shape[2] == d, "k / v must be [T, Hkv, D] matching the pool")
    slot_mapping = _dev_i32("slot_mapping", slot_mapping)
    t = k.shape[0]
    _need(slot_mapping.numel() == t, "slot_mapping must hold one slot per token")
    lib = _lib.load()
    _lib.check(_q8_entry(lib, "kv_append", kv_pool)(_ptr(k), _ptr(v), _rows("k", k), _rows("v", v),
                                                    _ptr(slot_mapping), _ptr(kv_pool), _ptr(scales), t, hkv, d,
                                                    slots, _stream()))


kv_append_fp8 = kv_append_quantised     # the name from before int8 pools


def page_dequant(kv_pool: torch.Tensor, dst_pool: torch.Tensor, src_ids: torch.Tensor,
                 dst_ids: Optional[torch.Tensor], scales: torch.Tensor, page_size: int = PAGE_SIZE) -> None:
    """dst_pool[page dst_ids[i]] (fp16) = decoded page src_ids[i] of the fp8 pool; dst_ids None means page i."""
    _dev_half("dst_pool", dst_pool)
    _, hkv, d, n_src, _ = pool_geometry(kv_pool, page_size)
    _, hkv_d, d_d, n_dst, _ = pool_geometry(dst_pool, page_size)
    _dev_fp8_pool(kv_pool, scales, hkv)
    _need((hkv, d) == (hkv_d, d_d), "pools differ in head geometry")
    src_ids = _dev_i32("src_ids", src_ids)
    if dst_ids is not None:
        dst_ids = _dev_i32("dst_ids", dst_ids)
        _need(dst_ids.numel() == src_ids.numel(), "src_ids and dst_ids differ in length")
    lib = _lib.load()
    fn = lib.litekv_page_dequant_int8 if is_int8_pool(kv_pool) else lib.litekv_page_dequant
    _lib.check(fn(_ptr(kv_pool), _ptr(dst_pool), _ptr(src_ids), _ptr(dst_ids), src_ids.numel(),
                  _ptr(scales), hkv, d, page_size, n_src, n_dst, _stream()))


def qk_norm_rope_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, slot_mapping: torch.Tensor,
                        kv_pool: torch.Tensor, q_norm_weight: Optional[torch.Tensor] = None,
                        k_norm_weight: Optional[torch.Tensor] = None, cos: Optional[torch.Tensor] = None,
                        sin: Optional[torch.Tensor] = None, rms_eps: float = 1e-6,
                        kv_scales: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Per-head RMSNorm (optional) and rotary embedding (optional) of q [T, Hq, D] in place and of
    k [T, Hkv, D] on its way into the pool, plus the append of v: one launch for the reference's
    skip_rmsnorm x2 + rope_emb_forward + cat + update_kv_buffer. cos / sin are [T, >= D/2] rows of
    each token's position. An fp8 pool (with its ``kv_scales``) receives the quantised rows. Returns q."""
    if q.is_cuda:
        done = _lib.calls().qk_norm_rope_append(q, k, v, slot_mapping, kv_pool, q_norm_weight, k_norm_weight, cos, sin,
                                                rms_eps, kv_scales, _stream())
        if done is not None:
            if done is not True:        # a status: q may have been written all the same, so never a second time
                _lib.check(done)
            return q
    # (not a plain call: found out below)
    _dev_half("q", q), _dev_half("k", k), _dev_half("v", v)
    slots, hkv, d, _, _ = pool_geometry(kv_pool, 1)
    fp8 = is_quantised_pool(kv_pool)
    if fp8:
        _dev_fp8_pool(kv_pool, kv_scales, hkv)
    else:
        _dev_half("kv_pool", kv_pool)
    t, hq = q.shape[0], q.shape[1]
    if not (q.dim() == 3 and q.shape[2] == d):
        raise ValueError("q must be [T, Hq, D]")
    if not (k.shape == (t, hkv, d) and v.shape == (t, hkv, d)):
        raise ValueError("k / v must be [T, Hkv, D] matching the pool")
    if not ((q_norm_weight is None) == (k_norm_weight is None)):
        raise ValueError("q_norm_weight and k_norm_weight go together")
    if not ((cos is None) == (sin is None)):
        raise ValueError("cos and sin go together")
    if q_norm_weight is not None:
        _dev_half("q_norm_weight", q_norm_weight), _dev_half("k_norm_weight", k_norm_weight)
        if not (q_norm_weight.numel() == d and k_norm_weight.numel() == d
                and q_norm_weight.is_contiguous() and k_norm_weight.is_contiguous()):
            raise ValueError("norm weights must be contiguous [D]")
    cs_stride = 0
    if cos is not None:
        _dev_half("cos", cos), _dev_half("sin", sin)
        if cos.dim() != 2 or sin.dim() != 2:
            cos, sin = cos.reshape(-1, cos.shape[-1]), sin.reshape(-1, sin.shape[-1])
        if not (cos.shape == sin.shape and cos.shape[0] == t and cos.shape[1] >= d // 2):
            raise ValueError("cos / sin must be [T, >= D/2]")
        if not (cos.stride(1) == 1 and sin.stride(1) == 1 and cos.stride(0) == sin.stride(0)):
            raise ValueError("cos / sin rows must be contiguous with equal row strides")
        cs_stride = cos.stride(0)
    slot_mapping = _dev_i32("slot_mapping", slot_mapping)
    if not (slot_mapping.numel() == t):
        raise ValueError("slot_mapping must hold one slot per token")
    lib = _lib.load()
    if fp8:
        _lib.check(_q8_entry(lib, "qk_norm_rope_append", kv_pool)(
            _ptr(q), _rows("q", q), _ptr(k), _rows("k", k), _ptr(v), _rows("v", v), _ptr(q_norm_weight),
            _ptr(k_norm_weight), _ptr(cos), _ptr(sin), cs_stride, _ptr(slot_mapping), _ptr(kv_pool),
            _ptr(kv_scales), t, hq, hkv, d, slots, float(rms_eps), _stream()))
        return q
    _lib.check(lib.litekv_qk_norm_rope_append(
        _ptr(q), _rows("q", q), _ptr(k), _rows("k", k), _ptr(v), _rows("v", v), _ptr(q_norm_weight),
        _ptr(k_norm_weight), _ptr(cos), _ptr(sin), cs_stride, _ptr(slot_mapping), _ptr(kv_pool), t, hq, hkv, d,
        slots, float(rms_eps), _stream()))
    return q


def page_gather(src_pool: torch.Tensor, dst_pool: torch.Tensor, src_ids: torch.Tensor,
                dst_ids: Optional[torch.Tensor] = None, page_size: int = PAGE_SIZE) -> None:
    """dst_pool[page dst_ids[i]] = src_pool[page src_ids[i]]; dst_ids None means page i. Pages are
    moved as bytes: fp16 pools or fp8 pools, both of the same kind."""
    _dev_pool("src_pool", src_pool), _dev_pool("dst_pool", dst_pool)
    _need(src_pool.element_size() == dst_pool.element_size(), "pools differ in element size")
    _, hs, ds, n_src, page_bytes = pool_geometry(src_pool, page_size)
    _, hd, dd, n_dst, page_bytes_d = pool_geometry(dst_pool, page_size)
    _need((hs, ds) == (hd, dd) and page_bytes == page_bytes_d, "pools differ in page geometry")
    src_ids = _dev_i32("src_ids", src_ids)
    if dst_ids is not None:
        dst_ids = _dev_i32("dst_ids", dst_ids)
        _need(dst_ids.numel() == src_ids.numel(), "src_ids and dst_ids differ in length")
    lib = _lib.load()
    _lib.check(lib.litekv_page_gather(_ptr(src_pool), _ptr(dst_pool), _ptr(src_ids), _ptr(dst_ids),
                                      src_ids.numel(), page_bytes, n_src, n_dst, _stream()))


def page_copy(kv_pool: torch.Tensor, src_ids: torch.Tensor, dst_ids: torch.Tensor,
              page_size: int = PAGE_SIZE) -> None:
    """kv_pool[page dst_ids[i]] = kv_pool[page src_ids[i]] (copy-on-write move inside one pool, fp16 or fp8)."""
    _dev_pool("kv_pool", kv_pool)
    _, _, _, n_pages, page_bytes = pool_geometry(kv_pool, page_size)
    src_ids = _dev_i32("src_ids", src_ids)
    dst_ids = _dev_i32("dst_ids", dst_ids)
    _need(dst_ids.numel() == src_ids.numel(), "src_ids and dst_ids differ in length")
    lib = _lib.load()
    _lib.check(lib.litekv_page_copy(_ptr(kv_pool), _ptr(src_ids), _ptr(dst_ids), src_ids.numel(),
                                    page_bytes, n_pages, _stream()))


def decode_split_plan(batch: int, num_kv_heads: int, max_blocks: int,
                      num_splits: Optional[int] = None) -> tuple[int, int]:
    """(max_splits, min_pages_per_split) for a decode launch.

    ``num_splits`` fixes the split count per sequence (every sequence with at
    least that many pages uses exactly that many). Otherwise pages per split
    are chosen so the launch has a few thousand wavefronts of at least 8 pages.
    """
    if num_splits is not None:
        return max(1, int(num_splits)), 1
    items = max(1, batch * num_kv_heads)
    target_waves = 4096
    pps = max(8, min(64, (items * max_blocks + target_waves - 1) // target_waves))
    return max(1, (max_blocks + pps - 1) // pps), pps


def decode_workspace(batch: int, num_q_heads: int, max_splits: int, device) -> Optional[torch.Tensor]:
    nbytes = _lib.load().litekv_paged_decode_workspace_bytes(batch, num_q_heads, HEAD_DIM, max_splits)
    if nbytes == 0:
        return None
    return torch.empty(nbytes // 4, dtype=torch.float32, device=device)


def balanced_chunks(num_kv_heads: int) -> int:
    """Chunks per kv head that give every CU of the current device one workgroup."""
    return int(_lib.load().litekv_paged_decode_balanced_chunks(int(num_kv_heads)))


def prefix_chunks(batch: int, num_q_heads: int, num_kv_heads: int, shared_pages: int,
                  page_size: int = PAGE_SIZE, head_dim: int = HEAD_DIM, fp16_pool: bool = True) -> int:
    """Chunks per kv head for a step behind ``shared_pages`` shared pages: the private pages get the
    compute units that the workgroups attending the shared pages (same launch) leave free."""
    return int(_lib.load().litekv_paged_decode_prefix_chunks(int(batch), int(num_q_heads), int(num_kv_heads),
                                                             int(head_dim), int(page_size), int(shared_pages),
                                                             1 if fp16_pool else 0))


SPLIT_COUNTS = (4, 8, 16)


def _whole_device_chunks(num_kv_heads: int, cus: int = 256) -> int:
    """``balanced_chunks`` of a device with so many compute units (no device is asked)."""
    per_group = min(num_kv_heads, 8)                       # kv heads of a workgroup, a wavefront each
    groups = (num_kv_heads + 7) // 8
    return (cus + groups - 1) // groups * (8 // per_group)


def decode_schedule_estimates(batch: int, num_kv_heads: int, max_pages: int, total_pages: int, token_bytes: int,
                              page_size: int = PAGE_SIZE, heads_per_kv_head: int = 8,
                              head_dim: int = HEAD_DIM, chunks: Optional[int] = None) -> dict:
    """Estimated microseconds per layer of every decode schedule a step could take, keyed as
    ``decode_schedule`` returns them. Fits to 3941 measured shapes on an MI355X: a grid of 1 to 2048 sequences of 32 to
    32768 tokens (equal, ragged, one long among short; ``tune_decode_schedule`` re-measures such tables) and 1890
    drawn ones (1 to 1500 sequences, those kinds and log-normal lengths, pages of 16 to 64, up to 900 000 tokens);
    64/8, 16/8 and 32/4 heads of 128 and 32/8 of 64 over fp16, 64/8 over fp8, 32/4 and 32/8 of 64 over int8; every
    schedule replayed from a graph.

    * 1, one wavefront per (sequence, kv head), one launch: 3.4 us + the largest (a 3.1-norm) of the
      longest sequence's dependent chain of 16-token steps at 0.44 us each -- 0.43 growing to 0.71 from 512 to 2048
      wavefronts, whose loads share the compute units' memory paths with the chain's, half as much again from there,
      four to a workgroup --, the placement of the launch's wavefronts at 1.9 ns each, and the bytes
      at 5.9 MB/us (codes 4.7, of rows of 64 4.1), up to 17 % more where the sequences are uneven.
    * 4 / 8 / 16 splits per sequence + the merge launch, for launches of at most 2048 wavefronts:
      5.3 us for the two launches, the chain of a split at 0.46 us a step up to 512 wavefronts, 0.47 growing to 0.60 from
      there, against the bytes at 5.8 MB/us (codes 5.2; a 2.8-norm), 0.8 ns per wavefront (codes: 1.3); where the bytes
      dominate, uneven sequences make uneven splits, which the balanced cut does not have: 14 to 44 % more with the
      bytes' share.
    * 0, balanced (fused step + merge): 7.2 us, 0.22 us per piece the merge folds for the longest
      sequence (up to 21; 0.46 us more for each past 16 in a step of many rows; 0.07 to 0.18 us where a step
      of few rows shares a long row out among several workgroups, by how many rows those are; a third of that
      with rows of 64), 3.6 ns + 0.35 ns per query head for every sequence, and the bytes at 7.5 MB/us
      against the chain inside one of ``chunks`` (a plan's own count; else what ``balanced_chunks`` gives 256
      compute units) at 1.2 us a step; with more than 8 query heads per kv head, 10 % more -- its page step
      carries twice the exponentials -- and the partial rows beyond 8 MB, written and read back,
      at 3 MB/us (117 shapes of 8 to 64 query heads per kv head, 1 to 8 kv heads: 2 to 3 % over the
      fastest schedule; 8 sequences of 4000 tokens, 32/1 heads, 2048 chunks: 31 us, 17 without).

    A step over a page of codes takes 0.9 to 1.2 times as long as over fp16 rows (half the bytes, the conversion),
    over rows of 64 elements 0.6 to 0.9 times."""
    steps = max(1, page_size // PAGE_SIZE)                 # the kernels step by 16 tokens
    chain = max_pages * steps
    total = total_pages * steps
    nbytes = float(total_pages) * page_size * token_bytes
    num_q_heads = num_kv_heads * heads_per_kv_head
    slices = (heads_per_kv_head + 15) // 16                # wavefronts per kv head
    norm = lambda p, *xs: sum(x ** p for x in xs) ** (1.0 / p)
    lone = batch * num_kv_heads * slices                   # wavefronts of a launch with one per sequence
    chunks = _whole_device_chunks(num_kv_heads) if chunks is None else chunks
    narrow = head_dim < HEAD_DIM
    codes = token_bytes < 4 * num_kv_heads * head_dim      # a pool of 8-bit codes
    uneven = min(1.0, chain * batch / max(1, total) - 1.0)
    pieces = min(chain / max(1.0, total / chunks), 20.6)
    # rows of more than 16 pieces are merged by several workgroups each while the step has few rows
    rows = batch * num_q_heads * head_dim / (256.0 * HEAD_DIM)
    per_piece = 0.0739 + 0.107 * rows if pieces > 16 and rows <= 1.0 else 0.219
    merge = per_piece * (0.367 if narrow else 1.0) * pieces + (0.462 * max(0.0, pieces - 16.0) if rows > 1.0 else 0.0)
    step = (0.62 if narrow else 1.0) * (0.983 if codes else 1.0)
    partials = (min(total, chunks) + batch) * num_q_heads * head_dim * 4.0
    estimates = {
        0: (7.21 + merge + (3.63e-3 + 3.52e-4 * num_q_heads) * batch
            + norm(2.0, nbytes / (6.86e6 if codes else 7.54e6), 1.22 * step * -(-total // chunks))) * (
                1.1 if heads_per_kv_head > 8 else 1.0)
           + (max(0.0, 2.0 * partials - 16.8e6) / 3.0e6 if heads_per_kv_head > 8 else 0.0),
    }
    if narrow and not codes:
        estimates[0] *= 0.986
    # the per-sequence kernels: two steps' pages in flight up to 512 wavefronts, one's beyond
    crowd = min(1.0, lone / 2048.0)
    page = 0.436 if lone <= 512 else 0.431 * (1.0 + 0.645 * crowd ** 1.65) * (0.911 if codes else 1.0)
    page *= (0.866 if narrow else 1.0) * (1.49 if lone >= 2048 else 1.0)
    chain_us = page * chain
    stream = nbytes / (5.92e6 if not codes else 4.06e6 if narrow else 4.66e6)
    estimates[1] = (3.42 * (0.707 if narrow else 1.0) + norm(3.1, chain_us, 1.9e-3 * lone, stream)) * (
        1.0 + 0.17 * uneven * stream / max(1e-9, chain_us + stream))
    for n in SPLIT_COUNTS:
        wavefronts = batch * n * num_kv_heads * slices
        if wavefronts > 2048:
            continue
        if wavefronts <= 512:
            page = 0.462 * (1.22 if codes else 1.0)
        else:
            page = 0.45 * (1.0 + 0.341 * (wavefronts / 2048.0) ** 1.44) * (0.926 if codes else 1.0)
        chain_us = page * (0.916 if narrow else 1.0) * ((chain + n - 1) // n)
        stream = nbytes / (5.2e6 if codes else 5.78e6)
        estimates[n] = (5.33 * (0.929 if narrow else 1.0) + norm(2.82, chain_us, stream)
                        + (1.33e-3 if codes else 8.3e-4) * wavefronts) * (
            1.0 + (0.136 + 0.299 * uneven) * stream / max(1e-9, chain_us + stream))
    return estimates


def decode_schedule(batch: int, num_kv_heads: int, max_pages: int, total_pages: int, token_bytes: int,
                    page_size: int = PAGE_SIZE, heads_per_kv_head: int = 8, current: Optional[int] = None,
                    hysteresis: float = 1.0, head_dim: int = HEAD_DIM, chunks: Optional[int] = None) -> int:
    """Which decode schedule a step should take, from what the host knows about it: 0 = balanced,
    1 = one wavefront per (sequence, kv head) in one launch, 4 / 8 / 16 = that many splits per
    sequence and the merge launch: the smallest of ``decode_schedule_estimates``. Choosing by this
    rule is 0.3 to 1.2 % slower on average than always choosing the fastest schedule over the shapes of
    a head layout and pool format, 3 to 32 % at worst. ``current``: the schedule
    in use; another must be estimated ``hysteresis`` times faster to replace it. ``head_dim`` tells rows
    of 64 fp16 elements from 128 codes, which ``token_bytes`` alone does not; ``chunks``: a plan's own
    count, see ``decode_schedule_estimates``."""
    if batch <= 0 or total_pages <= 0 or max_pages <= 0:
        return 0
    estimates = decode_schedule_estimates(batch, num_kv_heads, max_pages, total_pages, token_bytes, page_size,
                                          heads_per_kv_head, head_dim, chunks)
    if current in estimates:
        estimates[current] /= hysteresis
    return min(estimates, key=estimates.get)


def pool_head_dim(token_bytes: int, num_kv_heads: int, kv_dtype: Optional[torch.dtype] = None) -> int:
    """What ``decode_schedule`` takes for the width of a pool's heads: 64 where the K + V bytes of a token
    and the element type (None: fp16) say so, else 128, also for the widths the rule does not serve."""
    return 64 if token_bytes == 2 * num_kv_heads * 64 * (2 if kv_dtype is None else kv_dtype.itemsize) else HEAD_DIM


class DecodePlan:
    """Per-step decision how the batch's pages are attended, shared by every layer of the step.

    Balanced schedule (default): the cut of the batch's pages into equal chunks (one launch), the
    device plan buffer (chunk entries) and the partial-result workspace. Launches that share a
    plan share its workspace and must run one after the other (same stream).
    Per-sequence schedule (``per_sequence`` True, see ``choose_schedule``): no cut to build;
    ``decode_step`` then runs ``splits`` wavefronts per (sequence, kv head), the append fused in,
    and with more than one split the merge launch over ``split_workspace``.
    """

    def __init__(self, block_table: torch.Tensor, seq_lens: torch.Tensor, num_q_heads: int,
                 num_kv_heads: int, num_pages: int, chunks: Optional[int] = None,
                 page_size: int = PAGE_SIZE, shared_pages: int = 0,
                 host_seq_lens: Optional[Sequence[int]] = None, token_bytes: Optional[int] = None,
                 kv_dtype: Optional[torch.dtype] = None):
        """``shared_pages``: leading block-table entries that are the same physical pages in every
        row (a shared cached prefix); they are then attended once for the whole batch.
        ``host_seq_lens``: the lengths as the host knows them; with them the plan picks the
        per-sequence schedule (and its split count) where ``decode_schedule`` says so. ``token_bytes``:
        K + V bytes of one token in the pool (default: fp16). ``kv_dtype``: the pool's element type
        (default fp16); with a shared prefix it decides how the default chunk count is chosen, and
        with ``token_bytes`` it tells the width of the heads, which the schedule depends on."""
        lib = _lib.load()
        self.shared_pages = int(shared_pages)
        self.kv_dtype = kv_dtype
        self.per_sequence = False
        self.splits = 1
        self.split_workspace: Optional[torch.Tensor] = None
        self.token_bytes = int(token_bytes) if token_bytes is not None else 2 * int(num_kv_heads) * HEAD_DIM * 2
        self.head_dim = pool_head_dim(self.token_bytes, int(num_kv_heads), kv_dtype)
        _need(0 <= self.shared_pages <= block_table.shape[1], "shared_pages out of range")
        _need(block_table.dim() == 2, "block_table must be [B, max_blocks]")
        self.block_table = _dev_i32("block_table", block_table)
        self.seq_lens = _dev_i32("seq_lens", seq_lens)
        self.batch = int(self.block_table.shape[0])
        _need(self.seq_lens.numel() == self.batch, "seq_lens must be [B]")
        self.num_q_heads, self.num_kv_heads = int(num_q_heads), int(num_kv_heads)
        self.num_pages, self.page_size = int(num_pages), int(page_size)
        self.block_table, self.bt_stride = _table_rows(self.block_table)
        if chunks is not None:
            self.chunks = int(chunks)
        elif self.shared_pages > 0 and block_table.shape[0] > 0:
            self.chunks = prefix_chunks(block_table.shape[0], num_q_heads, num_kv_heads, self.shared_pages, page_size,
                                        fp16_pool=kv_dtype in (None, torch.float16))
        else:
            self.chunks = balanced_chunks(num_kv_heads)
        dev = self.block_table.device
        self.plan_bytes = int(lib.litekv_decode_plan_bytes_paged(self.batch, self.bt_stride, self.num_kv_heads,
                                                                 self.chunks, self.page_size))
        _need(self.plan_bytes > 0 or self.batch == 0, f"page_size {self.page_size} unsupported (16, 32, 64, 128 or 256)")
        self.buffer = torch.empty(max(4, self.plan_bytes // 4), dtype=torch.int32, device=dev)
        ws_fn = (lib.litekv_paged_decode_prefix_workspace_bytes if self.shared_pages > 0
                 else lib.litekv_paged_decode_balanced_workspace_bytes)
        ws_bytes = int(ws_fn(self.batch, self.num_q_heads, HEAD_DIM, self.chunks))
        self.workspace = torch.empty(max(4, ws_bytes // 4), dtype=torch.float32, device=dev)
        self.workspace_bytes = ws_bytes
        if host_seq_lens is not None:
            self.choose_schedule(host_seq_lens)
        self.refresh()

    def set_schedule(self, splits: int) -> None:
        """0: balanced; otherwise the per-sequence schedule with that many splits per sequence
        (the partial-result buffer of several splits is allocated here, not at the launch)."""
        self.per_sequence = splits > 0
        self.splits = max(1, int(splits))
        if self.splits > 1:
            need = int(_lib.load().litekv_paged_decode_workspace_bytes(self.batch, self.num_q_heads, HEAD_DIM,
                                                                       self.splits)) // 4
            if self.split_workspace is None or self.split_workspace.numel() < need:
                self.split_workspace = torch.empty(need, dtype=torch.float32, device=self.block_table.device)

    @property
    def schedule(self) -> int:
        """0 on the balanced schedule, else the splits per sequence."""
        return self.splits if self.per_sequence else 0

    def choose_schedule(self, host_seq_lens: Sequence[int], hysteresis: float = 1.0) -> bool:
        """Sets the schedule from the lengths as the host knows them (no device read): see
        ``decode_schedule``; the schedule in use keeps a ``hysteresis`` advantage. A plan with a
        shared prefix stays balanced. Returns ``per_sequence``."""
        if self.shared_pages > 0:
            self.set_schedule(0)
            return False
        pages = [(int(n) + self.page_size - 1) // self.page_size for n in host_seq_lens if n > 0]
        if not pages:
            self.set_schedule(0)
            return False
        # the rule is told what its defaults do not say
        differs = {} if self.head_dim == HEAD_DIM else {"head_dim": self.head_dim}
        if self.chunks != _whole_device_chunks(self.num_kv_heads):
            differs["chunks"] = self.chunks
        self.set_schedule(decode_schedule(self.batch, self.num_kv_heads, max(pages), sum(pages), self.token_bytes,
                                          self.page_size, self.num_q_heads // self.num_kv_heads,
                                          current=self.schedule, hysteresis=hysteresis, **differs))
        return self.per_sequence

    def refresh(self, block_table: Optional[torch.Tensor] = None, seq_lens: Optional[torch.Tensor] = None) -> None:
        """Recomputes the cuts after the tables or lengths changed (same shapes). Nothing to do
        while the plan is on the per-sequence schedule."""
        if block_table is not None:
            bt, stride = _table_rows(_dev_i32("block_table", block_table))
            _need(bt.shape == self.block_table.shape and stride == self.bt_stride, "block_table shape changed")
            self.block_table = bt
        if seq_lens is not None:
            sl = _dev_i32("seq_lens", seq_lens)
            _need(sl.numel() == self.batch, "seq_lens shape changed")
            self.seq_lens = sl
        if self.per_sequence:
            return
        lib = _lib.load()
        _lib.check(lib.litekv_decode_plan_prefix(_ptr(self.block_table), self.bt_stride, _ptr(self.seq_lens),
                                                 self.batch, self.num_kv_heads, self.page_size, self.num_pages,
                                                 self.chunks, self.shared_pages, _ptr(self.buffer),
                                                 self.plan_bytes, _stream()))


def _fixed(name: str, t: Optional[torch.Tensor], dtype: torch.dtype, numel: Optional[int] = None) -> None:
    """An output (or in/out) tensor must already have its final form: nothing is cast or copied."""
    if t is None:
        return
    _need(t.is_cuda and t.dtype == dtype and t.is_contiguous(), f"{name} must be a contiguous {dtype} GPU tensor")
    _need(numel is None or t.numel() == numel, f"{name} must hold {numel} elements")


def decode_advance(request_tables: torch.Tensor, request_ids: torch.Tensor, seq_lens: torch.Tensor,
                   slot_mapping: torch.Tensor, block_table: torch.Tensor, num_pages: int,
                   capacity: Optional[torch.Tensor] = None, seq_lens_i64: Optional[torch.Tensor] = None,
                   position_ids: Optional[torch.Tensor] = None, overflow: Optional[torch.Tensor] = None,
                   page_size: int = PAGE_SIZE, increment: int = 1) -> None:
    """One decode step of metadata on the device, in place: seq_lens += increment, slot_mapping[b] =
    slot of logical token seq_lens[b] - 1 in request request_ids[b]'s page list (a row of
    request_tables [max_requests, max_pages]), position_ids[b] = seq_lens[b] - 1, and block_table
    [B, width] = the batch's page lists. Rows that cannot advance (capacity reached, bad request id)
    raise the overflow flag and end empty for good (length -1, slot -1): every kernel of the path
    treats them as holding no tokens, so the step's append never lands on a cached token."""
    _need(request_tables.dim() == 2 and request_tables.stride(1) == 1, "request_tables must be [max_requests, max_pages]")
    _fixed("request_tables", request_tables, torch.int32)
    b = request_ids.numel()
    _fixed("request_ids", request_ids, torch.int32)
    _fixed("seq_lens", seq_lens, torch.int32, b)
    _fixed("slot_mapping", slot_mapping, torch.int32, b)
    _fixed("capacity", capacity, torch.int32, b)
    _fixed("seq_lens_i64", seq_lens_i64, torch.int64, b)
    _fixed("position_ids", position_ids, torch.int64, b)
    _fixed("overflow", overflow, torch.int32, 1)
    _need(block_table.is_cuda and block_table.dtype == torch.int32 and block_table.dim() == 2
          and block_table.shape[0] == b and block_table.stride(1) == 1, "block_table must be int32 [B, width] on the GPU")
    width = int(block_table.shape[1])
    _need(width <= request_tables.shape[1], "block_table is wider than request_tables")
    lib = _lib.load()
    _lib.check(lib.litekv_decode_advance(
        _ptr(request_tables), request_tables.stride(0), request_tables.shape[0], _ptr(request_ids), _ptr(capacity),
        _ptr(seq_lens), _ptr(seq_lens_i64), _ptr(slot_mapping), _ptr(position_ids), _ptr(block_table),
        block_table.stride(0) if b > 1 else max(block_table.stride(0), width), width, _ptr(overflow), b,
        int(page_size), int(num_pages), int(increment), _stream()))


def _segment(dst: torch.Tensor, src: torch.Tensor) -> Optional[tuple]:
    """(src, dst, rows, row bytes, src pitch, dst pitch) of a copy litekv_copy_segments can take, or None."""
    if not (src.is_cuda and src.dtype is dst.dtype and src.shape == dst.shape
            and src.get_device() == dst.get_device() == torch._C._cuda_getDevice()):   # a launch goes to the current device
        return None
    size = dst.element_size()
    if src.is_contiguous() and dst.is_contiguous():
        rows, row_bytes = 1, dst.numel() * size
        src_pitch = dst_pitch = row_bytes
    elif dst.dim() == 2 and dst.stride(1) == 1 and src.stride(1) == 1:
        rows, row_bytes = dst.shape[0], dst.shape[1] * size
        src_pitch, dst_pitch = src.stride(0) * size, dst.stride(0) * size
        if rows > 1 and (src_pitch < row_bytes or dst_pitch < row_bytes):    # a broadcast row
            return None
    else:
        return None
    entry = (src.data_ptr(), dst.data_ptr(), rows, row_bytes, src_pitch, dst_pitch)
    aligned = (entry[0] | entry[1] | row_bytes | src_pitch | dst_pitch) % 4 == 0
    return entry if aligned and rows * row_bytes <= 1 << 30 else None


# One type for every launch: ctypes drops an array type nobody holds and takes 30 us to make it again.
_SegmentArray = ctypes.c_int64 * (6 * 8)


def copy_tensors(pairs: Sequence[tuple]) -> None:
    """dst.copy_(src) for every (dst, src): small device tensors of equal type and shape go eight to a
    launch, whatever else there is one by one."""
    segments: list = []
    count = 0
    for dst, src in pairs:
        entry = _segment(dst, src) if dst.is_cuda else None
        if entry is None:
            dst.copy_(src)
            continue
        segments += entry
        count += 1
    for i in range(0, count, 8):
        part = segments[6 * i:6 * (i + 8)]
        _lib.check(_lib.load().litekv_copy_segments(_SegmentArray(*part), len(part) // 6, _stream()))


def decode_step(q: torch.Tensor, kv_pool: torch.Tensor, plan: DecodePlan,
                k_new: Optional[torch.Tensor] = None, v_new: Optional[torch.Tensor] = None,
                softmax_scale: Optional[float] = None, out: Optional[torch.Tensor] = None,
                kv_scales: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One layer of a decode step under ``plan``. Balanced schedule: optional append of k_new / v_new
    ([B, Hkv, D]) at logical position seq_lens[b] - 1 fused into the attention of q [B, Hq, D] over
    the planned pages, then the merge of the sequences that span several chunks. Per-sequence
    schedule (``plan.per_sequence``): the same by ``plan.splits`` wavefronts per (sequence, kv
    head); one launch and no merge with one split. An fp8 pool (uint8 / float8_e4m3fn) comes with
    its per-head ``kv_scales``."""
    if plan.per_sequence:
        return paged_decode(q, kv_pool, plan.block_table, plan.seq_lens, softmax_scale, num_splits=plan.splits,
                            out=out, workspace=plan.split_workspace if plan.splits > 1 else None,
                            page_size=plan.page_size, schedule="splits", kv_scales=kv_scales,
                            k_new=k_new, v_new=v_new)
    _dev_half("q", q)
    fp8 = is_quantised_pool(kv_pool)
    if not fp8:
        _dev_half("kv_pool", kv_pool)
    if not (q.dim() == 3 and q.stride(2) == 1 and q.stride(1) == q.shape[2]):
        raise ValueError("q must be [B, Hq, D] with contiguous heads")
    b, hq, d = q.shape
    _, hkv, dk, n_pages, _ = pool_geometry(kv_pool, plan.page_size)
    if not (d == dk):
        raise ValueError("q and kv_pool differ in head_dim")
    if not ((b, hq, hkv, n_pages) == (plan.batch, plan.num_q_heads, plan.num_kv_heads, plan.num_pages)):
        raise ValueError("plan was made for another batch / head / pool geometry")
    if not ((k_new is None) == (v_new is None)):
        raise ValueError("k_new and v_new go together")
    kn_stride = vn_stride = 0
    if k_new is not None:
        _dev_half("k_new", k_new), _dev_half("v_new", v_new)
        if not (k_new.shape == (b, hkv, d) and v_new.shape == (b, hkv, d)):
            raise ValueError("k_new / v_new must be [B, Hkv, D]")
        kn_stride, vn_stride = _rows("k_new", k_new), _rows("v_new", v_new)
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if out is None:
        out = torch.empty((b, hq, d), dtype=torch.float16, device=q.device)
    else:
        _dev_half("out", out)
        if not (out.shape == (b, hq, d) and out.is_contiguous()):
            raise ValueError("out must be contiguous [B, Hq, D]")
    q_stride = q.stride(0) if b > 1 else max(q.stride(0), hq * d)
    lib = _lib.load()
    if fp8:
        _dev_fp8_pool(kv_pool, kv_scales, hkv)
        if plan.shared_pages > 0:
            _lib.check(_q8_entry(lib, "paged_decode_prefix", kv_pool)(
                _ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales), _ptr(plan.block_table), _ptr(plan.seq_lens),
                _ptr(plan.buffer), plan.plan_bytes, _ptr(k_new), _ptr(v_new), kn_stride, vn_stride, _ptr(out),
                _ptr(plan.workspace), plan.workspace_bytes, b, hq, hkv, d, plan.page_size, n_pages, plan.bt_stride,
                plan.chunks, plan.shared_pages, float(softmax_scale), _stream()))
            return out
        _lib.check(_q8_entry(lib, "paged_decode_balanced", kv_pool)(
            _ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales), _ptr(plan.seq_lens), _ptr(plan.buffer),
            plan.plan_bytes, _ptr(k_new), _ptr(v_new), kn_stride, vn_stride, _ptr(out), _ptr(plan.workspace),
            plan.workspace_bytes, b, hq, hkv, d, plan.page_size, n_pages, plan.bt_stride, plan.chunks,
            float(softmax_scale), _stream()))
        return out
    if plan.shared_pages > 0:
        _lib.check(lib.litekv_paged_decode_prefix(
            _ptr(q), q_stride, _ptr(kv_pool), _ptr(plan.block_table), _ptr(plan.seq_lens), _ptr(plan.buffer),
            plan.plan_bytes, _ptr(k_new), _ptr(v_new), kn_stride, vn_stride, _ptr(out), _ptr(plan.workspace),
            plan.workspace_bytes, b, hq, hkv, d, plan.page_size, n_pages, plan.bt_stride, plan.chunks,
            plan.shared_pages, float(softmax_scale), _stream()))
        return out
    _lib.check(lib.litekv_paged_decode_balanced(
        _ptr(q), q_stride, _ptr(kv_pool), _ptr(plan.seq_lens), _ptr(plan.buffer), plan.plan_bytes,
        _ptr(k_new), _ptr(v_new), kn_stride, vn_stride, _ptr(out), _ptr(plan.workspace), plan.workspace_bytes,
        b, hq, hkv, d, plan.page_size, n_pages, plan.bt_stride, plan.chunks, float(softmax_scale), _stream()))
    return out


_STAGES = ("both", "split", "merge")


def paged_decode(q: torch.Tensor, kv_pool: torch.Tensor, block_table: torch.Tensor,
                 seq_lens: torch.Tensor, softmax_scale: Optional[float] = None,
                 num_splits: Optional[int] = None, min_pages_per_split: Optional[int] = None,
                 max_splits: Optional[int] = None, out: Optional[torch.Tensor] = None,
                 workspace: Optional[torch.Tensor] = None, page_size: int = PAGE_SIZE,
                 stage: str = "both", schedule: Optional[str] = None,
                 chunks: Optional[int] = None, plan: Optional[DecodePlan] = None,
                 shared_pages: int = 0, kv_scales: Optional[torch.Tensor] = None,
                 k_new: Optional[torch.Tensor] = None, v_new: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Decode attention of q [B, Hq, D] over the pages named by block_table [B, max_blocks].

    ``shared_pages`` (balanced schedule): the first that many entries of every block-table row are
    the same physical pages; they are attended once for the whole batch.

    schedule "balanced" (default): all pages of the batch are cut into `chunks` equal pieces per
    kv head (default: one workgroup per CU); a DecodePlan is built for the call unless one is
    passed. schedule "splits" (chosen when num_splits, max_splits or min_pages_per_split is
    given): every sequence is cut into its own splits; two launches (`stage` selects one).
    An fp8 pool comes with its ``kv_scales``; either schedule reads it.
    ``k_new`` / ``v_new`` [B, Hkv, D] (splits schedule, both stages): the step's new token of every
    sequence is written at logical position seq_lens[b] - 1 by the same launch and attended.
    """
    _dev_half("q", q)
    if not is_quantised_pool(kv_pool):
        _dev_half("kv_pool", kv_pool)
    if not (q.dim() == 3 and q.stride(2) == 1 and q.stride(1) == q.shape[2]):
        raise ValueError("q must be [B, Hq, D] with contiguous heads")
    b, hq, d = q.shape
    _, hkv, dk, n_pages, _ = pool_geometry(kv_pool, page_size)
    if not (d == dk):
        raise ValueError("q and kv_pool differ in head_dim")
    if not (stage in _STAGES):
        raise ValueError(f"unknown stage {stage!r}")
    if schedule is None:
        split_args = (num_splits, max_splits, min_pages_per_split)
        schedule = "splits" if any(x is not None for x in split_args) or stage != "both" else "balanced"
    if not (schedule in ("balanced", "splits")):
        raise ValueError(f"unknown schedule {schedule!r}")

    if not ((k_new is None) == (v_new is None)):
        raise ValueError("k_new and v_new go together")
    if schedule == "balanced":
        if not (stage == "both"):
            raise ValueError("the balanced schedule is a single launch")
        if not (k_new is None):
            raise ValueError("the balanced schedule appends through decode_step")
        if plan is None:
            plan = DecodePlan(block_table, seq_lens, hq, hkv, n_pages, chunks, page_size, shared_pages,
                              kv_dtype=kv_pool.dtype)
        return decode_step(q, kv_pool, plan, None, None, softmax_scale, out, kv_scales)

    fp8 = is_quantised_pool(kv_pool)
    if fp8:
        _dev_fp8_pool(kv_pool, kv_scales, hkv)
        if not (stage == "both"):
            raise ValueError("an fp8 pool is read by both stages in one call")
    if not (block_table.dim() == 2 and block_table.shape[0] == b):
        raise ValueError("block_table must be [B, max_blocks]")
    block_table, bt_stride = _table_rows(_dev_i32("block_table", block_table))
    seq_lens = _dev_i32("seq_lens", seq_lens)
    if not (seq_lens.numel() == b):
        raise ValueError("seq_lens must be [B]")
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if out is None:
        out = torch.empty((b, hq, d), dtype=torch.float16, device=q.device)
    else:
        _dev_half("out", out)
        if not (out.shape == (b, hq, d) and out.is_contiguous()):
            raise ValueError("out must be contiguous [B, Hq, D]")
    lib = _lib.load()
    q_stride = q.stride(0) if b > 1 else max(q.stride(0), hq * d)
    if max_splits is None or min_pages_per_split is None:
        s, pps = decode_split_plan(b, hkv, block_table.shape[1], num_splits)
        max_splits = s if max_splits is None else max_splits
        min_pages_per_split = pps if min_pages_per_split is None else min_pages_per_split
    if workspace is None:
        workspace = decode_workspace(b, hq, max_splits, q.device)
    ws_bytes = 0 if workspace is None else workspace.numel() * workspace.element_size()
    if k_new is not None:
        if not (stage == "both"):
            raise ValueError("the fused append belongs to the call that runs both stages")
        _dev_half("k_new", k_new), _dev_half("v_new", v_new)
        if not (k_new.shape == (b, hkv, d) and v_new.shape == (b, hkv, d)):
            raise ValueError("k_new / v_new must be [B, Hkv, D]")
        rows = (_ptr(k_new), _ptr(v_new), _rows("k_new", k_new), _rows("v_new", v_new))
        tail = (_ptr(out), _ptr(workspace), ws_bytes, b, hq, hkv, d, page_size, n_pages, max_splits,
                min_pages_per_split, float(softmax_scale), _stream())
        if fp8:
            _lib.check(_q8_entry(lib, "paged_decode_append", kv_pool)(_ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales),
                                                          _ptr(block_table), bt_stride, _ptr(seq_lens),
                                                          *rows, *tail))
        else:
            _lib.check(lib.litekv_paged_decode_append(_ptr(q), q_stride, _ptr(kv_pool), _ptr(block_table),
                                                      bt_stride, _ptr(seq_lens), *rows, *tail))
    elif fp8:
        _lib.check(_q8_entry(lib, "paged_decode", kv_pool)(_ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales), _ptr(block_table),
                                               bt_stride, _ptr(seq_lens), _ptr(out), _ptr(workspace),
                                               ws_bytes, b, hq, hkv, d, page_size, n_pages, max_splits,
                                               min_pages_per_split, float(softmax_scale), _stream()))
    elif stage in ("both", "split"):
        fn = lib.litekv_paged_decode if stage == "both" else lib.litekv_paged_decode_split
        _lib.check(fn(_ptr(q), q_stride, _ptr(kv_pool), _ptr(block_table), bt_stride,
                      _ptr(seq_lens), _ptr(out), _ptr(workspace), ws_bytes, b, hq, hkv, d, page_size,
                      n_pages, max_splits, min_pages_per_split, float(softmax_scale), _stream()))
    else:
        _lib.check(lib.litekv_paged_decode_merge(_ptr(seq_lens), _ptr(out), _ptr(workspace), ws_bytes, b,
                                                 hq, d, page_size, max_splits, min_pages_per_split,
                                                 _stream()))
    return out


def paged_decode_static(q: torch.Tensor, kv_pool: torch.Tensor, block_table: torch.Tensor,
                        seq_lens: torch.Tensor, out: torch.Tensor, max_splits: int,
                        min_pages_per_split: int, softmax_scale: Optional[float] = None,
                        page_size: int = PAGE_SIZE) -> torch.Tensor:
    """``paged_decode`` on the splits schedule without any allocation: ``out`` comes from the
    caller, index tensors must already be int32 on the device, and the partial results live in
    the scratch array built into the library (at most STATIC_SCRATCH_BYTES of them, else
    LiteKVError). Calls that overlap in time on one GPU share that array and race."""
    _dev_half("q", q), _dev_half("kv_pool", kv_pool), _dev_half("out", out)
    _need(q.dim() == 3 and q.stride(2) == 1 and q.stride(1) == q.shape[2], "q must be [B, Hq, D] with contiguous heads")
    b, hq, d = q.shape
    _, hkv, dk, n_pages, _ = pool_geometry(kv_pool, page_size)
    _need(d == dk, "q and kv_pool differ in head_dim")
    _need(out.shape == (b, hq, d) and out.is_contiguous(), "out must be contiguous [B, Hq, D]")
    for name, t in (("block_table", block_table), ("seq_lens", seq_lens)):
        _need(t.is_cuda and t.dtype == torch.int32, f"{name} must be an int32 device tensor")
    _need(block_table.dim() == 2 and block_table.shape[0] == b and block_table.stride(1) == 1,
          "block_table must be [B, max_blocks]")
    block_table, bt_stride = _table_rows(block_table)
    _need(seq_lens.numel() == b and seq_lens.is_contiguous(), "seq_lens must be contiguous [B]")
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    q_stride = q.stride(0) if b > 1 else max(q.stride(0), hq * d)
    _lib.check(_lib.load().litekv_paged_decode_static(
        _ptr(q), q_stride, _ptr(kv_pool), _ptr(block_table), bt_stride, _ptr(seq_lens),
        _ptr(out), b, hq, hkv, d, page_size, n_pages, int(max_splits), int(min_pages_per_split),
        float(softmax_scale), _stream()))
    return out


def paged_prefill(q: torch.Tensor, kv_pool: torch.Tensor, block_table: torch.Tensor,
                  cu_q_lens: torch.Tensor, context_lens: Optional[torch.Tensor], max_q_len: int,
                  softmax_scale: Optional[float] = None, out: Optional[torch.Tensor] = None,
                  page_size: int = PAGE_SIZE, kv_scales: Optional[torch.Tensor] = None,
                  key_slices: Optional[int] = None, max_kv_len: Optional[int] = None,
                  workspace: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal varlen attention of packed q [T, Hq, D] over paged KV (history + the chunk itself).
    An fp8 pool (uint8 / float8_e4m3fn) comes with its per-head ``kv_scales``.

    A launch with too few query rows to fill the device (one request's chunk over a long history)
    is cut along the keys as well: ``key_slices`` workgroups per row block and a merge launch
    (head_dim 64 / 128, any pool format). None lets the library choose from the launch shape and
    ``max_kv_len`` (the most keys a row sees: history + chunk, as the host knows it; without it
    the launch is not cut, and its form is the one for few keys); 1 switches it off. ``workspace`` (float32, see ``paged_prefill_workspace_floats``) is
    allocated when not given."""
    if q.is_cuda and out is None and key_slices is None and workspace is None and softmax_scale is not None:
        done = _lib.calls().paged_prefill(q, kv_pool, block_table, cu_q_lens, context_lens, max_q_len, softmax_scale,
                                          page_size, kv_scales, max_kv_len, _stream())
        if done is not None:
            if type(done) is int:
                _lib.check(done)
            return done
    # (not a plain call)
    _dev_half("q", q)
    fp8 = is_quantised_pool(kv_pool)
    if not fp8:
        _dev_half("kv_pool", kv_pool)
        if not (kv_scales is None):
            raise ValueError("kv_scales belong to an fp8 pool")
    q_stride = _rows("q", q)
    t, hq, d = q.shape
    _, hkv, dk, n_pages, _ = pool_geometry(kv_pool, page_size)
    if fp8:
        _dev_fp8_pool(kv_pool, kv_scales, hkv)
    if not (d == dk):
        raise ValueError("q and kv_pool differ in head_dim")
    cu_q_lens = _dev_i32("cu_q_lens", cu_q_lens)
    b = cu_q_lens.numel() - 1
    if not (block_table.dim() == 2 and block_table.shape[0] == b):
        raise ValueError("block_table must be [B, max_blocks]")
    block_table = _dev_i32("block_table", block_table)
    if context_lens is not None:
        context_lens = _dev_i32("context_lens", context_lens)
        if not (context_lens.numel() == b):
            raise ValueError("context_lens must be [B]")
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if out is None:
        out = torch.empty((t, hq, d), dtype=torch.float16, device=q.device)
    lib = _lib.load()
    if key_slices is None:
        # a workgroup takes 128 (row, head) columns: beyond 512 of them the device is full as it is;
        # and without the lengths on the host there is nothing to choose by (what the block table
        # could name says little: a fresh prompt cut into eight slices takes twice as long)
        few_rows = 0 < t * hq <= 128 * 512 and max_kv_len is not None
        key_slices = int(lib.litekv_paged_prefill_key_slices(b, hq, hkv, d, int(max_q_len), int(max_kv_len))) if few_rows else 1
    key_slices = int(key_slices)
    if key_slices > 1:
        need = paged_prefill_workspace_floats(t, hq, d, key_slices)
        if workspace is None:
            workspace = torch.empty(need, dtype=torch.float32, device=q.device)
        if not (workspace.is_cuda and workspace.dtype == torch.float32
                and workspace.is_contiguous() and workspace.numel() >= need):
            raise ValueError(f"workspace must be {need} contiguous float32 on the device")
    if key_slices <= 1:
        # (max_kv_len 0: not known)
        _lib.check(lib.litekv_paged_prefill_bounded(
            _ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales), 1 if is_int8_pool(kv_pool) else 0, _ptr(block_table),
            block_table.stride(0), _ptr(cu_q_lens), _ptr(context_lens), _ptr(out), _rows("out", out), b, hq, hkv, d,
            page_size, n_pages, int(max_q_len), 0 if max_kv_len is None else int(max_kv_len), float(softmax_scale),
            _stream()))
        return out
    if fp8:
        _lib.check(lib.litekv_paged_prefill_split_q8(
            _ptr(q), q_stride, _ptr(kv_pool), _ptr(kv_scales), 1 if is_int8_pool(kv_pool) else 0,
            _ptr(block_table), block_table.stride(0), _ptr(cu_q_lens), _ptr(context_lens), _ptr(out),
            _rows("out", out), b, hq, hkv, d, page_size, n_pages, int(max_q_len), t, key_slices,
            _ptr(workspace), workspace.numel() * 4, float(softmax_scale), _stream()))
        return out
    _lib.check(lib.litekv_paged_prefill_split(_ptr(q), q_stride, _ptr(kv_pool), _ptr(block_table),
                                              block_table.stride(0), _ptr(cu_q_lens), _ptr(context_lens),
                                              _ptr(out), _rows("out", out), b, hq, hkv, d, page_size, n_pages,
                                              int(max_q_len), t, key_slices, _ptr(workspace),
                                              workspace.numel() * 4, float(softmax_scale), _stream()))
    return out


def paged_prefill_workspace_floats(num_tokens: int, num_q_heads: int, head_dim: int, key_slices: int) -> int:
    """float32 elements of the workspace a paged prefill over ``key_slices`` key slices needs."""
    nbytes = int(_lib.load().litekv_paged_prefill_split_workspace_bytes(int(num_tokens), int(num_q_heads),
                                                                        int(head_dim), int(key_slices)))
    return nbytes // 4


def varlen_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, seq_starts: torch.Tensor,
                   seq_lens: torch.Tensor, max_seq_len: int, softmax_scale: Optional[float] = None,
                   out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal varlen attention of packed q over packed contiguous k, v ([T, Hkv, D])."""
    _dev_half("q", q), _dev_half("k", k), _dev_half("v", v)
    q_stride, k_stride, v_stride = _rows("q", q), _rows("k", k), _rows("v", v)
    t, hq, d = q.shape
    if not (k.shape == v.shape and k.shape[0] == t and k.shape[2] == d):
        raise ValueError("k/v shape mismatch")
    hkv = k.shape[1]
    seq_starts = _dev_i32("seq_starts", seq_starts)
    seq_lens = _dev_i32("seq_lens", seq_lens)
    b = seq_lens.numel()
    if not (seq_starts.numel() == b):
        raise ValueError("seq_starts and seq_lens differ in length")
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if out is None:
        out = torch.empty((t, hq, d), dtype=torch.float16, device=q.device)
    lib = _lib.load()
    _lib.check(lib.litekv_varlen_prefill(_ptr(q), q_stride, _ptr(k), k_stride, _ptr(v), v_stride,
                                         _ptr(seq_starts), _ptr(seq_lens), _ptr(out), _rows("out", out),
                                         b, hq, hkv, d, int(max_seq_len), t, float(softmax_scale),
                                         _stream()))
    return out
