"""What this framework is asked to do, as measurable cases over its real range of sizes.

Every case is one model step's share of the attention path, called the way a model calls it: an
``AttentionInfo`` with the batch's block table, lengths and pools, and one ``Attention`` per layer.

* ``decode``: a decode step of ``layers`` layers (one new token per sequence: append + attention over
  the paged cache) through ``DecodeGraphRunner``, which a serving loop keeps for its model. The pools
  of the layers are separate, as a model's are; small pools stay small.
* ``prefill``: fresh prompts, packed without padding: QK norm + rotary embedding + append, then
  causal attention over the pages just written, layer by layer without a graph (lengths change
  from call to call).
* ``chunk``: the next chunk of a chunked prefill: the same two calls, with keys from the request's
  cached history as well.

Pages are placed by a random permutation of the pool, which is what a pool looks like after it has
served for a while. Lengths come from the case (``lengths`` seeds them), everything else from the seed.
"""

import math

import torch

from llama_lite_npu_amd import ops, workloads
from llama_lite_npu_amd.attention import Attention
from llama_lite_npu_amd.executor.decode_graph import DecodeGraphRunner
from llama_lite_npu_amd.executor.executor_struct import AttentionInfo

DEVICE = "cuda:0"
LOG2E = 1.4426950408889634

# query heads, kv heads, head dim
HEADS = {
    "qwen3-0.6b": (16, 8, 128),
    "qwen3-32b": (64, 8, 128),
    "qwen3-30b-a3b": (32, 4, 128),
    "llama-3.2-1b": (32, 8, 64),
    "wide": (16, 4, 256),        # 256-wide heads, no model in particular
}


def _decode(name, heads, batch, lo, hi, layers, kv="f16", page=16, prefix=0, lengths=1):
    """``batch`` sequences that hold ``prefix`` shared tokens and lo..hi of their own before the step."""
    return {"name": name, "kind": "decode", "heads": heads, "batch": batch, "lo": lo, "hi": hi, "prefix": prefix,
            "layers": layers, "kv": kv, "page": page, "lengths": lengths}


def _prefill(name, heads, batch, lo, hi, layers, kv="f16", page=16, history=0, lengths=1):
    """``batch`` prompts (chunks) of lo..hi tokens; ``history``: the longest cached history of a chunk."""
    return {"name": name, "kind": "chunk" if history else "prefill", "heads": heads, "batch": batch, "lo": lo, "hi": hi,
            "history": history, "layers": layers, "kv": kv, "page": page, "lengths": lengths}


def listed():
    return [
        # one user chatting with a small model: all of its layers, nothing but latency
        _decode("decode-1", "qwen3-0.6b", 1, 778, 778, 28),
        # a handful of users on a small model with narrow heads, larger pages
        _decode("decode-12-hd64", "llama-3.2-1b", 12, 100, 3000, 16, page=64, lengths=7),
        # the benchmark's serving batch: 32 sequences of 256 to 4096 tokens, 302 MB of K/V per layer
        _decode("decode-32", "qwen3-32b", 32, 256, 4096, 8, lengths=1002),
        # the same batch over an fp8 pool
        _decode("decode-32-fp8", "qwen3-32b", 32, 256, 4096, 8, kv="fp8", lengths=1002),
        # 64 requests behind one cached system prompt of 2048 tokens
        _decode("decode-64-prefix", "qwen3-32b", 64, 64, 512, 8, prefix=2048, lengths=1004),
        # long contexts, many of them, over an int8 pool: 2.6 GB of K/V in one layer
        _decode("decode-128-long-int8", "qwen3-30b-a3b", 128, 8192, 32768, 1, kv="int8", lengths=1005),
        # one short prompt through all layers of a small model: time to first token, mostly launches
        _prefill("prefill-1", "qwen3-0.6b", 1, 203, 203, 28),
        # the benchmark's prefill batch: 8 prompts of 128 to 2048 tokens
        _prefill("prefill-8", "qwen3-32b", 8, 128, 2048, 2, lengths=1003),
        # documents: a few prompts of several thousand tokens
        _prefill("prefill-4-long", "qwen3-32b", 4, 5000, 8192, 1, lengths=11),
        # a batch of ordinary prompts on narrow heads
        _prefill("prefill-16-hd64", "llama-3.2-1b", 16, 100, 2048, 2, page=64, lengths=13),
        # ... and on 256-wide heads
        _prefill("prefill-4-hd256", "wide", 4, 300, 2048, 1, page=32, lengths=17),
        # chunked prefill of a long document: 512 more tokens behind up to 12 000 cached ones
        _prefill("chunk-1-history", "qwen3-32b", 1, 512, 512, 4, history=12000, lengths=19),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above. At most 2.6 GB of K/V and 28 layers in a decode step, at most
    0.6 TFLOP in a prefill (0.015 on 256-wide heads)."""
    kind = rng.choice(["decode", "decode", "decode-prefix", "prefill", "prefill", "chunk"])
    page = rng.choice([16, 16, 32, 64])
    kv = rng.choice(["f16", "f16", "fp8", "int8"])
    seed = rng.randrange(1, 1 << 30)
    if kind.startswith("decode"):
        heads = rng.choice(["qwen3-0.6b", "qwen3-32b", "qwen3-30b-a3b", "llama-3.2-1b"])
        _, hkv, d = HEADS[heads]
        prefix = 0
        if kind == "decode-prefix":
            batch = _log_int(rng, 8, 96)
            prefix = 64 * _log_int(rng, 4, 48)       # full pages of every page size
            hi = _log_int(rng, 64, 1024)
        else:
            batch = _log_int(rng, 1, 128)
            hi = _log_int(rng, 64, 32768)
        lo = rng.randint(max(1, hi // 8), hi)
        size = 2 * hkv * d * (2 if kv == "f16" else 1) * ((lo + hi) // 2 * batch + prefix)
        while size > 2_500_000_000:
            batch = max(1, batch // 2)
            size //= 2
        layers = max(1, min(rng.choice([4, 8, 16, 28]), 2_500_000_000 // size))
        c = _decode("", heads, batch, lo, hi, layers, kv, page, prefix, seed)
    else:
        heads = rng.choice(["qwen3-0.6b", "qwen3-32b", "qwen3-30b-a3b", "llama-3.2-1b", "wide"])
        hq, _, d = HEADS[heads]
        history = _log_int(rng, 500, 12000) if kind == "chunk" else 0
        hi = _log_int(rng, 48, 512) if history else _log_int(rng, 64, 8192)
        lo = rng.randint(max(1, hi // 8), hi)
        batch = _log_int(rng, 1, 4 if history else 24)
        # the wide heads' listed case is 4 prompts of up to 2048 tokens
        most = 0.6e12 if d < 256 else 0.015e12
        if d == 256:
            history = min(history, 2048)
            hi, lo = min(hi, 2048), min(lo, 2048)
        flops = 2 * hq * d * hi * (hi + 2 * history)
        while batch > 1 and flops * batch > most:
            batch -= 1
        if flops * batch > most:
            hi = lo = max(1, int(hi * math.sqrt(most / (flops * batch)) * 0.9))
            flops = 2 * hq * d * hi * (hi + 2 * history)
        layers = max(1, min(rng.choice([1, 2, 8, 28]), int(most / (flops * batch))))
        c = _prefill("", heads, batch, lo, hi, layers, kv if history else "f16", page, history, seed)
    del c["name"]
    return c


def _lens(case):
    """(tokens of the step, tokens cached before it) per sequence."""
    own = workloads.uniform_lens(case["lengths"], case["batch"], case["lo"], case["hi"])
    if case["kind"] == "decode":
        return [1] * len(own), [case["prefix"] + n for n in own]
    if case["kind"] == "chunk":
        h = case["history"]
        return own, workloads.uniform_lens(case["lengths"] + 1, case["batch"], (h + 1) // 2, h)
    return own, [0] * len(own)


def _pools(case, slots, gen):
    """[layers, slots, 2 * Hkv, D] of cached rows ~ N(0, 1) in the pool's format, and the scales."""
    _, hkv, d = HEADS[case["heads"]]
    shape = (slots, 2 * hkv, d)
    kv = case["kv"]
    pools = torch.empty((case["layers"],) + shape, device=DEVICE,
                        dtype={"f16": torch.float16, "fp8": torch.uint8, "int8": torch.int8}[kv])
    for layer in pools:
        rows = torch.randn(shape, generator=gen, dtype=torch.float16, device=DEVICE)
        if kv == "f16":
            layer.copy_(rows)
        elif kv == "fp8":
            layer.copy_(rows.to(torch.float8_e4m3fn).view(torch.uint8))
        else:
            layer.copy_(rows.mul_(127.0 / 5.0).round_().clamp_(-127, 127))
    if kv == "f16":
        return pools, [None] * case["layers"]
    scales = torch.full((2 * hkv,), 1.0 if kv == "fp8" else 5.0 / 127.0, dtype=torch.float32, device=DEVICE)
    return pools, [scales] * case["layers"]


class _Layers:
    """The attention layers of a model; q, k, v are what its projections would have left."""

    def __init__(self, case, q, k, v):
        self.attn = Attention(*HEADS[case["heads"]])
        self.q, self.k, self.v = list(q), list(k), list(v)

    def forward(self, input_ids, position_ids, atten_info):
        return [self.attn.token_forward(q, k, v, atten_info, i)
                for i, (q, k, v) in enumerate(zip(self.q, self.k, self.v))]


def prepare(case, seed):
    hq, hkv, d = HEADS[case["heads"]]
    page, layers = case["page"], case["layers"]
    new, cached = _lens(case)
    total = [a + b for a, b in zip(new, cached)]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    # block tables: private pages from a permutation, behind the shared prefix if there is one
    shared = case.get("prefix", 0) // page
    need = [-(-n // page) - shared for n in total]
    num_pages = math.ceil(1.1 * (sum(need) + shared)) + 1
    lists = workloads.assign_pages([shared] + need, num_pages, seed)
    table = workloads.table_from_lists([torch.cat([lists[0], own]) for own in lists[1:]])
    pools, scales = _pools(case, num_pages * page, gen)

    def rows(heads):
        return torch.randn((layers, sum(new), heads, d), generator=gen, dtype=torch.float16, device=DEVICE)

    q, k, v = rows(hq), rows(hkv), rows(hkv)
    slots = torch.cat([pages[torch.arange(c, n) // page] * page + torch.arange(c, n) % page
                       for pages, c, n in zip(table.long(), cached, total)])
    cu = torch.zeros(len(new) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(new), 0)

    info = AttentionInfo()
    info.kv_buffer, info.kv_scales = list(pools), scales
    info.page_size = page
    info.block_table = table.to(DEVICE)
    info.cur_select_index = slots.to(torch.int32).to(DEVICE)
    info.seq_lens_i32 = torch.tensor(total, dtype=torch.int32, device=DEVICE)
    info.b_seq_len = info.seq_lens_i32.long()
    info.b_req_idx = torch.arange(len(new), dtype=torch.int32, device=DEVICE)
    info.cu_q_lens = cu.to(DEVICE)
    info.b_start_loc = info.cu_q_lens[:-1]
    info.max_actual_seq_len = max(total)

    if case["kind"] == "decode":
        info.decode_plan = ops.DecodePlan(info.block_table, info.seq_lens_i32, hq, hkv, num_pages, page_size=page,
                                          shared_pages=shared, host_seq_lens=total,
                                          token_bytes=2 * hkv * d * pools.element_size(), kv_dtype=pools.dtype)
        runner = DecodeGraphRunner(_Layers(case, q, k, v), max_blocks=table.shape[1])
        ids = torch.zeros((len(new), 1), dtype=torch.long, device=DEVICE)
        position = (info.b_seq_len - 1).view(-1, 1)
        if not runner.capture(ids, position, info):
            raise RuntimeError("the decode step was not captured")
        return {"kind": "decode", "runner": runner, "ids": ids, "position": position, "info": info, "pools": pools}

    if case["kind"] == "chunk":
        info.is_paged_chunk_prefill = True
        info.context_lens_i32 = torch.tensor(cached, dtype=torch.int32, device=DEVICE)
        info.max_actual_q_seq_len = max(new)
    at = torch.cat([torch.arange(c, n) for c, n in zip(cached, total)]).to(DEVICE)
    angle = at[:, None] * (1e6 ** (-torch.arange(0, d, 2, device=DEVICE) / d))[None, :]
    angle = torch.cat([angle, angle], 1)
    weight = [1 + 0.1 * torch.randn(d, generator=gen, dtype=torch.float16, device=DEVICE) for _ in range(2)]
    return {"kind": case["kind"], "layers": _Layers(case, q, k, v), "q": q, "norm": weight,
            "rope": (angle.cos().half(), angle.sin().half()), "info": info, "pools": pools,
            "scale": LOG2E / math.sqrt(d)}


def run(state):
    info = state["info"]
    if state["kind"] == "decode":
        return {"out": state["runner"](state["ids"], state["position"], info), "pools": state["pools"]}
    model, (q_norm, k_norm) = state["layers"], state["norm"]
    out = []
    for i, (q, k, v) in enumerate(zip(model.q, model.k, model.v)):
        xq = model.attn.qkv_epilogue(q, k, v, info, i, q_norm, k_norm, state["rope"])
        out.append(model.attn.context_forward(xq, None, None, info, i, state["scale"]))
    return {"out": out, "q": state["q"], "pools": state["pools"]}


def work(case):
    """K/V of every token attended read once (a shared prefix once for the batch), q and the new rows
    read, their slots and the output written; a prefill also writes the rotated q. QK^T and PV over the
    visible keys."""
    hq, hkv, d = HEADS[case["heads"]]
    new, cached = _lens(case)
    item = 2 if case["kv"] == "f16" else 1
    fresh = sum(new)
    prefix = case.get("prefix", 0)
    read = sum(cached) - prefix * (case["batch"] - 1 if prefix else 0)
    tensors = 2 if case["kind"] == "decode" else 3                 # q, out (and q again)
    size = (read + fresh) * 2 * hkv * d * item + fresh * (2 * hkv * d * 2 + tensors * hq * d * 2)
    if case["kind"] != "decode":
        size += fresh * d * 2 * 2                                  # cos, sin
    flops = sum(2 * hq * d * n * (n + 1 + 2 * c) for n, c in zip(new, cached))
    return {"bytes": case["layers"] * size, "flops": case["layers"] * flops}


def tolerance(case):
    """fp16 results of fp32 sums over probabilities rounded to fp16. Against the same path in float64 the
    listed cases show rel 2.0e-4 to 2.9e-4 and max 5e-4 to 5.1e-3 (rows of long prompts that see few
    keys are many times the rms); four times that."""
    return {"rel": 1.2e-3, "max": 2e-2}
