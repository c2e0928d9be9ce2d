"""The native form of the per-layer prefill calls (csrc/torch_calls.cpp): it answers None to whatever
is not a plain call, and the wrappers then behave as they do without it -- the same results bit for
bit, the same errors."""

import sys
import types

import pytest
import torch

import llama_lite_npu_amd
from llama_lite_npu_amd import _lib, build, ops

DEV = "cuda:0"


def test_anything_but_a_plain_call_is_left_alone():
    calls = _lib.calls()
    x = torch.zeros((2, 4, 128), dtype=torch.float16)
    pool = torch.zeros((32, 4, 128), dtype=torch.float16)
    idx = torch.zeros(2, dtype=torch.int32)
    assert calls.qk_norm_rope_append() is None and calls.paged_prefill(1, 2) is None
    assert calls.qk_norm_rope_append(x, x, x, idx, pool, None, None, None, None, 1e-6, None, 0) is None   # on the CPU
    assert calls.qk_norm_rope_append(*[None] * 12) is None and calls.paged_prefill(*["q"] * 11) is None
    assert calls.paged_prefill(x, pool, idx[None], idx, None, 2, 1.0, 16, None, None, 0) is None


@pytest.mark.parametrize("built", [dict(), dict(ABI_VERSION=_lib.ABI_VERSION - 1), dict(ABI_VERSION=_lib.ABI_VERSION, TORCH_VERSION="1.0.0")])
def test_a_module_of_another_library_or_torch_is_refused(built, monkeypatch):
    right = _lib.calls()
    assert right.ABI_VERSION == _lib.ABI_VERSION and torch.__version__.startswith(right.TORCH_VERSION)
    other = types.ModuleType("llama_lite_npu_amd._calls")
    vars(other).update(built)
    monkeypatch.setitem(sys.modules, other.__name__, other)
    monkeypatch.setattr(llama_lite_npu_amd, "_calls", other)
    monkeypatch.setattr(_lib, "_calls", None)
    with pytest.raises(_lib.LiteKVError, match="was built for"):
        _lib.calls()


def test_building_the_library_builds_the_module(monkeypatch):
    made = []
    monkeypatch.setattr(build, "build_calls", lambda force=False: made.append(force))
    monkeypatch.setattr(build, "is_stale", lambda: False)
    build.build_library()
    assert made == [False]


class _NoCalls:
    @staticmethod
    def qk_norm_rope_append(*a):
        return None

    @staticmethod
    def paged_prefill(*a):
        return None


class _Sub(torch.Tensor):
    pass


def _state(fmt, d, hq=8, hkv=2, rows=37):
    gen = torch.Generator(device=DEV).manual_seed(d + rows)
    r = lambda *s: torch.randn(s, generator=gen, device=DEV, dtype=torch.float16)
    dtype = {"f16": torch.float16, "fp8": torch.uint8, "e4m3": torch.float8_e4m3fn, "int8": torch.int8}[fmt]
    st = dict(q=r(rows, hq, d), k=r(rows, hkv, d), v=r(rows, hkv, d), qw=1 + r(d) / 8, kw=1 + r(d) / 8, cos=r(rows, d),
              sin=r(rows, d), pool=torch.zeros((96, 2 * hkv, d), dtype=dtype, device=DEV),
              scales=None if fmt == "f16" else torch.full((2 * hkv,), 0.03, device=DEV),
              slots=torch.randperm(48, generator=gen, device=DEV)[:rows].to(torch.int32),
              table=torch.tensor([[1, 0, 2]], dtype=torch.int32, device=DEV),
              cu=torch.tensor([0, rows], dtype=torch.int32, device=DEV), ctx=None, max_q=rows, scale=d ** -0.5)
    return st


def _run(st):
    q = ops.qk_norm_rope_append(st["q"], st["k"], st["v"], st["slots"], st["pool"], st["qw"], st["kw"], st["cos"], st["sin"],
                                1e-6, kv_scales=st["scales"])
    out = ops.paged_prefill(q, st["pool"], st["table"], st["cu"], st["ctx"], st["max_q"], st["scale"], page_size=16,
                            kv_scales=st["scales"], max_kv_len=st["max_q"])
    torch.cuda.synchronize()
    return [out, st["q"].clone(), st["pool"].view(torch.int16 if st["pool"].dtype == torch.float16 else torch.uint8).clone()]


def _strided_q(st):      # q as a slice of a wider projection
    wide = torch.randn((37, 12, st["q"].shape[2]), device=DEV, dtype=torch.float16)
    wide[:, 2:10] = st["q"]
    st["q"] = wide[:, 2:10]


CHANGES = {
    "plain": lambda st: None,
    "q rows of a wider tensor": _strided_q,
    "no norm": lambda st: st.update(qw=None, kw=None),
    "no rotary": lambda st: st.update(cos=None, sin=None),
    "parameters": lambda st: st.update(qw=torch.nn.Parameter(st["qw"]), kw=torch.nn.Parameter(st["kw"])),
    "long cos": lambda st: st.update(cos=torch.cat([st["cos"]] * 2, 1), sin=torch.cat([st["sin"]] * 2, 1)),
    "cos with a batch dim": lambda st: st.update(cos=st["cos"][None], sin=st["sin"][None]),
    "int64 slots": lambda st: st.update(slots=st["slots"].long()),
    "int64 table": lambda st: st.update(table=st["table"].long()),
    "a view of a table": lambda st: st.update(table=torch.cat([st["table"]] * 2, 1)[:, :3]),
    "history": lambda st: st.update(ctx=torch.tensor([5], dtype=torch.int32, device=DEV)),
    "a subclass": lambda st: st.update(q=st["q"].as_subclass(_Sub)),
    # refused
    "q in bf16": lambda st: st.update(q=st["q"].bfloat16()),
    "k of another length": lambda st: st.update(k=st["k"][:-1]),
    "one norm": lambda st: st.update(kw=None),
    "short cos": lambda st: st.update(cos=st["cos"][:, :8], sin=st["sin"][:, :8]),
    "slots too few": lambda st: st.update(slots=st["slots"][:-1]),
    "scales of the wrong size": lambda st: st.update(scales=torch.ones(3, device=DEV)),
    "heads not contiguous": lambda st: st.update(q=st["q"].transpose(0, 1).contiguous().transpose(0, 1)),
    "misaligned q": lambda st: st.update(q=torch.zeros(st["q"].numel() + 1, device=DEV, dtype=torch.float16)[1:].view_as(st["q"])),
    "table of another batch": lambda st: st.update(table=torch.cat([st["table"]] * 2)),
    "odd pool": lambda st: st.update(pool=st["pool"][:, :3].contiguous()),
}


# What the native epilogue and the native prefill answer: T(aken), D(eclined), S(tatus of the library), - (not asked:
# the wrapper had refused the call before). Any other entry is taken by both.
ANSWERS = {
    "cos with a batch dim": "DT", "int64 slots": "DT", "int64 table": "TD", "a subclass": "DD", "q in bf16": "D-",
    "k of another length": "D-", "one norm": "D-", "short cos": "D-", "slots too few": "D-",
    "heads not contiguous": "D-", "misaligned q": "S-", "table of another batch": "TD", "odd pool": "D-",
}


class _Recorded:
    """The native calls and what they answered."""

    def __init__(self, calls):
        self.calls, self.answers = calls, ""

    def _note(self, answer):
        self.answers += "D" if answer is None else "S" if type(answer) is int else "T"
        return answer

    def qk_norm_rope_append(self, *a):
        return self._note(self.calls.qk_norm_rope_append(*a))

    def paged_prefill(self, *a):
        return self._note(self.calls.paged_prefill(*a))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["f16", "fp8", "e4m3", "int8"])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_the_wrappers_do_the_same_with_and_without_it(fmt, d, monkeypatch):
    print(f"native calls: {fmt} pool, heads of {d}", flush=True)
    native_calls = _lib.calls()
    for name, change in CHANGES.items():
        results, recorded = [], _Recorded(native_calls)
        for native in (True, False):
            st = _state(fmt, d)
            change(st)
            with monkeypatch.context() as m:
                m.setattr(_lib, "calls", lambda: recorded if native else _NoCalls)
                try:
                    results.append(_run(st))
                except (ValueError, _lib.LiteKVError) as e:
                    results.append(f"{type(e).__name__}: {e}")
        a, b = results
        if isinstance(b, str):
            assert a == b, name
        else:
            assert all(torch.equal(x, y) for x, y in zip(a, b)), name
        wrong_scales = "DD" if fmt == "f16" else "D-"       # an fp16 pool's epilogue does not look at them
        want = wrong_scales if name == "scales of the wrong size" else ANSWERS.get(name, "TT")
        assert recorded.answers.ljust(2, "-") == want, name


@pytest.mark.gpu
def test_a_plain_call_is_taken():
    print("native calls: taken", flush=True)
    st = _state("f16", 128)
    calls = _lib.calls()
    stream = torch.cuda.current_stream().cuda_stream
    assert calls.qk_norm_rope_append(st["q"], st["k"], st["v"], st["slots"], st["pool"], st["qw"], st["kw"], st["cos"],
                                     st["sin"], 1e-6, None, stream) is True
    out = calls.paged_prefill(st["q"], st["pool"], st["table"], st["cu"], None, 37, st["scale"], 16, None, 37, stream)
    torch.cuda.synchronize()
    assert out.shape == st["q"].shape and out.dtype == torch.float16 and bool(torch.isfinite(out).all())


class _LaunchError:
    """Native calls that reached the library and brought back a launch status."""

    def __init__(self):
        self.calls = 0

    def _status(self, *a):
        self.calls += 1
        return 2

    qk_norm_rope_append = paged_prefill = _status


class _Library:
    """Stands for liblitekv: any entry point but litekv_last_error is a second launch."""

    def __getattr__(self, name):
        raise AssertionError(f"{name} called after the native call had reached the library")

    @staticmethod
    def litekv_last_error():
        return b"launch failed"


def test_a_launch_error_is_raised_and_nothing_is_launched_again(monkeypatch):
    native = _LaunchError()
    monkeypatch.setattr(_lib, "calls", lambda: native)
    monkeypatch.setattr(_lib, "load", lambda: _Library())
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    q = type("OnTheGpu", (), {"is_cuda": True, "dtype": torch.float16})()
    with pytest.raises(_lib.LiteKVError, match="status 2: launch failed"):
        ops.qk_norm_rope_append(q, q, q, None, q)
    with pytest.raises(_lib.LiteKVError, match="status 2: launch failed"):
        ops.paged_prefill(q, q, None, None, None, 1, 1.0)
    assert native.calls == 2


@pytest.mark.gpu
def test_a_status_of_the_library_comes_back():
    print("native calls: statuses", flush=True)
    st = _state("f16", 128)
    CHANGES["misaligned q"](st)         # the library's own check
    calls, before = _lib.calls(), st["q"].clone()
    stream = torch.cuda.current_stream().cuda_stream
    for status in (calls.qk_norm_rope_append(st["q"], st["k"], st["v"], st["slots"], st["pool"], st["qw"], st["kw"], st["cos"],
                                             st["sin"], 1e-6, None, stream),
                   calls.paged_prefill(st["q"], st["pool"], st["table"], st["cu"], None, 37, st["scale"], 16, None, 37, stream)):
        assert type(status) is int and status == 1
        with pytest.raises(_lib.LiteKVError, match="align"):
            _lib.check(status)
    assert torch.equal(st["q"], before)
