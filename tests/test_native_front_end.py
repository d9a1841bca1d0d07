"""The ops' native front end (_native) against the general Python code it stands in for:
the same outputs bit for bit over the argument forms it takes and those it leaves, and the
same errors."""
import importlib.util
import math
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

import oxide_paged_kv as ox
from oxide_paged_kv import ops

REPO = Path(__file__).resolve().parent.parent

def _general(monkeypatch):
    """ops with the native front end declining every call."""
    class Declines:
        def __getattr__(self, name):
            return lambda *args: None

    monkeypatch.setattr(ops, "_native", Declines())


def _inputs(device, dtype=torch.bfloat16, B=3, Hq=8, Hkv=4, D=128, BS=64):
    g = torch.Generator(device="cpu").manual_seed(3)
    rnd = lambda *s: torch.randn(s, generator=g).to(dtype).to(device)  # noqa: E731
    lens = torch.tensor([70, 1, 130], dtype=torch.int32)
    table = torch.tensor([[2, 5, 0], [1, 0, 0], [7, 3, 4]], dtype=torch.int32)
    cu = torch.zeros(B + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(lens, 0)
    slots = torch.tensor([5 * BS + 5, BS, 4 * BS + 1], dtype=torch.int64)
    return {"q": rnd(B, Hq, D), "k": rnd(8, BS, Hkv, D), "v": rnd(8, BS, Hkv, D), "key": rnd(B, Hkv, D),
            "value": rnd(B, Hkv, D), "qkv": rnd(B, (Hq + 2 * Hkv) * D), "w": rnd(D), "cu": cu.to(device),
            "lens": lens.to(device), "table": table.to(device), "slots": slots.to(device),
            "rope": ox.rope_cos_sin_cache(256, D, device=device), "pos": (lens - 1).to(device), "BS": BS}


def _calls(s):
    """The calls of a step, in the forms the native code takes and in others."""
    BS, sc = s["BS"], 1 / math.sqrt(128)
    out = []
    for window, append, cu, scale in ((None, None, s["cu"], sc), (50, None, s["cu"].view(torch.uint32), sc),
                                      (None, (s["key"], s["value"], s["slots"]), s["cu"], sc),
                                      (None, [s["key"], s["value"], s["slots"]], s["cu"], np.float64(sc))):
        k, v = s["k"].clone(), s["v"].clone()
        out += [ox.decode_attn(s["q"], k, v, cu, s["table"], 130, scale, window_left=window, page_block_size=BS,
                               append=append), k, v]
    given, ws = torch.empty_like(s["q"]), torch.empty(1 << 22, dtype=torch.uint8, device=s["q"].device)
    r = ox.decode_attn(s["q"], s["k"], s["v"], s["cu"], s["table"], 130, sc, page_block_size=BS, out=given,
                       workspace=ws)
    assert r is given
    out.append(r.clone())
    cq = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device=s["q"].device)
    rows = s["k"].reshape(-1, *s["k"].shape[2:])
    for window in (None, 40):
        out.append(ox.prefill_attn(s["q"], s["k"], s["v"], cq, s["cu"], 1, 130, sc, s["table"], window))
        out.append(ox.prefill_attn(s["q"], rows, s["v"].reshape(rows.shape), cq, s["cu"], 1, 130, sc,
                                   window_left=window))
    for w, slots in ((s["w"], s["slots"]), (None, None)):
        k, v = s["k"].clone(), s["v"].clone()
        cache = (k, v, slots) if slots is not None else (None, None, None)
        out += [ox.qk_norm_rope_and_cache(s["qkv"], 8, 4, w, w, 1e-6, s["rope"], s["pos"], *cache), k, v]
    out.append(ox.qk_norm_rope_and_cache(s["qkv"], 8, 4, s["w"], s["w"], 1e-6, s["rope"], s["pos"], return_k=True)[1])
    return out + list(ox.build_decode_metadata(s["lens"], s["table"], BS))


class _Counts:
    """The native front end, noting which calls it took (True) and which it declined."""

    def __init__(self, native):
        self.native, self.taken = native, []

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.native, name)(*args)
            self.taken.append((name, r is not None))
            return r
        return call


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_native_calls_equal_general_calls(device, dtype, monkeypatch):
    print(f"native front end {dtype}", flush=True)
    counts = _Counts(ops._native)
    monkeypatch.setattr(ops, "_native", counts)
    got = _calls(_inputs(device, dtype))
    # Declined: the decode call with an append list and a numpy scale; return_k is not asked.
    assert counts.taken == [("decode", True)] * 3 + [("decode", False), ("decode", True)] + \
        [("prefill", True)] * 4 + [("prologue", True)] * 2 + [("metadata", True)]
    _general(monkeypatch)
    want = _calls(_inputs(device, dtype))
    torch.cuda.synchronize()
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and g.shape == w.shape and torch.equal(g, w)


@pytest.mark.gpu
def test_library_errors_raise_through_the_native_calls(device, monkeypatch):
    """Errors the library records (a workspace-free shape check here: head size 96)."""
    counts = _Counts(ops._native)
    monkeypatch.setattr(ops, "_native", counts)
    q = torch.zeros(1, 4, 96, dtype=torch.bfloat16, device=device)
    k = torch.zeros(2, 64, 2, 96, dtype=torch.bfloat16, device=device)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=device)  # noqa: E731
    for _ in range(2):  # the error is cleared when it is raised
        with pytest.raises(ox.OxideError):
            ox.decode_attn(q, k, k, i32(0, 5), i32(0)[None], 5, 0.1, page_block_size=64)
        with pytest.raises(ox.OxideError):
            ox.prefill_attn(q, k, k, i32(0, 1), i32(0, 5), 1, 5, 0.1, i32(0)[None])
    assert counts.taken == [("decode", True), ("prefill", True)] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("general", [False, True], ids=["native", "general"])
def test_prefill_without_room_for_a_workspace(device, general, monkeypatch):
    """A prefill call whose workspace does not fit into the memory left attends without one."""
    if general:
        _general(monkeypatch)
    g = torch.Generator(device=device).manual_seed(5)
    rnd = lambda *s: torch.randn(s, generator=g, device=device, dtype=torch.bfloat16)  # noqa: E731
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=device)  # noqa: E731
    q, k, v = rnd(512, 32, 128), rnd(8192, 8, 128), rnd(8192, 8, 128)
    out = torch.empty_like(q)
    cq, ck = i32(0, 512), i32(0, 8192)
    L = ox.load()
    need = L.prefill_attention_workspace_size(1, 32, 8, 128, 512, 8192, -1)
    assert need > 30 << 20
    call = lambda o: ox.prefill_attn(q, k, v, cq, ck, 512, 8192, 0.09, out=o)  # noqa: E731
    want = torch.empty_like(out)
    L.varlen_prefill_attention(want.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), cq.data_ptr(), ck.data_ptr(),
                               8192, 1, 32, 8, 128, 512, 8192, -1, 0.09, 1, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(device) + (1 << 20)) / total, device)
        held = []  # what the allocator still has of that size (after other tests)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while True:
                held.append(torch.empty(need, dtype=torch.uint8, device=device))
        assert call(out) is out
    finally:
        held = None
        torch.cuda.set_per_process_memory_fraction(1.0, device)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    assert not torch.equal(call(torch.empty_like(out)), want)  # with a workspace its keys are split


def test_host_tensors_are_refused_alike(monkeypatch):
    s = _inputs("cpu")
    calls = [lambda: ox.decode_attn(s["q"], s["k"], s["v"], s["cu"], s["table"], 130, 0.1, page_block_size=64),
             lambda: ox.decode_attn(s["q"], s["k"], s["v"], s["cu"], s["table"], 130, 0.1, page_block_size=32),
             lambda: ox.decode_attn(s["q"], s["k"].float(), s["v"], s["cu"], s["table"], 130, 0.1, page_block_size=64),
             lambda: ox.prefill_attn(s["q"], s["k"], s["v"], s["cu"], s["cu"], 1, 130, 0.1, s["table"]),
             lambda: ox.qk_norm_rope_and_cache(s["qkv"], 8, 4, None, None, 1e-6, s["rope"], s["pos"].long()),
             lambda: ox.build_decode_metadata(s["lens"].long(), s["table"], 64)]
    messages = []
    for general in (False, True):
        if general:
            _general(monkeypatch)
        for call in calls:
            with pytest.raises(ox.OxideError) as e:
                call()
            messages.append(str(e.value))
    assert messages[:len(calls)] == messages[len(calls):]


_STEP = """
import sys
sys.path[:0] = [{root!r}, {pkg!r}]
{before}
import torch
import oxide_paged_kv as ox
from oxide_paged_kv import _lib, ops
ox.load()
assert _lib._native is None
q = torch.zeros(1, 4, 128, dtype=torch.bfloat16)
k = torch.zeros(2, 64, 2, 128, dtype=torch.bfloat16)
i = torch.tensor([0, 5], dtype=torch.int32)
try:
    ox.decode_attn(q, k, k, i, i[None], 5, 0.1, page_block_size=64)
except ox.OxideError as e:
    print("general:", e)
"""


@pytest.mark.parametrize("before", ["sys.modules['oxide_paged_kv._native'] = None",
                                    "import torch; torch.__version__ += '.other'"], ids=["absent", "other-torch"])
def test_package_works_without_the_native_module(before):
    """No module (as after make), or one built against another torch: the general code runs."""
    code = _STEP.format(root=str(REPO), pkg=str(REPO / "vllm-oxide_amd"), before=before)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout == "general: expected a device tensor\n"


def _build_module():
    spec = importlib.util.spec_from_file_location("oxide_build", REPO / "vllm-oxide_amd" / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_c_libraries_are_linked_whatever_the_native_module_does(monkeypatch, tmp_path):
    b = _build_module()
    done = []

    def run(cmd, **kw):
        done.append("archive" if cmd[0] == "ar" else "link" if "-shared" in cmd else "compile")
        return subprocess.CompletedProcess(cmd, 0, "", "")

    def fails():
        raise RuntimeError("no native module")

    monkeypatch.setattr(b, "BUILD", tmp_path)
    monkeypatch.setattr(b, "RESOURCES", tmp_path / "r.json")
    monkeypatch.setattr(b, "LIB", tmp_path / "l.so")
    monkeypatch.setattr(b, "STATIC_LIB", tmp_path / "l.a")
    monkeypatch.setattr(b, "build_native", fails)
    monkeypatch.setattr(b, "build_host_test", lambda: done.append("host test"))
    monkeypatch.setattr(b.subprocess, "run", run)
    with pytest.raises(RuntimeError, match="no native module"):
        b.build()
    assert done[-3:] == ["link", "archive", "host test"]


def test_native_module_is_left_out_without_torch_or_compiler(monkeypatch, tmp_path, capsys):
    b = _build_module()
    monkeypatch.setattr(b, "NATIVE_LIB", tmp_path / b.NATIVE_LIB.name)
    (tmp_path / "_native.so").write_bytes(b"stale")
    monkeypatch.setattr(b.shutil, "which", lambda name: None)
    assert b.build_native() is None and not list(tmp_path.iterdir())
    monkeypatch.setitem(sys.modules, "torch", None)
    assert b.build_native() is None
    assert capsys.readouterr().err.count("native front end not built") == 2
