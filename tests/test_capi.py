"""The C ABI: the built library loads and exports every entry point the
header declares, and the ctypes table matches the header (CPU only; no
kernel is launched)."""

from __future__ import annotations

import ctypes
import os
import re
import sys

import pytest

from opengenie_amd import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "opengenie_amd.h")


def declared_functions() -> list[str]:
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(oga_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    names = declared_functions()
    assert "oga_fp8_linear" in names and "oga_adazero_from_ada" in names
    assert len(names) >= 20


def test_ctypes_table_matches_header():
    assert sorted(_lib.SIGNATURES) == declared_functions()


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, missing


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_abi_version_and_error_reporting():
    lib = _lib.load()
    assert lib.oga_abi_version() == 1
    # Argument errors are reported without touching a device.
    rc = lib.oga_fp8_linear(None, 0, None, 0, None, None, None, 0, None, 0, 1, 1, 128, None)
    assert rc == -1
    assert b"null" in lib.oga_last_error()
    rc = lib.oga_bias_add_bf16(None, None, 0, None, 1, 1, None)
    assert rc == -1


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_native_module_binds_the_same_library():
    """The compiled module's functions are the library's: arguments of every
    kind (None, ints, a tuple and a ctypes array as int64_t arrays, a float)
    reach the checks of the entry point, whose message the ctypes handle of
    the same library reports; wrong counts and types raise."""
    from opengenie_amd import _native

    names = {n for n in dir(_native) if n.startswith("oga_")}
    assert names and names <= set(_lib.SIGNATURES)
    for st in ((1, 1, 1, 1), _lib.strides((1, 1, 1, 1))):
        rc = _native.oga_adazero_from_ada(4096, 4096, 1, 1, 100, 4096, 0, 1, 1, 4096, 0, st, 0, 1, 1e-6, None)
        assert rc < 0 and _lib.load().oga_last_error()
    assert _lib.function("oga_bias_add_bf16")(None, None, 0, None, 1, 1, None) == -1
    assert b"null" in _lib.load().oga_last_error()
    with pytest.raises(TypeError):
        _native.oga_bias_add_bf16(None)
    with pytest.raises(TypeError):
        _native.oga_bias_add_bf16(None, None, "0", None, 1, 1, None)
    with pytest.raises(OverflowError):
        _native.oga_bias_add_bf16(None, None, 1 << 40, None, 1, 1, None)
    with pytest.raises(ValueError):
        _native.oga_adazero_from_ada(4096, 4096, 1, 1, 4096, 4096, 0, 1, 1, 4096, 0, (1,) * 9, 0, 1, 1e-6, None)
    with pytest.raises(_lib.KernelError):
        _lib.call("oga_bias_add_bf16", None, None, 0, None, 1, 1, None)


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_wrappers_call_through_ctypes_without_the_native_module(monkeypatch):
    """An interpreter the compiled module was not built for calls the same
    library through ctypes, with the arguments the wrappers pass to either."""
    monkeypatch.setitem(sys.modules, "opengenie_amd._native", None)  # its import fails
    monkeypatch.delattr("opengenie_amd._native", raising=False)
    monkeypatch.setattr(_lib, "_fns", {})
    assert _lib.function("oga_adazero_from_ada") is _lib.load().oga_adazero_from_ada
    for st in ((1, 1, 1, 1), _lib.strides((1, 1, 1, 1))):
        with pytest.raises(_lib.KernelError, match="4096"):  # channels
            _lib.call("oga_adazero_from_ada", 4096, 4096, 1, 1, 100, 4096, 0, 1, 1, 4096, 0, st, 0, 1, 1e-6, None)
    with pytest.raises(_lib.KernelError, match="null"):
        _lib.call("oga_attention_ws", None, (1, 1, 1), None, (1, 1, 1), None, (1, 1, 1), None, (1, 1, 1), 1, 1, 1, 1,
                  128, 1.0, None, 0, None)
    assert _lib.function("oga_attention_workspace_bytes")(0, 1, 1, 1, 128) == 0


def test_the_library_builds_without_python_headers(monkeypatch, tmp_path):
    """Without Python.h there is no compiled module, an older one goes, and
    building says so instead of failing."""
    from opengenie_amd import build

    old = tmp_path / "_native.cpython-39-x86_64-linux-gnu.so"
    old.write_bytes(b"")
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build._build_native() is False and not old.exists()


def _attention_plan(fp8, batch, nq, nk, heads, cus=256):
    plan = (ctypes.c_int64 * 4)()
    assert _lib.load().oga_attention_plan(fp8, batch, nq, nk, heads, cus, plan) == 0
    return tuple(plan)


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_attention_plans():
    """Schedules on 256 CUs: the blocks of a plan cover the queries, whole ones
    fill rounds of the resident workgroups, parts are two to eight and no
    shorter than a key step, and none up to 16 key steps; the forms and splits
    of a few shapes as their comments in the kernels' source describe them."""
    for fp8, n in [(f, n) for f in (0, 1) for n in (1, 63, 512, 1024, 1025, 1537, 2304, 3500, 4999, 9216, 14080)]:
        for batch, heads in ((1, 32), (1, 1), (2, 24), (3, 40)):
            qpb, blocks, full, parts = _attention_plan(fp8, batch, n, n, heads)
            slots = {(0, 256): 256, (0, 128): 512, (1, 384): 256, (1, 128): 768}[fp8, qpb]
            assert blocks == batch * heads * -(-n // qpb) and 1 <= parts <= 8
            assert full == blocks if parts == 1 else full == blocks // slots * slots < blocks
            assert parts == 1 or n > 1024
    assert _attention_plan(0, 1, 1537, 1537, 32) == (256, 224, 224, 1)
    assert _attention_plan(0, 1, 9216, 9216, 32) == (256, 1152, 1024, 2)
    assert _attention_plan(1, 1, 4999, 4999, 32) == (128, 1280, 1280, 1)
    assert _attention_plan(1, 1, 4352, 4352, 32) == (384, 384, 256, 2)
    assert _attention_plan(1, 1, 9216, 9216, 32) == (384, 768, 768, 1)
    lib = _lib.load()
    assert lib.oga_attention_plan(0, 1, 1, 1, 1, 256, None) < 0
    assert lib.oga_attention_plan(0, 1, 0, 1, 1, 256, (ctypes.c_int64 * 4)()) < 0


def _linear_plan(m, n, k, ws=1 << 62, cus=256):
    plan = (ctypes.c_int64 * 4)()
    assert _lib.load().oga_fp8_linear_plan(m, n, k, ws, cus, plan) == 0
    return tuple(plan)


@pytest.mark.skipif(not _lib.available(), reason="library not built")
def test_fp8_linear_plans():
    """Schedules on 256 CUs: whole tiles cover the output, K-chunks are cut
    from 256 x 256 tiles past whole rounds only, and never without a
    workspace; the tiles of shapes that the kernel's comments name."""
    for n, k in ((128, 256), (4096, 4096), (4096, 16384), (16384, 4096), (12288, 4096), (4224, 384)):
        for m in (1, 64, 65, 256, 1152, 1537, 2304, 4100, 4352, 4999, 9216, 14080):
            for ws in (0, 1 << 62):
                bm, bn, full, split = _linear_plan(m, n, k, ws)
                tiles = -(-m // bm) * -(-n // bn)
                assert split == 1 or (ws and (bm, bn) == (256, 256) and full == tiles // 256 * 256 < tiles)
                assert split > 1 or full == tiles
    assert _linear_plan(256, 4096, 4096) == (64, 128, 128, 1)
    assert _linear_plan(1152, 4096, 4096) == (192, 128, 192, 1)
    assert _linear_plan(1537, 4096, 4096) == (128, 256, 208, 1)
    assert _linear_plan(9216, 4096, 4096) == (192, 256, 768, 1)
    assert _linear_plan(9216, 4096, 16384) == (256, 256, 512, 4)
    assert _linear_plan(9216, 4096, 16384, 0)[3] == 1
    lib = _lib.load()
    assert lib.oga_fp8_linear_plan(1, 128, 128, 0, 256, (ctypes.c_int64 * 4)()) < 0
    assert lib.oga_fp8_linear_plan(1, 128, 256, 0, 256, None) < 0
