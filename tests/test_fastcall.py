"""GemmPlan.run's binding of the launch (csrc/fastcall.c): what it takes, what it refuses, and that refusals are ctypes'."""
import ctypes
import importlib.machinery

import numpy as np
import pytest

from aster_amd import _capi, build
from aster_amd.gemm import GemmPlan


def empty_plan():
    return GemmPlan.create(0, 16, 64, "bf16", "f32")   # M = 0: accepted, nothing is launched


def test_integers_none_and_what_ctypes_takes():
    p = empty_plan()
    p.run(16, 32, 48)
    p.run(16, 32, 48, bias=None, stream=0, workspace=None)
    p.run(ctypes.c_void_p(16), 32, 48)                  # not an integer: the structure takes it
    p.run(True, 2 ** 63 + 16, -16)                      # masked to 64 bits, as in the structure


@pytest.mark.parametrize("bad", ["16", 1.5, np.int64(16), object()])
def test_refusals_are_type_errors(bad):
    p = empty_plan()
    with pytest.raises(TypeError):
        p.run(bad, 32, 48)
    with pytest.raises(TypeError):
        p.run(16, 32, 48, workspace_bytes=None)


def test_binding_checks_its_arguments():
    _capi.load()
    with pytest.raises(TypeError):
        _capi.fast_run(empty_plan().config, 1, 2, 3)
    with pytest.raises(TypeError):
        _capi.fast_run(ctypes.c_int(3), *[None] * 9, 0, None)


def test_status_becomes_the_exception():
    p = GemmPlan.create(16, 16, 64, "bf16", "f32")
    with pytest.raises(_capi.AsterGemmError, match="non-null"):
        p.run(0, 32, 48)


def test_without_the_binding_launches_go_through_ctypes(monkeypatch, tmp_path):
    monkeypatch.setattr(_capi, "_lib", None)
    monkeypatch.setattr(_capi, "fast_run", None)
    monkeypatch.setattr(_capi, "_FASTCALL_PATH", str(tmp_path / "none.so"))
    p = empty_plan()
    p.run(16, 32, 48, stream=0)
    assert _capi.fast_run is None
    with pytest.raises(TypeError):
        p.run("16", 32, 48)
    p = GemmPlan.create(16, 16, 64, "bf16", "f32")
    with pytest.raises(_capi.AsterGemmError, match="non-null"):
        p.run(0, 32, 48)


def test_the_binding_belongs_to_one_interpreter(monkeypatch, tmp_path):
    assert any(_capi._FASTCALL_PATH.endswith(s) and len(s) > 3 for s in importlib.machinery.EXTENSION_SUFFIXES)
    monkeypatch.setattr(build, "FASTCALL_PATH", str(tmp_path / "aster_fastcall.so"))
    monkeypatch.setenv("CC", str(tmp_path / "no-such-compiler"))
    assert not build.build_fastcall() and not list(tmp_path.iterdir())


@pytest.mark.parametrize("where", ["dA", "dB", "dC", "scale_a", "scale_b", "bias"])
def test_addresses_past_48_bits_are_refused(where):
    """Kernels take theirs in 48 bits (PackedArgs): one more would be another address."""
    p = GemmPlan.create(16, 16, 64, "fp8_e4m3", "f32", has_bias=True)
    ops = dict(dA=16, dB=32, dC=48, scale_a=64, scale_b=64, bias=64)
    ops[where] = 1 << 48
    with pytest.raises(_capi.AsterGemmError, match="48 bits"):
        p.run(**ops)


def test_workspaces_past_48_bits_are_refused_where_they_are_used():
    p = GemmPlan.create(500, 4096, 14336, "bf16", "bf16")
    with pytest.raises(_capi.AsterGemmError, match="48 bits"):
        p.run(16, 32, 48, workspace=1 << 48, workspace_bytes=p.workspace_bytes() or 1)
    assert p.workspace_bytes() > 0


def test_pitches_of_c_past_58_bits_are_refused():
    p = GemmPlan.create(2, 16, 64, "bf16", "f32", ldc=1 << 58)
    with pytest.raises(_capi.AsterGemmError, match="58"):
        p.run(16, 32, 48)
