"""Operand checks in native code: they say what the Python check says, for every form of a call, and where the module is neither
built nor can be built the Python check is what runs."""

from __future__ import annotations

import os

import pytest
import torch

from kvforge_amd.kernels import library, ops


def outcome(f, args, kwargs):
    try:
        return f(*args, **kwargs)
    except Exception as e:  # noqa: BLE001
        return type(e).__name__, str(e).replace("_check() ", "").replace("check() ", "")


def forms(dev):
    """Calls of the check: tensors of every kind, shapes as tuples, lists and torch's, by place and by name."""
    f32, i32 = torch.float32, torch.int32
    t = torch.zeros(3, 8, device=dev)
    tensors = [t, t.to(torch.bfloat16), t[:, :4], t.t(), t[:0], torch.zeros((), device=dev), torch.zeros(8, dtype=i32, device=dev),
               torch.zeros(3, 8), torch.nn.Parameter(t), torch.zeros(1, 8, device=dev)[:, ::2], t.to_sparse(), None, 5, [1.0]]
    shapes = [None, (3, 8), (None, 8), (None, None), (3, None), (3,), (), (8,), (True, 8), [3, 8], [None, 8], torch.Size([3, 8]), (3, -1),
              (3, 1 << 70), (3, 8.0), (3, "8"), (0, 8), (3, 4)]
    for x in tensors:
        for shape in shapes:
            for dtype in (None, f32, i32):
                for contiguous in (True, False):
                    yield (x, "x", dtype, shape, contiguous), {}
        yield (x, "x"), {}
        yield (x, "x", f32), {}
        yield (x, "x", f32, (None, 8)), {}
        yield (x, "x"), dict(contiguous=False)
        yield (x, "x"), dict(shape=(3, 8), dtype=f32)
        yield (x, "x", None), dict(shape=(3, None), contiguous=False)
        yield (x,), dict(name="x", contiguous=False)
        yield (), dict(t=x, name="x")
        yield (x, "x"), dict(contiguous=1)
        yield (x, "x"), dict(contiguous=0)
        yield (x, "x", "float32"), {}
    yield (t, "x", f32), dict(dtype=f32)
    yield (t, "x"), dict(strides=(8, 1))
    yield (t, "x", f32, (3, 8), True, 1), {}
    yield (t,), {}
    yield (), {}


def native_check():
    native = library.load_host("hostcheck")
    assert native is not None
    native.set_slow(ops._check_in_python)
    return native


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_native_check_says_what_the_python_check_says(dev):
    native, passed = native_check(), 0
    for args, kwargs in forms(dev):
        want = outcome(ops._check_in_python, args, kwargs)
        assert outcome(native.check, args, kwargs) == want, (args, kwargs)
        passed += want is None
    assert passed > 100 if dev == "cuda" else passed == 0


@pytest.mark.gpu
def test_native_operands_are_those_of_the_python_form(monkeypatch):
    native, f = native_check(), torch.zeros
    g = dict(device="cuda")
    calls = [(f(4, 16, **g), f(8, 16, **g), f(4, 8, **g)), (f(4, 32, **g)[:, :16], f(8, 16, **g), f(4, 24, **g)[:, 8:16]),
             (f(1, 32, **g)[:, :16], f(8, 16, **g), f(1, 24, **g)[:, :8]), (f(0, 16, **g), f(8, 16, **g), f(0, 8, **g)),
             (f(4, 16, **g), f(8, 16, **g), f(4, 4, **g)), (f(4, 16, **g), f(7, 16, **g), f(4, 3, **g)), (f(4, 15, **g), f(8, 16, **g), f(4, 8, **g)),
             (f(4, 16), f(8, 16, **g), f(4, 8, **g)), (f(4, 16, **g), f(8, 16), f(4, 8, **g)), (f(16, 4, **g).t(), f(8, 16, **g), f(4, 8, **g)),
             (f(4, 16, **g), f(16, 8, **g).t(), f(4, 8, **g)), (f(4, 16, **g), f(8, 16, **g), f(8, 4, **g).t()),
             (f(2, 4, 16, **g), f(8, 16, **g), f(4, 8, **g)), (f(4, 16, **g), f(8, 16, **g), f(4, 8, **g).to_sparse())]
    for call in calls:
        for columns in (ops._whole, ops._halves):
            got = []
            for form in (None, native.operands):
                monkeypatch.setattr(ops, "_operands", form)
                got.append(outcome(ops._gemm_operands, (*call, columns), {}))
            assert got[0] == got[1], [tuple(t.shape) for t in call]


@pytest.fixture
def no_compiler(monkeypatch, tmp_path):
    """A process that has loaded no host module and finds no compiler (the module has been built before)."""
    library.build_module("hostcheck")
    monkeypatch.setattr(library, "_loaded_host", {})
    monkeypatch.setenv("PATH", str(tmp_path))
    said = []
    monkeypatch.setattr(library, "_log", said.append)
    return said


def test_a_built_host_module_needs_no_compiler(no_compiler):
    path = library.build_module("hostcheck")
    assert os.path.isfile(path) and library.load_host("hostcheck") is not None and not no_compiler


def test_without_host_module_and_compiler_python_checks(no_compiler, monkeypatch):
    monkeypatch.setattr(library, "_find_built", lambda name, want: None)
    with pytest.raises(library.KernelBuildError, match="hostcheck"):
        library.build_module("hostcheck", verbose=False)
    monkeypatch.setattr(ops, "_check", ops._check_in_python)
    monkeypatch.setattr(ops, "_operands", None)
    del no_compiler[:]
    library.ensure([])
    ops._check_natively()
    ops._check_natively()
    assert ops._check is ops._check_in_python and ops._operands is None
    assert sum("hostcheck is done without" in line for line in no_compiler) == 1


def test_a_host_module_that_does_not_load_is_done_without(no_compiler, monkeypatch, tmp_path):
    broken = tmp_path / "hostcheck.so"
    broken.write_bytes(b"no library")
    monkeypatch.setattr(library, "_find_built", lambda name, want: str(broken))
    assert library.load_host("hostcheck") is None and len(no_compiler) == 1
