"""The calls of the native libraries' functions, against the same calls through ctypes."""

import ctypes
import random
import subprocess

import numpy as np
import pytest
import torch

from distie_amd.kernels import calls

P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
C_NAMES = {P: "void*", I: "int", L: "long", F: "float"}


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    """-> a function that gives a library whose `distie_all` writes down the arguments that it got"""
    folder = tmp_path_factory.mktemp("calls")

    def make(kinds):
        name = "k" + "".join({P: "p", I: "i", L: "l", F: "f"}[k] for k in kinds)
        args = ", ".join(f"{C_NAMES[k]} a{i}" for i, k in enumerate(kinds))
        # (a float goes down as its bits)
        body = "".join(f"{{ float f = a{i}; unsigned u; __builtin_memcpy(&u, &f, 4); seen[{i}] = u; }}" if k is F else
                       f"seen[{i}] = (long)a{i};" for i, k in enumerate(kinds))
        (folder / f"{name}.c").write_text(f"long seen[64]; long* distie_seen(void) {{ return seen; }}\n"
                                          f"int distie_all({args}) {{ {body} return {-3 - len(kinds)}; }}\n")
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(folder / f"{name}.c"), "-o", str(folder / f"{name}.so")], check=True)
        lib = ctypes.CDLL(str(folder / f"{name}.so"))
        lib.distie_seen.restype = ctypes.POINTER(ctypes.c_long)
        lib.distie_all.argtypes = kinds
        return lib
    return make


@pytest.mark.parametrize("count, floats", [(1, 0), (6, 0), (7, 1), (14, 8), (21, 2), (40, 0), (48, 8)])
def test_a_function_gets_what_ctypes_gives_it(build, count, floats):
    rng = random.Random(count)
    kinds = [F] * floats + [rng.choice([P, I, L]) for _ in range(count - floats)]
    rng.shuffle(kinds)
    lib = build(kinds)
    tensors = [torch.zeros(3), torch.zeros(4, 5)[:, 1:], torch.zeros(0)]
    for trial in range(3):
        given = [{P: lambda: rng.choice([None, 0, (1 << 63) + 5, rng.choice(tensors)]), I: lambda: rng.choice([-1, 0, 2**31 - 1, True]),
                  L: lambda: rng.choice([-1, -(1 << 62), 7, np.int64(9)]), F: lambda: rng.choice([0.1, -3, np.float32(2.5), float("inf")])}[k]()
                 for k in kinds]
        plain = [g.data_ptr() if isinstance(g, torch.Tensor) else g for g in given]
        slow = ctypes.CDLL(lib._name)
        slow.distie_seen.restype, slow.distie_all.argtypes = ctypes.POINTER(ctypes.c_long), kinds
        assert slow.distie_all(*plain) == -3 - count
        want = slow.distie_seen()[:count]
        calls.quicken(lib)
        assert lib.distie_all(*given) == -3 - count
        assert lib.distie_seen()[:count] == want


def test_arguments_that_are_no_numbers(build):
    lib = build([P, I, P])
    calls.quicken(lib)
    array = (ctypes.c_int * 2)(1, 2)
    t = torch.zeros(2)
    assert lib.distie_all(t, 4, array) == -6                       # as ctypes takes it
    assert lib.distie_seen()[:3] == [t.data_ptr(), 4, ctypes.addressof(array)]
    for bad in ((t, 4), (t, 4, None, 5), (t, t, None), (t, 0.5, None), (object(), 4, None)):
        with pytest.raises((TypeError, ctypes.ArgumentError)):
            lib.distie_all(*bad)
    other = ctypes.CDLL(lib._name)
    other.distie_all.argtypes = [P, I, ctypes.POINTER(I)]         # not for the quick way: left as it is
    before = other.distie_all
    calls.quicken(other)
    assert other.distie_all is before


@pytest.mark.gpu
def test_allocations_and_owners_on_the_device():
    native = calls.native()
    for shape, dtype in (((3, 5), torch.bfloat16), ((0, 4), torch.float32), (torch.Size([2]), torch.int32), (7, torch.uint8)):
        t = native.empty(0, shape, dtype)
        assert (tuple(t.shape), t.dtype, t.device, t.is_contiguous()) == \
            ((shape,) if isinstance(shape, int) else tuple(shape), dtype, torch.device("cuda:0"), True)
    with pytest.raises(torch.OutOfMemoryError):
        native.empty(0, (1 << 44,), torch.float32)
    a = torch.zeros(4, 6, device="cuda:0")
    assert native.owned(0, a, None, a[1:]) and native.owned(0)
    assert not native.owned(0, a, a[:, 1:]) and not native.owned(0, a.cpu()) and not native.owned(-1, a) and not native.owned(0, 3)
