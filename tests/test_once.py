"""The tables' set-up (tp_once.h): made once over all threads, and a failure is
not kept: the next caller tries again."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("once") / "libonce.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "once_check.cpp"), "-o", str(out)], check=True)
    return C.CDLL(str(out))


@pytest.mark.parametrize("threads,rounds,failures", [(1, 5, 0), (1, 5, 3), (8, 200, 0), (8, 200, 5), (4, 1, 100)])
def test_made_once_and_tried_again(lib, threads, rounds, failures):
    ok, early = C.c_int(), C.c_int()
    made = lib.tp_once_check(threads, rounds, failures, C.byref(ok), C.byref(early))
    calls = threads * rounds
    assert made == (1 if calls > failures else -1)
    assert ok.value == max(0, calls - failures) and early.value == 0
