"""The numbers by which the host tells the answer of a decomposition from that of an earlier one (host code only)."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparsetir_amd", "csrc")
SOURCE = """
#include "call_answer.h"
extern "C" {
uint32_t numbers() { return stir::kCallNumbers; }
uint32_t next(uint32_t n) { return stir::next_call(n); }
void forget(uint64_t* a, int n) { stir::forget_answers(a, n); }
int there(const uint64_t* a, uint32_t n) { return stir::answered(a, n); }
int64_t rows(uint64_t a) { return stir::answered_rows(a); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("answer")
    (d / "a.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "a.cpp"), "-o", str(d / "a.so")],
                   check=True)
    out = ctypes.CDLL(str(d / "a.so"))
    out.numbers.restype = out.next.restype = ctypes.c_uint32
    out.next.argtypes = [ctypes.c_uint32]
    out.forget.argtypes = [ctypes.c_void_p, ctypes.c_int]
    out.there.argtypes = [ctypes.c_void_p, ctypes.c_uint32]
    out.rows.argtypes, out.rows.restype = [ctypes.c_uint64], ctypes.c_int64
    return out


def test_an_answer_never_written_is_no_answer(lib):
    """At the number behind the last one, and everywhere else."""
    box = (ctypes.c_uint64 * 1)(0)
    number = lib.numbers() - 3
    for _ in range(6):
        number = lib.next(number)
        assert not lib.there(box, number)


def test_an_old_answer_of_the_same_number_is_no_answer(lib):
    """A bucket answered as many calls ago as there are numbers."""
    box = (ctypes.c_uint64 * 2)((5 << 40) | 77, (5 << 40) | 78)
    assert lib.there(box, 5) and lib.rows(box[0]) == 77
    lib.forget(box, 1)
    assert not lib.there(box, 5)
    assert box[1] == (5 << 40) | 78


def test_numbers_go_round(lib):
    last = lib.numbers() - 1
    assert lib.next(0) == 1 and lib.next(1) == 2 and lib.next(last - 1) == last and lib.next(last) == 1
