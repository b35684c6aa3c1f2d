"""The MFMA gridder's work shape (csrc/work_shape.hpp), compiled for the CPU with the sanitizer that ends
the program at an undefined division or shift: how many pieces a half window's records make."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "svdimager_amd", "csrc")

PROBE = r"""
#include "work_shape.hpp"
extern "C" {
void pieces(long n, const unsigned* records, const unsigned* cap, unsigned* count, unsigned* per) {
    for (long i = 0; i < n; ++i) {
        const svdi::Pieces p = svdi::dense_pieces(records[i], cap[i]);
        count[i] = p.count;
        per[i] = p.per;
    }
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("work_shape")
    src = d / "probe.cpp"
    src.write_text(PROBE)
    so = d / "probe.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fsanitize=integer-divide-by-zero,shift",
                    "-fsanitize-undefined-trap-on-error", "-I", CSRC, str(src), "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    u32 = np.ctypeslib.ndpointer(np.uint32, flags="C_CONTIGUOUS")
    L.pieces.argtypes = [ctypes.c_long, u32, u32, u32, u32]
    return L


def _pieces(lib, records, cap):
    records, cap = np.broadcast_arrays(np.asarray(records, np.uint32), np.asarray(cap, np.uint32))
    records, cap = np.ascontiguousarray(records), np.ascontiguousarray(cap)
    count, per = np.zeros_like(records), np.zeros_like(records)
    lib.pieces(records.size, records, cap, count, per)
    return count.astype(np.int64), per.astype(np.int64)


def test_no_records_make_no_pieces(lib):
    """Every half that is not dense asks with no records."""
    count, per = _pieces(lib, np.zeros(4), [32, 2048, 16384, 1 << 31])
    assert (count == 0).all() and (per == 0).all()


def test_pieces_cover_the_records(lib):
    rng = np.random.default_rng(3)
    records = np.concatenate([[1, 31, 32, 33, 16384, 16385, (1 << 31) - 2, (1 << 31) - 2],
                              np.exp(rng.uniform(0.0, np.log(2.0**31 - 2), 4000))]).astype(np.uint32)
    cap = np.concatenate([[2048, 2048, 2048, 2048, 16384, 16384, 2048, 1 << 31],
                          np.exp(rng.uniform(np.log(2048), np.log(2.0**31), 4000))]).astype(np.uint32)
    count, per = _pieces(lib, records, cap)
    records, cap = records.astype(np.int64), cap.astype(np.int64)
    assert (count >= 1).all() and (per % 32 == 0).all()
    assert (count * per >= records).all() and ((count - 1) * per < records).all()   # no empty piece
    assert (per < cap + 32).all()
    assert (count <= (records - 1) // cap + 1).all()
