"""The MFMA gridder's work shape (csrc/work_shape.hpp), compiled for the CPU with the sanitizer that ends
the program at an undefined division or shift: how many pieces a half window's records make, and the shape
that fits a given number of partial slots."""
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
void shape(unsigned long samples, unsigned coop_min, unsigned coop_cap, unsigned* out) {
    const svdi::WorkShape s = svdi::work_shape(samples, coop_min, coop_cap);
    out[0] = s.coop_min;
    out[1] = s.coop_cap;
}
unsigned long most(unsigned coop_min, unsigned coop_cap, unsigned long records, unsigned long halves) {
    return svdi::most_pieces({coop_min, coop_cap}, records, halves);
}
void fit(long n, const unsigned* records, unsigned slots, unsigned* shape) {
    svdi::WorkShape s = {shape[0], shape[1]};
    unsigned words[svdi::kShapeWords] = {};
    for (long i = 0; i < n; ++i) {
        if (records[i] <= s.coop_min) continue;
        const int b = svdi::shape_bucket(s.coop_min, records[i]);
        if (!(svdi::shape_threshold(s.coop_min, b) < records[i] &&
              (b + 1 == svdi::kShapeBuckets || records[i] <= svdi::shape_threshold(s.coop_min, b + 1))))
            __builtin_trap();
        words[0] += 1;
        words[1] += records[i];
        words[2 + 2 * b] += 1;
        words[3 + 2 * b] += records[i];
    }
    svdi::fit_shape(words, slots, s);
    shape[0] = s.coop_min;
    shape[1] = s.coop_cap;
}
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
    L.shape.argtypes = [ctypes.c_ulong, ctypes.c_uint, ctypes.c_uint, u32]
    L.most.argtypes = [ctypes.c_uint, ctypes.c_uint, ctypes.c_ulong, ctypes.c_ulong]
    L.most.restype = ctypes.c_ulong
    L.fit.argtypes = [ctypes.c_long, u32, ctypes.c_uint, u32]
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


def _fit(lib, sizes, shape, slots):
    out = np.array(shape, np.uint32)
    lib.fit(len(sizes), np.ascontiguousarray(sizes, np.uint32), slots, out)
    return int(out[0]), int(out[1])


def _made(sizes, shape):
    dense = sizes[sizes > shape[0]]
    return int(((dense - 1) // shape[1] + 1).sum())


def test_the_shape_asked_for_is_the_shape_that_runs(lib):
    """A caller's numbers stand, whatever the slots of the worst case would take, and so do the defaults by the
    number of samples (16.7 M samples at 4096^2, of either term count, and 33 M: 1024 / 16384)."""
    def shape(samples, cmin=0, cap=0):
        out = np.zeros(2, np.uint32)
        lib.shape(samples, cmin, cap, out)
        return tuple(int(v) for v in out)
    assert shape(16_744_448) == shape(33_488_896) == (1024, 16384)
    assert shape(32_256) == (256, 2048) and shape(2_097_152) == (512, 4096)
    for tuned in ((32, 4096), (65536, 1 << 24), (300, 0), (0, 5000)):
        got = shape(33_488_896, *tuned)
        assert all(g == t for g, t in zip(got, tuned) if t != 0)
    # 1117 dense halves of 9.6 M records, as in the SKA-Low snapshot: enough slots for what it makes are enough.
    rng = np.random.default_rng(1)
    sizes = np.exp(rng.uniform(np.log(1025), np.log(200_000), 1117)).astype(np.int64)
    assert _fit(lib, sizes, (1024, 16384), 5912) == (1024, 16384)


@pytest.mark.parametrize("slots", [0, 1, 7, 40, 400, 4000])
@pytest.mark.parametrize("spread", [2.0, 5.0, 9.0])
def test_pieces_fit_the_slots(lib, slots, spread):
    """Where they do not, the least coarser shape that does: pieces that take what the halves leave, at least half the
    slots, then a threshold higher by quarters of an octave, under which only smaller halves are left out."""
    rng = np.random.default_rng([slots, int(spread)])
    for cmin, cap in ((32, 4096), (256, 2048), (1024, 16384)):
        sizes = np.minimum(np.exp(rng.normal(np.log(4.0 * cmin), spread / 2, 3000)), 6e5).astype(np.int64)
        m, c = _fit(lib, sizes, (cmin, cap), slots)
        dense = sizes[sizes > cmin]
        if len(dense) + dense.sum() // cap <= slots:
            assert (m, c) == (cmin, cap)
        assert _made(sizes, (m, c)) <= slots
        cuts = max(slots - len(dense), slots // 2)
        assert c >= cap and (cuts == 0 or dense.sum() // c <= cuts)
        assert c == cap or cuts == 0 or dense.sum() // (c - 1) >= cuts
        if len(dense) < slots // 2:
            assert m == cmin
        if m > cmin:                                       # a quarter of an octave lower would not have fitted
            lower = max(cmin, int(m / 1.26) - 1) if m < 0xffffffff else int(sizes.max()) - 1
            left = sizes[sizes > lower]
            assert len(left) + left.sum() // c > slots


def test_worst_case_bounds_any_sizes(lib):
    rng = np.random.default_rng(9)
    for _ in range(200):
        halves = int(rng.integers(1, 5000))
        sizes = np.exp(rng.normal(rng.uniform(2, 9), rng.uniform(0, 3), halves)).astype(np.int64) + 1
        cmin, cap = int(rng.integers(32, 3000)), int(rng.integers(2048, 30000))
        records = int(sizes.sum()) + int(rng.integers(0, 1000))
        assert _made(sizes, (cmin, cap)) <= lib.most(cmin, cap, records, halves)
