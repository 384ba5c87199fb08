"""The host half of a readback (mpm_host.h), compiled alone: a status other than
OK leaves the world as it was, whichever piece it comes with."""

import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include "mpm_host.h"
using Column = std::vector<double>;
struct World {
  Column pos, vel, F, C, force, plastic;
  std::vector<uint8_t> enabled, fixed;
  std::vector<int> material;
};
// columns of `state`: 3 pos, 3 vel, 9 F, 9 C, 3 force, 3 plastic per particle, one column after the other
extern "C" int readback(double* state, const uint8_t* enabled, const uint8_t* fixed, const int* material,
                        const float* records, uint64_t n, uint64_t per, int plastic, int fail_at, int twice) {
  World w;
  double* at = state;
  auto take = [&](Column& c, size_t k) { c.assign(at, at + k * n); at += k * n; };
  take(w.pos, 3); take(w.vel, 3); take(w.F, 9); take(w.C, 9); take(w.force, 3); take(w.plastic, 3);
  w.enabled.assign(enabled, enabled + n);
  w.fixed.assign(fixed, fixed + n);
  w.material.assign(material, material + n);
  tmpm::StateColumns<Column> spare;
  int st = 0;
  for (int r = 0; r <= twice; ++r)
    st = tmpm::read_pieces(w, spare, n, per, plastic != 0, [](int m) { return m != 0; },
                           [&](size_t k, const float*& rec) {
                             rec = records ? records + tmpm::kRecordFloats * k * per : nullptr;
                             return (int)k == fail_at ? 7 : 0;
                           });
  at = state;
  auto put = [&](const Column& c) { at = std::copy(c.begin(), c.end(), at); };
  put(w.pos); put(w.vel); put(w.F); put(w.C); put(w.force); put(w.plastic);
  return st;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("readback")
    (d / "r.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-pthread", "-I",
                    str(ROOT / "tessera_amd" / "csrc"), str(d / "r.cpp"), "-o", str(d / "r.so")], check=True)
    return C.CDLL(str(d / "r.so"))


def call(lib, state, enabled, fixed, material, records, per, plastic, fail_at=-1, twice=0):
    out = state.copy()
    ptr = lambda a, t: None if a is None else a.ctypes.data_as(C.POINTER(t))
    st = lib.readback(ptr(out, C.c_double), ptr(enabled, C.c_uint8), ptr(fixed, C.c_uint8), ptr(material, C.c_int),
                      ptr(records, C.c_float), C.c_uint64(len(enabled)), C.c_uint64(per), int(plastic), fail_at, twice)
    return st, out


def case(n):
    rng = np.random.default_rng(n)
    return (rng.normal(size=30 * n), (rng.random(n) < 0.8).astype(np.uint8), (rng.random(n) < 0.2).astype(np.uint8),
            (rng.random(n) < 0.5).astype(np.int32), rng.normal(size=29 * n).astype(np.float32))


def expected(state, enabled, fixed, material, records, plastic):
    n = len(enabled)
    ends = np.cumsum([3, 3, 9, 9, 3, 3])[:-1] * n
    pos, vel, F, Cm, force, pl = (c.reshape(n, -1) for c in np.split(state.copy(), ends))
    force[:] = 0.0
    on, still = enabled.astype(bool), fixed.astype(bool)
    vel[on & still] = 0.0
    Cm[on & still] = 0.0
    if records is not None:
        rec, moved = records.reshape(n, 29).astype(np.float64), on & ~still
        for col, lo, hi in ((pos, 0, 3), (vel, 4, 7), (Cm, 8, 17), (F, 17, 26)):
            col[moved] = rec[moved, lo:hi]
        if plastic:
            moved &= material != 0
            pl[moved] = rec[moved, 26:29]
    return np.concatenate([c.ravel() for c in (pos, vel, F, Cm, force, pl)])


@pytest.mark.parametrize("plastic", [False, True])
@pytest.mark.parametrize("n,per", [(1, 1), (7, 7), (7, 3), (8, 4), (40000, 40000), (40000, 17000)])
def test_records_become_the_world(lib, n, per, plastic):
    state, *flags, records = case(n)
    want = expected(state, *flags, records, plastic)
    for twice in (0, 1):  # the second readback writes the columns that the first one left spare
        st, got = call(lib, state, *flags, records, per, plastic, twice=twice)
        assert st == 0 and np.array_equal(got, want)
    st, got = call(lib, state, *flags, None, per, plastic)
    assert st == 0 and np.array_equal(got, expected(state, *flags, None, plastic))


@pytest.mark.parametrize("plastic", [False, True])
@pytest.mark.parametrize("n,per,pieces", [(7, 7, 1), (7, 3, 3), (40000, 17000, 3)])
def test_a_failed_piece_leaves_the_world_as_it_was(lib, n, per, pieces, plastic):
    state, *flags, records = case(n)
    for k in range(pieces):
        st, got = call(lib, state, *flags, records, per, plastic, fail_at=k)
        assert st == 7 and np.array_equal(got, state)
