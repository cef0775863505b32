"""The tile and K-split plan of the MFMA engine (csrc/tile_plan.hpp, host code)."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "tile_plan.hpp"
using namespace ohip;
extern "C" float plan(int kind, int P, int Q, int kc, int forced, int batch, int wide, int* out) {
  const TilePlan t = plan_tiles((PlanKind)kind, P, Q, kc, forced, batch, wide != 0);
  out[0] = t.splits;
  out[1] = t.tile;
  return t.us;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "p.cpp").write_text(SOURCE)
    so = str(d / "p.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "oxionnx_amd", "csrc"),
                    str(d / "p.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.plan.restype = ctypes.c_float

    def call(kind, p, q, kc, forced=0, batch=1, wide=0):
        out = (ctypes.c_int * 2)()
        us = lib.plan(kind, p, q, kc, forced, batch, wide, out)
        return out[0], out[1], us
    return call


def test_every_k_slice_has_stages(plan):
    r = random.Random(1)
    seen = 0
    for _ in range(20000):
        kind, p, q = r.randrange(3), r.randint(1, 4096), r.randint(1, 1200)
        nk = r.randint(2, 256)
        forced = r.choice([0, 0, 0, 10, 11])
        splits, _, _ = plan(kind, p, q, nk * 8 - r.randrange(8), forced, r.choice([1, 1, 4]), r.randrange(2))
        if splits > 1:
            seen += 1
            per = -(-nk // splits)   # what the kernel gives each slice
            assert (splits - 1) * per < nk, (kind, p, q, nk, forced, splits)
    assert seen > 1000


@pytest.mark.parametrize("kind,k,rate", [(0, 8, 2.5e9), (1, 4, 160e6), (2, 8, 2.5e9)], ids=["dense", "f32", "conv"])
def test_every_plan_has_an_estimate(plan, kind, k, rate):
    """No plan is faster than the matrix units (2.5 PFLOP/s in 16 bits, 160
    TFLOP/s in f32): callers compare estimates with those of other kernels."""
    r = random.Random(2)
    tiles = set()
    for _ in range(4000):
        p, q, kc = (int(2 ** r.uniform(5, top)) for top in (18, 13, 11))
        _, tile, us = plan(kind, p, q, kc)
        tiles.add(tile)
        assert us >= 2.0 * p * q * kc * k / rate, (p, q, kc, tile, us)
    assert 16 in tiles
