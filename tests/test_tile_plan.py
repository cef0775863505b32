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
extern "C" void plan(int kind, int P, int Q, int kc, int forced, int batch, int wide, int* out) {
  const TilePlan t = plan_tiles((PlanKind)kind, P, Q, kc, forced, batch, wide != 0);
  out[0] = t.splits;
  out[1] = t.tile;
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

    def call(kind, p, q, kc, forced=0, batch=1, wide=0):
        out = (ctypes.c_int * 2)()
        lib.plan(kind, p, q, kc, forced, batch, wide, out)
        return out[0], out[1]
    return call


def test_every_k_slice_has_stages(plan):
    r = random.Random(1)
    seen = 0
    for _ in range(20000):
        kind, p, q = r.randrange(3), r.randint(1, 4096), r.randint(1, 1200)
        nk = r.randint(2, 256)
        forced = r.choice([0, 0, 0, 10, 11])
        splits, _ = plan(kind, p, q, nk * 8 - r.randrange(8), forced, r.choice([1, 1, 4]), r.randrange(2))
        if splits > 1:
            seen += 1
            per = -(-nk // splits)   # what the kernel gives each slice
            assert (splits - 1) * per < nk, (kind, p, q, nk, forced, splits)
    assert seen > 1000
