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
extern "C" int skinny(int f32, int m, int n, int kc, int pack, int odd) {
  const TilePlan t = m <= kMaxGemvM ? TilePlan{1, 0} : plan_tiles(f32 ? PlanKind::DenseF32 : PlanKind::Dense, n, m, kc, 0);
  return skinny_wins(f32 != 0, m, n, kc, pack != 0, odd != 0, t);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "p.cpp").write_text(SOURCE)
    so = str(d / "p.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "oxionnx_amd", "csrc"),
                    str(d / "p.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.plan.restype = ctypes.c_float
    return lib


@pytest.fixture(scope="module")
def plan(lib):
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


# (type, rows, K, N): skinny kernel against GEMV / engine in us, both timed
FEW_ROWS = [("f16", 2, 768, 3072, 4.8, 5.2), ("f16", 2, 1024, 8192, 6.0, 7.2), ("f16", 16, 2048, 70001, 78.7, 85.5), ("f16", 8, 8192, 1100, 14.5, 16.4),
            ("f16", 23, 3787, 1658, 20.3, 13.0), ("f16", 23, 3788, 1658, 10.2, 13.0),
            ("f16", 16, 2046, 512, 7.1, 10.3), ("f16", 8, 5001, 512, 12.8, 9.9), ("f16", 8, 3787, 1658, 11.1, 18.7),
            ("f16", 8, 4096, 4096, 9.6, 30.2), ("f16", 9, 4096, 4096, 9.5, 11.7),
            ("f16", 32, 768, 768, 5.6, 8.1), ("f16", 24, 2048, 8192, 13.3, 11.7), ("f16", 32, 2048, 8192, 14.6, 12.4),
            ("f16", 24, 4096, 11008, 31.8, 22.3), ("f16", 32, 4096, 11008, 35.7, 22.7), ("f16", 24, 4096, 4096, 13.2, 12.3),
            ("f16", 32, 3072, 768, 11.4, 8.9), ("f16", 32, 2048, 70001, 114.8, 87.4), ("f16", 2, 2048, 70001, 55.7, 49.1),
            ("f32", 9, 4096, 11008, 44.8, 64.6), ("f32", 32, 1024, 8192, 16.7, 17.7), ("f32", 16, 4096, 4096, 20.7, 26.4), ("f32", 32, 768, 3072, 8.6, 11.2),
            ("f32", 24, 4096, 11008, 73.0, 65.9), ("f32", 32, 4096, 32000, 231.9, 152.0), ("f32", 32, 2048, 2048, 16.4, 13.3),
            ("f32", 2, 768, 30522, 25.7, 19.1), ("f32", 2, 1024, 50257, 45.3, 35.7), ("f32", 16, 2048, 70001, 172.0, 916.3)]


@pytest.mark.parametrize("case", FEW_ROWS, ids=lambda c: "%s-%dx%dx%d" % c[:4])
def test_few_rows_take_the_faster_kernel(lib, case):
    dt, m, k, n, skinny, other = case
    per = 4 if dt == "f32" else 8
    odd = dt == "f16" and k % 2   # rows at odd addresses
    assert bool(lib.skinny(int(dt == "f32"), m, n, -(-k // per), int(k % per != 0), odd)) == (skinny < other)


# (kind, elements a chunk, rows, K, N): us by K slices (1: the fastest tile unsplit)
SPLITS = [((1, 4, 128, 768, 3072), {1: 20.2, 2: 15.6, 3: 18.0, 4: 16.8, 5: 16.7, 6: 20.1, 8: 18.8}),
          ((1, 4, 128, 1024, 4096), {1: 25.3, 2: 19.4, 3: 22.4, 4: 21.5, 5: 24.4, 8: 23.1}),
          ((1, 4, 200, 2048, 768), {1: 46.6, 3: 21.8, 4: 18.3, 5: 16.7, 6: 19.5, 7: 20.1, 8: 18.5, 10: 17.9}),
          ((1, 4, 527, 2064, 662), {1: 49.0, 2: 30.0, 3: 32.2, 4: 28.0, 5: 25.2, 6: 29.8, 8: 29.2}),
          ((1, 4, 132, 2818, 766), {1: 68.0, 4: 26.2, 5: 23.4, 6: 21.7, 7: 20.9, 8: 23.0, 9: 24.6, 12: 23.4}),
          ((1, 4, 156, 6864, 1074), {1: 149.6, 5: 37.4, 8: 39.0, 9: 36.8, 10: 35.0, 12: 42.9}),
          ((1, 4, 256, 768, 3072), {1: 21.0, 2: 23.2, 3: 26.8, 4: 23.5, 5: 24.8}),
          ((0, 8, 128, 768, 3072), {1: 7.4, 2: 9.0, 3: 10.3, 4: 10.8}),
          ((0, 8, 148, 1331, 2336), {1: 12.9, 2: 12.8, 3: 14.0, 4: 14.7}),
          ((0, 8, 165, 768, 128), {1: 6.8, 2: 8.3, 3: 8.4, 4: 8.2}),   # (eager; by replay 7.1, 7.4, 6.9, 6.7)
          ((0, 8, 128, 8192, 4096), {1: 57.9, 3: 26.2, 4: 23.7, 5: 28.2, 8: 28.3}),
          ((0, 16, 300, 2048, 512), {1: 10.1, 2: 9.6, 3: 9.2, 4: 8.8, 5: 9.5, 6: 9.5, 8: 10.3}),
          ((0, 16, 206, 1931, 159), {1: 13.1, 2: 12.0, 3: 11.4, 4: 10.8, 5: 11.3, 6: 11.1, 8: 10.9, 12: 11.5})]


@pytest.mark.parametrize("shape,us", SPLITS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_k_slices_near_the_fastest_measured(plan, shape, us):
    kind, per, m, k, n = shape
    splits, _, _ = plan(kind, n, m, -(-k // per))
    assert splits in us and us[splits] <= 1.05 * min(us.values()), (splits, us)
