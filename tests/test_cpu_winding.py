"""The voxelizer's bounded FP32 solid angles (taichi_lbm3d_amd/csrc/winding.h), compiled for
the host and compared with wide arithmetic: every sum lies within the bound it states.
The device's approximate square root and reciprocals are taken exact, and one place off."""
import ctypes
import itertools
import math
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "taichi_lbm3d_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

DRIVER = r"""
#include <cmath>
#include <cstdint>
#define __device__
#define __host__
#define __forceinline__ inline
struct float3 { float x, y, z; };
static int ulps = 0;  // places every approximate function is off
static float off(float v) {
  for (int k = 0; k < std::abs(ulps); ++k) v = std::nextafter(v, ulps > 0 ? INFINITY : -INFINITY);
  return v;
}
static inline float __builtin_amdgcn_sqrtf(float v) { return v > 0.f ? off(std::sqrt(v)) : std::sqrt(v); }
static inline float __builtin_amdgcn_rsqf(float v) { return off((float)(1.0 / std::sqrt((double)v))); }
static inline float __builtin_amdgcn_rcpf(float v) { return off(1.f / v); }
#include "winding.h"
using namespace lbm3d_winding;
extern "C" {
void set_ulps(int n) { ulps = n; }
// the product of n triangles (corners from the point, in cells): argument and its bound
void product(const float *t, int n, float slack, float *out) {
  Product p;
  for (int i = 0; i < n; ++i, t += 9) p.take(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], slack, 0.f, 0.f, 0.f);
  out[0] = p.angle();
  out[1] = p.bound();
}
}
"""


@pytest.fixture(scope="module")
def winding(tmp_path_factory):
    d = tmp_path_factory.mktemp("winding")
    src, so = d / "driver.cpp", d / "driver.so"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-o", str(so),
                    str(src)], check=True, capture_output=True, text=True)
    return ctypes.CDLL(str(so))


def product(lib, corners, slack=0.0):
    t = np.ascontiguousarray(corners, np.float32).reshape(-1, 9)
    out = (ctypes.c_float * 2)()
    lib.product(t.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), len(t), ctypes.c_float(slack), out)
    return out[0], out[1]


def half_angles(corners):
    """Omega / 2 of every triangle seen from the origin, in 80 bits."""
    a, b, c = (np.asarray(corners, np.longdouble).reshape(-1, 3, 3)[:, k] for k in range(3))
    la, lb, lc = (np.sqrt((v * v).sum(1)) for v in (a, b, c))
    det = (a * np.cross(b, c)).sum(1)
    den = la * lb * lc + (a * b).sum(1) * lc + (b * c).sum(1) * la + (c * a).sum(1) * lb
    return np.arctan2(det, den)


def right_angles():
    """Triangles of whole coordinates and lengths whose den is exactly 0: half angles of exactly -pi/2 and pi/2."""
    sized = [(v, math.isqrt(sum(x * x for x in v))) for v in itertools.product(range(-4, 5), repeat=3)]
    sized = [np.array(v) for v, n in sized if n and n * n == sum(x * x for x in v)]
    for a, b, c in itertools.product(sized[::5], sized[::3], sized[::2]):
        la, lb, lc = (math.isqrt(int(v @ v)) for v in (a, b, c))
        if la * lb * lc + a @ b * lc + b @ c * la + c @ a * lb == 0 and a @ np.cross(b, c):
            yield np.array([a, b, c], float)


def test_two_exact_right_angles_make_one_half_turn(winding):
    """(0 - i)(0 - i) = -1 - 0 i: a negative zero must not count as a turn and as -pi too."""
    tris = list(right_angles())
    assert len(tris) > 100
    both = {s: [t for t in tris if half_angles(t)[0] * s > 0] for s in (1, -1)}
    for s, ts in both.items():
        for t, u in zip(ts, reversed(ts)):
            got, bound = product(winding, [t, u])
            assert bound < 0.1 and abs(got - s * math.pi) <= bound, (t, u, got)


@pytest.mark.parametrize("ulps", [-1, 0, 1])
def test_products_stay_within_their_bound(winding, ulps):
    """Many factors, general ones and exact right angles, in every order of signs."""
    winding.set_ulps(ulps)
    rng = np.random.default_rng(11)
    exact = list(right_angles())
    settled = 0
    for n in (1, 2, 3, 10, 100):
        for _ in range(300):
            tris = rng.normal(size=(n, 3, 3)) * np.exp(rng.uniform(-3, 6, (n, 1, 1)))
            for k in range(n):
                if rng.random() < 0.4:
                    tris[k] = exact[rng.integers(len(exact))]
                elif rng.random() < 0.5:  # small and far
                    tris[k] = rng.normal(size=3) * 30 + rng.normal(size=(3, 3)) * 0.5
            tris = tris.astype(np.float32)
            got, bound = product(winding, tris)
            if bound < 1e29:
                settled += 1
                assert abs(float(half_angles(tris).sum()) - got) <= bound
    winding.set_ulps(0)
    assert settled > 500
