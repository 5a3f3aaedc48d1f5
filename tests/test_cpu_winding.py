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
  for (int i = 0; i < n; ++i, t += 9)
    p.take(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], slack, 0.f, 0.f, 0.f);
  out[0] = p.angle();
  out[1] = p.bound();
}
// a triangle seen from the point hi + lo of p: 9 corners, area2, edge, near; then its
// corners from the offset o, the bound on a corner's error at length 0 and per length
void seen(const float *t, const double *p, double dx, float eta, float o, float *out) {
  const float3 hi{(float)p[0], (float)p[1], (float)p[2]};
  const float3 lo{(float)(p[0] - (double)hi.x), (float)(p[1] - (double)hi.y), (float)(p[2] - (double)hi.z)};
  const Seen s(t, 0, hi, lo, (float)(1.0 / dx), point_slack(eta));
  const float f[12] = {s.ax, s.ay, s.az, s.bx, s.by, s.bz, s.cx, s.cy, s.cz, s.area2, s.edge, s.near};
  for (int k = 0; k < 12; ++k) out[k] = f[k];
  for (int k = 0; k < 9; ++k) out[12 + k] = f[k] - o;
  out[21] = child_slack(1.7320509f * o, eta);
  out[22] = kCornerRoundings;
}
int blocks(int n, int s) { return blocks_of(n, s); }
float error_of_point(double far, double dx) { return point_error(far, dx); }
float clear(float lmin, float slack, float edge, float rho) { return clear_of(lmin, slack, edge, rho); }
}
"""


@pytest.fixture(scope="module")
def winding(tmp_path_factory):
    d = tmp_path_factory.mktemp("winding")
    src, so = d / "driver.cpp", d / "driver.so"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-o", str(so),
                    str(src)], check=True, capture_output=True, text=True)
    lib = ctypes.CDLL(str(so))
    lib.error_of_point.restype = lib.clear.restype = ctypes.c_float
    return lib


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


def triangles(rng, n, dx, p):
    """Triangles of many shapes around p: general, small and far, slivers."""
    size = np.exp(rng.uniform(-7, 4, (n, 1, 1))) * dx
    t = rng.normal(size=(n, 3, 3)) * size
    thin = rng.random(n) < 0.4
    t[thin, 2] = t[thin, 0] + rng.random((thin.sum(), 1)) * (t[thin, 1] - t[thin, 0]) + 1e-2 * (t[thin, 2] - t[thin, 0])
    return (t + rng.normal(size=(n, 1, 3)) * np.exp(rng.uniform(-2, 6, (n, 1, 1))) * dx + p).astype(np.float32)


@pytest.mark.parametrize("dx", [1.0, 0.3, 7e-4])
@pytest.mark.parametrize("offset", [0.5, 2.0])
@pytest.mark.parametrize("origin", [0.0, 20.0, 1e6])
def test_corners_areas_and_reaches_within_their_bounds(winding, dx, offset, origin):
    rng = np.random.default_rng(5)
    wide = lambda a: np.asarray(a, np.longdouble)
    length = lambda v: np.sqrt((v * v).sum(-1))
    out = np.zeros(23, np.float32)
    for t in triangles(rng, 3000, dx, origin * dx):
        p = (origin + rng.uniform(-1, 1, 3) * rng.choice([1.0, 30.0])) * dx  # a block's centre
        far = np.abs(p).max()
        eta = winding.error_of_point(ctypes.c_double(far), ctypes.c_double(dx))
        winding.seen(t.ctypes.data_as(ctypes.c_void_p), p.ctypes.data_as(ctypes.c_void_p), ctypes.c_double(dx),
                     ctypes.c_float(eta), ctypes.c_float(offset), out.ctypes.data_as(ctypes.c_void_p))
        exact = (wide(t) - wide(p)) / wide(dx)
        child = exact - offset
        err = length(wide(out[12:21].reshape(3, 3)) - child)
        assert (err <= 2.0 ** -24 * (out[22] * length(child) + out[21]) * (1 + 1e-5)).all()
        u, w = exact[1] - exact[0], exact[2] - exact[0]
        assert out[9] >= length(np.cross(u, w))
        longest = max(length(u), length(w), length(u - w))
        assert out[10] >= longest / math.sqrt(3)
        lmin = length(out[12:21].reshape(3, 3)).min()
        gap = winding.clear(*(ctypes.c_float(float(v)) for v in (lmin, out[21], out[10], 0.0)))
        assert gap <= length(child).min() - longest / math.sqrt(3) + 1e-6


def test_a_point_far_from_the_origin_is_off_by_no_more_than_stated(winding):
    """Coordinates whose second FP32 rounds as much as it can, on all three axes."""
    rng = np.random.default_rng(2)
    for far in (1e3, 2.0 ** 20, 3e7):
        worst = 0.0
        for _ in range(20000):
            p = far * (1 + rng.random(3) * 2.0 ** -10)
            hi = p.astype(np.float32)
            lo = (p - hi.astype(np.float64)).astype(np.float32)
            off = p.astype(np.longdouble) - hi.astype(np.longdouble) - lo.astype(np.longdouble)
            worst = max(worst, float(np.sqrt((off * off).sum())))
        roundings = 4 * 2.0 ** -53 * math.sqrt(3) * far
        bound = winding.error_of_point(ctypes.c_double(far * (1 + 2.0 ** -10)), ctypes.c_double(1.0))
        assert worst + roundings <= bound


def test_blocks_cover_every_extent_up_to_the_largest(winding):
    for n in (1, 2, 7, 8, 9, 1000, 2 ** 31 - 8, 2 ** 31 - 1):
        for s in (2, 4, 8):
            assert winding.blocks(n, s) == -(-n // s)
