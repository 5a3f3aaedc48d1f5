// Bounded FP32 arithmetic of the voxelizer's solid angles (lbm3d_voxelize_blocks).
// Nothing here is the device's alone but the approximate square root and
// reciprocals, so a host compiler that is given those can check the bounds.
#pragma once

#include <cstdint>

namespace lbm3d_winding {

// how many blocks of side s cover n nodes (n >= 1; n + s may pass 2^31)
__host__ __device__ __forceinline__ int32_t blocks_of(int32_t n, int32_t s) { return (n - 1) / s + 1; }

// Corners.  With u = 2^-24: a triangle's corner c seen from a parent's centre is off by
// at most u (4 |c| + s0): v - hi, - lo, * inv and inv itself round once each (v - hi is
// exact where it is not much larger than lo), and s0 = 2^24 eta is the centre's own error.
// Seen from a child's centre at the offset o it rounds once more, and |c| <= |c - o| + |o|:
// u (5 |c - o| + 4 |o| + s0).
constexpr float kCornerRoundings = 5.f;
__host__ __device__ __forceinline__ float point_slack(float eta) { return 1.7e7f * eta; }  // s0
__host__ __device__ __forceinline__ float child_slack(float offset, float eta) {
  return 4.01f * offset + point_slack(eta);
}

// Error in cells of a block's centre as two FP32 and of its nodes in FP64, for grid
// coordinates up to far: 2^-49 of an axis for the second FP32, 4 roundings of 2^-53, and
// the square root of 3 axes.
__host__ __device__ __forceinline__ float point_error(double far, double dx) { return (float)(5e-15 * far / dx); }

// A triangle's corners from a point, in cells.
struct Corners {
  float ax, ay, az, bx, by, bz, cx, cy, cz;
  __device__ __forceinline__ Corners(const float *tris, int32_t t, const float3 hi, const float3 lo, float inv) {
    const float *v = tris + (int64_t)t * 9;
    ax = ((v[0] - hi.x) - lo.x) * inv, ay = ((v[1] - hi.y) - lo.y) * inv, az = ((v[2] - hi.z) - lo.z) * inv;
    bx = ((v[3] - hi.x) - lo.x) * inv, by = ((v[4] - hi.y) - lo.y) * inv, bz = ((v[5] - hi.z) - lo.z) * inv;
    cx = ((v[6] - hi.x) - lo.x) * inv, cy = ((v[7] - hi.y) - lo.y) * inv, cz = ((v[8] - hi.z) - lo.z) * inv;
  }
};

// The same with bounds on twice its area and on how far it reaches from its nearest corner
// (the longest edge over the square root of 3), and that corner's distance.  Of an edge of
// length m seen from the distance D the corners' errors leave u (8 D + 8 m + 2 s0) open, of
// twice the area u (16 D m + 21 m^2 + 4 s0 m).
struct Seen : Corners {
  float area2, edge, near;
  __device__ __forceinline__ Seen(const float *tris, int32_t t, const float3 hi, const float3 lo, float inv, float s0)
      : Corners(tris, t, hi, lo, inv) {
    const float ux = bx - ax, uy = by - ay, uz = bz - az, wx = cx - ax, wy = cy - ay, wz = cz - az;
    const float vx = cx - bx, vy = cy - by, vz = cz - bz;
    const float nx = uy * wz - uz * wy, ny = uz * wx - ux * wz, nz = ux * wy - uy * wx;
    const float u2 = ux * ux + uy * uy + uz * uz, w2 = wx * wx + wy * wy + wz * wz, v2 = vx * vx + vy * vy + vz * vz;
    // the lengths that Product::take forms too
    near = fminf(fminf(__builtin_amdgcn_sqrtf(ax * ax + ay * ay + az * az),
                       __builtin_amdgcn_sqrtf(bx * bx + by * by + bz * bz)),
                 __builtin_amdgcn_sqrtf(cx * cx + cy * cy + cz * cz));
    edge = 0.58f * __builtin_amdgcn_sqrtf(fmaxf(fmaxf(u2, w2), v2)) + (3e-7f * near + 7.5e-8f * s0);
    area2 = 1.02f * __builtin_amdgcn_sqrtf(nx * nx + ny * ny + nz * nz) + 1e-5f * (u2 + w2) +
            (1.7e-6f * near + 4.2e-7f * s0) * edge;
  }
};

// A bound from below on how far points within rho of the origin stay from a triangle:
// its nearest corner at lmin, off as above with `slack`.
__device__ __forceinline__ float clear_of(float lmin, float slack, float edge, float rho) {
  return lmin * 0.999f - 6e-8f * slack - edge - rho;
}

// a running product of den + i det with its turns, and the bound on its argument's error
struct Product {
  float zr = 1.f, zi = 0.f, err = 0.f;
  int turns = 0;

  // The factor of a triangle seen from the origin.  slack: how far its corners may be
  // off, in units of 2^-24, besides kCornerRoundings of their lengths; rho > 0: it
  // stands for all points within rho.
  __device__ __forceinline__ void take(float Ax, float Ay, float Az, float Bx, float By, float Bz, float Cx, float Cy,
                                       float Cz, float slack, float area2, float edge, float rho) {
    const float la = __builtin_amdgcn_sqrtf(Ax * Ax + Ay * Ay + Az * Az);
    const float lb = __builtin_amdgcn_sqrtf(Bx * Bx + By * By + Bz * Bz);
    const float lc = __builtin_amdgcn_sqrtf(Cx * Cx + Cy * Cy + Cz * Cz);
    const float det = Ax * (By * Cz - Bz * Cy) - Ay * (Bx * Cz - Bz * Cx) + Az * (Bx * Cy - By * Cx);
    const float L = la * lb * lc;
    const float den = L + (Ax * Bx + Ay * By + Az * Bz) * lc + (Bx * Cx + By * Cy + Bz * Cz) * la +
                      (Cx * Ax + Cy * Ay + Cz * Az) * lb;
    const float lmin = fminf(fminf(la, lb), lc);
    const float rz = __builtin_amdgcn_rsqf(det * det + den * den);
    // Rounding.  A corner is off by at most 2^-24 kappa of its length, kappa =
    // kCornerRoundings + slack / lmin; det then by 3 kappa and den by 12 kappa of 2^-24 L,
    // their own roundings add less than 74, and the angle is off by the sum over
    // |den + i det| (1.5 times for the arc).
    const float kappa = kCornerRoundings + slack * __builtin_amdgcn_rcpf(lmin);
    const float q = L * rz;  // at least 17^-1/2, unless something under- or overflowed
    float e = (1.6e-6f * kappa + 7e-6f) * q;
    // near the branch cut the sign of det, and with it a full turn, is open
    if (!(q > 0.2f && e < 0.2f) || (den < 0.f && fabsf(det) * rz <= e)) e = 1e30f;
    e += 1e-6f;  // the product's own rounding
    if (rho > 0.f) {
      const float gap = clear_of(lmin, slack, edge, rho);
      const float r = __builtin_amdgcn_rcpf(gap);
      e += gap > 0.05f ? 0.51f * rho * area2 * (r * r * r) : 1e30f;  // of Omega / 2
    }
    err += e;
    const float ur = den * rz, ui = det * rz;
    const float nr = zr * ur - zi * ui, ni = zr * ui + zi * ur;
    // past +-pi: both angles on one side of the real axis, their sum on the other
    turns += (zi >= 0.f && ui >= 0.f && ni < 0.f ? 1 : 0) - (zi < 0.f && ui < 0.f && ni >= 0.f ? 1 : 0);
    zr = nr;
    zi = ni + 0.f;  // no -0: atan2f would put it at -pi, where the test above has it at pi
  }
  __device__ __forceinline__ float angle() const { return atan2f(zi, zr) + 6.2831853f * (float)turns; }
  __device__ __forceinline__ float bound() const { return err + 5e-6f * (1.f + fabsf((float)turns)); }
};

}  // namespace lbm3d_winding
