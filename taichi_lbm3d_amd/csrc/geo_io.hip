// Geometry input: the init_geo ASCII reader and an STL voxelizer.  The C ABI is
// declared in include/lbm3d_io.h.
//
// lbm3d_read_geo_ascii parses the reference's voxel file (one number per line,
// x fastest, SP:173-177) on the host with a hand-written number scanner
// (geo_ascii.h, plain C++ shared with the sanitizer build).
//
// lbm3d_voxelize flags grid nodes inside a closed triangle mesh, the job of the
// reference's Convert_stl_to_binary.cpp:29-157 (libigl's signed distance with
// the fast winding number sign).  Here every node sums the exact generalized
// winding number of all triangles, w(p) = 1/(4 pi) sum_t Omega_t(p), with the
// solid angle of Van Oosterom and Strackee,
//   tan(Omega/2) = a.(b x c) / (|a||b||c| + (a.b)|c| + (b.c)|a| + (c.a)|b|),
// a, b, c the triangle's corners relative to p, in FP64; the node is solid when
// w >= 1/2.  k_winding does that for every node, one thread each, triangles
// staged through LDS in tiles.  lbm3d_voxelize_blocks gives the same flags from
// far fewer sums: away from the surface whole blocks of nodes share a flag, and a
// bounded FP32 sum settles nearly every node of the others.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cerrno>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "geo_ascii.h"
#include "lbm3d.h"
#include "lbm3d_io.h"
#include "winding.h"

namespace {

using lbm3d_winding::blocks_of;
using lbm3d_winding::child_slack;
using lbm3d_winding::point_error;
using lbm3d_winding::point_slack;
using lbm3d_winding::Product;
using lbm3d_winding::Seen;

thread_local char io_err[512] = "";

int iofail(int code, const char *msg, const char *what = "") {
  snprintf(io_err, sizeof(io_err), "%s%s", msg, what);
  return code;
}

constexpr int kTriTile = 256;

// twice the FP64 angle of one triangle's solid angle at (px, py, pz)
__device__ __forceinline__ double triangle_angle(const float *v, double px, double py, double pz) {
  const double ax = v[0] - px, ay = v[1] - py, az = v[2] - pz;
  const double bx = v[3] - px, by = v[4] - py, bz = v[5] - pz;
  const double cx = v[6] - px, cy = v[7] - py, cz = v[8] - pz;
  const double la = sqrt(ax * ax + ay * ay + az * az);
  const double lb = sqrt(bx * bx + by * by + bz * bz);
  const double lc = sqrt(cx * cx + cy * cy + cz * cz);
  const double det = ax * (by * cz - bz * cy) - ay * (bx * cz - bz * cx) + az * (bx * cy - by * cx);
  const double den = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + (bx * cx + by * cy + bz * cz) * la +
                     (cx * ax + cy * ay + cz * az) * lb;
  return 2.0 * atan2(det, den);
}

__device__ __forceinline__ int8_t winding_flag(double omega) {
  const double w = omega / (4.0 * M_PI);
  return w >= 0.5 ? 1 : 0;
}

__global__ void __launch_bounds__(256)
    k_winding(const float *__restrict__ tris, int32_t n_tris, double x0, double y0, double z0, double dx, int32_t nx,
              int32_t ny, int32_t nz, int8_t *__restrict__ solid) {
  __shared__ float s_tri[kTriTile * 9];
  const int64_t n = (int64_t)nx * ny * nz;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double px = 0, py = 0, pz = 0;
  if (id < n) {
    const int64_t k = id % nz, t = id / nz;
    const int64_t j = t % ny, i = t / ny;
    px = x0 + dx * (double)i;
    py = y0 + dx * (double)j;
    pz = z0 + dx * (double)k;
  }
  double omega = 0.0;
  for (int32_t base = 0; base < n_tris; base += kTriTile) {
    const int cnt = n_tris - base < kTriTile ? n_tris - base : kTriTile;
    __syncthreads();
    for (int e = threadIdx.x; e < cnt * 9; e += blockDim.x) s_tri[e] = tris[(int64_t)base * 9 + e];
    __syncthreads();
    if (id < n) {
      for (int t = 0; t < cnt; ++t) omega += triangle_angle(s_tri + 9 * t, px, py, pz);
    }
  }
  if (id < n) solid[id] = winding_flag(omega);
}

// ---------------------------------------------------------------------------
// The same flags block by block.  The solid angle Omega of the mesh changes by at
// most rho * sum_t 2 A_t / (d_t - rho)^3 within rho of a point (A_t a triangle's
// area, d_t its distance; the field of a surface element falls off as 1/r^2), so
// if Omega at a block's centre is further from the threshold 2 pi than that and
// than the error of the sum, all of the block's nodes have one flag.  Blocks of 4
// nodes a side are tried first, 2 a side where those are undecided, then single
// nodes, whose sum needs no such bound; a node that the error bound leaves open
// (on the surface, in the plane of a triangle next to it) gets the FP64 sum in
// triangle order, bit for bit k_winding's.
//
// Omega / 2 is the argument of prod_t (den_t + i det_t): a wave takes a parent
// block, its lanes the triangles in turn, and each lane keeps running products,
// normalised, with the turns they have made.  A triangle further than kFar times the
// parent's reach R (centre to outermost node) is taken once, at the parent's centre,
// for all 8 children, which adds R * 2 A / (d - R)^3 to the bound; the others once per
// child, as soon as there are 64 of them.  Over a plane the far ones add about
// 2 pi / (kFar - 1), of the distance pi that Omega / 2 has from the threshold on either
// side of a closed surface; a smaller kFar leaves more nodes open where surfaces meet.
// Lengths are in cells, relative to the parent's centre.
// Bound by FP32 arithmetic.  7,680 triangles on 96 x 104 x 88 nodes: every node in FP64
// 33.2 ms; every triangle for every child 3.2 ms; kFar 10.5 to 12 1.65 ms, 9 1.87 ms
// and 16 1.74 ms.  With corners from FP64 differences and near triangles as they come
// kFar 12 took 2.02 ms, 6 8.3 ms.  Loading the next triangle ahead changed nothing.
// ---------------------------------------------------------------------------
constexpr float kFar = 11.f;

struct VoxGrid {
  double x0, y0, z0, dx;
  int32_t nx, ny, nz;
  int32_t n_tris;
  float eta;  // point_error
};

// The children of side S of the parents (side 2S) in `list` (all parents if it is
// null): flags of the decided ones, the others' block indices to `next`.
template <int S>
__global__ void __launch_bounds__(256)
    k_winding_blocks(const float *__restrict__ tris, const VoxGrid gr, const int32_t *__restrict__ list,
                     const int32_t *__restrict__ count, int32_t all, int32_t *__restrict__ next,
                     int32_t *__restrict__ next_count, int8_t *__restrict__ solid) {
  // near triangles wait here until there is one for every lane (up to 63 + 64 of them)
  __shared__ int32_t queue[4][128];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t waves = (int32_t)(gridDim.x * 4);
  const int32_t n = list ? *count : all;
  const int32_t pny = blocks_of(gr.ny, 2 * S), pnz = blocks_of(gr.nz, 2 * S);
  const int32_t cnx = blocks_of(gr.nx, S), cny = blocks_of(gr.ny, S), cnz = blocks_of(gr.nz, S);
  const float inv = (float)(1.0 / gr.dx);
  for (int64_t it = blockIdx.x * 4 + (threadIdx.x >> 6); it < n; it += waves) {  // n may be near 2^31
    const int32_t id = __builtin_amdgcn_readfirstlane(list ? list[it] : (int32_t)it);
    const int32_t bk = id % pnz, bt = id / pnz, bj = bt % pny, bi = bt / pny;
    // the parent's reference point, and its children's centres relative to it, in cells
    const double pi = 2 * S * bi + S - 0.5, pj = 2 * S * bj + S - 0.5, pk = 2 * S * bk + S - 0.5;
    const double px = gr.x0 + gr.dx * pi, py = gr.y0 + gr.dx * pj, pz = gr.z0 + gr.dx * pk;
    const float3 hi = make_float3((float)px, (float)py, (float)pz);
    const float3 lo = make_float3((float)(px - (double)hi.x), (float)(py - (double)hi.y), (float)(pz - (double)hi.z));
    Product child[8], all8;
    constexpr float off = 0.5f * S;                    // a child's centre, per axis
    constexpr float rho = 0.866026f * (S - 1);         // its half diagonal
    constexpr float R = 1.7320509f * off + rho;        // the parent's, from its centre
    const float slack = point_slack(gr.eta), near_slack = child_slack(1.7320509f * off, gr.eta);
    // the children's factors of the first `n` triangles from queue[wave][from]
    const auto near = [&](int from, int n) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (lane < n) {
        const Seen s(tris, queue[wave][from + lane], hi, lo, inv, slack);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const float ox = c & 4 ? off : -off, oy = c & 2 ? off : -off, oz = c & 1 ? off : -off;
          child[c].take(s.ax - ox, s.ay - oy, s.az - oz, s.bx - ox, s.by - oy, s.bz - oz, s.cx - ox, s.cy - oy,
                        s.cz - oz, near_slack, s.area2, s.edge, rho);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    int queued = 0;  // uniform in the wave
    for (int32_t base = 0; base < gr.n_tris; base += 64) {
      const int32_t t = base + lane;
      bool close = false;
      if (t < gr.n_tris) {
        const Seen s(tris, t, hi, lo, inv, slack);
        const float far = kFar * R + s.edge;
        close = !(s.near2 > far * far);  // NaN too
        if (!close) all8.take(s.ax, s.ay, s.az, s.bx, s.by, s.bz, s.cx, s.cy, s.cz, slack, s.area2, s.edge, R);
      }
      const uint64_t m = __ballot(close);
      if (close)
        queue[wave][queued + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = t;
      queued += __popcll(m);
      if (queued >= 64) {
        queued -= 64;
        near(queued, 64);
      }
    }
    if (queued > 0) near(0, queued);
    const float half8 = all8.angle(), err8 = all8.bound();
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      float half = child[c].angle() + half8, e = child[c].bound() + err8 + 1e-6f * (fabsf(half8) + 1.f);
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) {
        half += __shfl_xor(half, d);
        e += __shfl_xor(e, d);
      }
      const int32_t ci = 2 * bi + (c >> 2 & 1), cj = 2 * bj + (c >> 1 & 1), ck = 2 * bk + (c & 1);
      if (ci >= cnx || cj >= cny || ck >= cnz) continue;  // uniform in the wave
      // Omega >= 2 pi, Omega / 2 >= pi; rounding of the wave's sum included
      const bool in = half >= 3.14159265f;
      if (fabsf(half - 3.14159265f) > 1.01f * e + 1e-4f) {  // false for NaN
        for (int q = lane; q < S * S * S; q += 64) {
          const int i = S * ci + q / (S * S), j = S * cj + q / S % S, k = S * ck + q % S;
          if (i < gr.nx && j < gr.ny && k < gr.nz) solid[((int64_t)i * gr.ny + j) * gr.nz + k] = in ? 1 : 0;
        }
      } else if (lane == 0) {
        next[atomicAdd(next_count, 1)] = (ci * cny + cj) * cnz + ck;
      }
    }
  }
}

// Nodes left open: one wave per node, the lanes' angles added in triangle order.
__global__ void __launch_bounds__(256)
    k_winding_nodes(const float *__restrict__ tris, const VoxGrid gr, const int32_t *__restrict__ list,
                    const int32_t *__restrict__ count, int8_t *__restrict__ solid) {
  const int lane = threadIdx.x & 63;
  const int32_t n = *count, waves = (int32_t)(gridDim.x * 4);
  for (int64_t it = blockIdx.x * 4 + (threadIdx.x >> 6); it < n; it += waves) {  // n may be near 2^31
    const int32_t id = __builtin_amdgcn_readfirstlane(list[it]);
    const int32_t k = id % gr.nz, t0 = id / gr.nz, j = t0 % gr.ny, i = t0 / gr.ny;
    const double px = gr.x0 + gr.dx * (double)i, py = gr.y0 + gr.dx * (double)j, pz = gr.z0 + gr.dx * (double)k;
    double omega = 0.0;
    for (int32_t base = 0; base < gr.n_tris; base += 64) {
      const int32_t t = base + lane;
      const double term = t < gr.n_tris ? triangle_angle(tris + (int64_t)t * 9, px, py, pz) : 0.0;
      const int cnt = gr.n_tris - base < 64 ? gr.n_tris - base : 64;
      for (int q = 0; q < cnt; ++q) omega += __shfl(term, q);
    }
    if (lane == 0) solid[id] = winding_flag(omega);
  }
}

__global__ void k_clear_counts(int32_t *counts) {
  if (threadIdx.x < 4) counts[threadIdx.x] = 0;
}

// list places of a workspace, in int32: 4 counts, then the undecided blocks of 4,
// of 2 and the open nodes
int64_t vox_list(int32_t nx, int32_t ny, int32_t nz, int level) {
  int64_t at = 64;
  if (level > 0) at += (int64_t)blocks_of(nx, 4) * blocks_of(ny, 4) * blocks_of(nz, 4);
  if (level > 1) at += (int64_t)blocks_of(nx, 2) * blocks_of(ny, 2) * blocks_of(nz, 2);
  if (level > 2) at += (int64_t)nx * ny * nz;
  return at;
}

}  // namespace

extern "C" {

const char *lbm3d_io_last_error(void) { return io_err; }

int64_t lbm3d_read_geo_ascii(const char *path, int32_t nx, int32_t ny, int32_t nz, int8_t *solid) {
  return lbm3d_ascii::read_geo(path, nx, ny, nz, solid, io_err, sizeof(io_err));
}

size_t lbm3d_voxelize_workspace_bytes(int32_t nx, int32_t ny, int32_t nz) {
  if (nx < 1 || ny < 1 || nz < 1) return 0;
  return (size_t)vox_list(nx, ny, nz, 3) * sizeof(int32_t);
}

int lbm3d_voxelize_blocks(void *stream, const float *tris, int32_t n_tris, double x0, double y0, double z0, double dx,
                          int32_t nx, int32_t ny, int32_t nz, int8_t *solid, void *workspace,
                          size_t workspace_bytes) {
  if (nx < 1 || ny < 1 || nz < 1 || n_tris < 0 || !(dx > 0)) return iofail(LBM3D_EINVAL, "bad grid or mesh size");
  if ((n_tris > 0 && !tris) || !solid || !workspace) return iofail(LBM3D_EINVAL, "NULL mesh, output or workspace");
  if ((int64_t)nx * ny * nz > INT32_MAX) return iofail(LBM3D_ESIZE, "grid has more than 2^31-1 nodes");
  if (workspace_bytes < lbm3d_voxelize_workspace_bytes(nx, ny, nz)) return iofail(LBM3D_EINVAL, "workspace too small");
  // the error bound of the FP32 sums grows by about 4e-6 a triangle: past 400,000
  // it would leave most nodes open
  if (n_tris > 400000) return lbm3d_voxelize(stream, tris, n_tris, x0, y0, z0, dx, nx, ny, nz, solid);
  VoxGrid gr{x0, y0, z0, dx, nx, ny, nz, n_tris, 0.f};
  // a block's centre may lie up to 8 cells past the last node
  const double far = std::fmax(std::fmax(std::fmax(std::fabs(x0), std::fabs(x0 + dx * (nx + 8.0))),
                                         std::fmax(std::fabs(y0), std::fabs(y0 + dx * (ny + 8.0)))),
                               std::fmax(std::fabs(z0), std::fabs(z0 + dx * (nz + 8.0))));
  gr.eta = point_error(far, dx);
  int32_t *const ws = (int32_t *)workspace;
  int32_t *const list4 = ws + vox_list(nx, ny, nz, 0), *const list2 = ws + vox_list(nx, ny, nz, 1),
                 *const list1 = ws + vox_list(nx, ny, nz, 2);
  hipStream_t s = (hipStream_t)stream;
  const int32_t all = blocks_of(nx, 8) * blocks_of(ny, 8) * blocks_of(nz, 8);
  constexpr unsigned kMost = 2048;  // workgroups of 4 waves: 8 per CU
  k_clear_counts<<<1, 64, 0, s>>>(ws);
  k_winding_blocks<4><<<std::min<unsigned>(kMost, (unsigned)(all + 3) / 4), 256, 0, s>>>(tris, gr, nullptr, nullptr,
                                                                                       all, list4, ws, solid);
  k_winding_blocks<2><<<kMost, 256, 0, s>>>(tris, gr, list4, ws, 0, list2, ws + 1, solid);
  k_winding_blocks<1><<<kMost, 256, 0, s>>>(tris, gr, list2, ws + 1, 0, list1, ws + 2, solid);
  k_winding_nodes<<<kMost, 256, 0, s>>>(tris, gr, list1, ws + 2, solid);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return iofail(LBM3D_EHIP, "lbm3d_voxelize_blocks: ", hipGetErrorString(e));
  return LBM3D_OK;
}

int lbm3d_voxelize(void *stream, const float *tris, int32_t n_tris, double x0, double y0, double z0, double dx,
                   int32_t nx, int32_t ny, int32_t nz, int8_t *solid) {
  if (nx < 1 || ny < 1 || nz < 1 || n_tris < 0 || !(dx > 0)) return iofail(LBM3D_EINVAL, "bad grid or mesh size");
  if ((n_tris > 0 && !tris) || !solid) return iofail(LBM3D_EINVAL, "NULL mesh or output");
  const int64_t n = (int64_t)nx * ny * nz;
  if (n > INT32_MAX) return iofail(LBM3D_ESIZE, "grid has more than 2^31-1 nodes");
  k_winding<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(tris, n_tris, x0, y0, z0, dx, nx, ny, nz,
                                                                         solid);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return iofail(LBM3D_EHIP, "lbm3d_voxelize: ", hipGetErrorString(e));
  return LBM3D_OK;
}

}  // extern "C"
