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
// bounded FP32 sum settles nearly every node of the others.  Where that cannot pay it
// runs k_winding.
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
using lbm3d_winding::Corners;
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

// A count on the device that sends every node to k_winding when it is past `most`.
struct Gate {
  const int32_t *count;
  int32_t most;
  __device__ __forceinline__ bool past() const { return count && *count > most; }
};

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
              int32_t ny, int32_t nz, int8_t *__restrict__ solid, const Gate gate) {
  __shared__ float s_tri[kTriTile * 9];
  if (gate.count && !gate.past()) return;  // lbm3d_voxelize_blocks settles the nodes block by block
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
// nodes, 8 of a parent together and at last each by itself; a node that the error
// bound leaves open (on the surface, in the plane of a triangle next to it) gets the
// FP64 sum in triangle order, bit for bit k_winding's.
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
// 33.2 ms, every triangle for every child 3.2 ms, kFar 8 / 9 / 10 / 11 / 12 1.37 / 1.35 /
// 1.36 / 1.40 / 1.45 ms; 1,000 triangles of 6 cells on 48^3 560 / 522 / 462 / 425 / 393 us.
// With corners from FP64 differences and near triangles as they come (kFar 12) 2.02 ms
// instead of 1.65; loading the next triangle ahead changed nothing.
// ---------------------------------------------------------------------------
constexpr float kFar = 10.f;

struct VoxGrid {
  double x0, y0, z0, dx;
  int32_t nx, ny, nz;
  int32_t n_tris;
  float eta;  // point_error
};

// Omega >= 2 pi, Omega / 2 >= pi
__device__ __forceinline__ bool inside(float half) { return half >= 3.14159265f; }
// whether the bound e leaves no doubt of it, rounding of the wave's sum included (false for NaN)
__device__ __forceinline__ bool settled(float half, float e) { return fabsf(half - 3.14159265f) > 1.01f * e + 1e-4f; }

// a point as two FP32
__device__ __forceinline__ void split_point(double x, double y, double z, float3 &hi, float3 &lo) {
  hi = make_float3((float)x, (float)y, (float)z);
  lo = make_float3((float)(x - (double)hi.x), (float)(y - (double)hi.y), (float)(z - (double)hi.z));
}

// The children of side S of the parents (side 2S) in `list` (all parents if it is
// null): flags of the decided ones, the others' block indices to `next`.
template <int S>
__global__ void __launch_bounds__(256)
    k_winding_blocks(const float *__restrict__ tris, const VoxGrid gr, const int32_t *__restrict__ list,
                     const int32_t *__restrict__ count, int32_t all, int32_t *__restrict__ next,
                     int32_t *__restrict__ next_count, int8_t *__restrict__ solid,
                     const Gate gate) {
  if (gate.past()) return;  // k_winding takes every node
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
    float3 hi, lo;
    split_point(px, py, pz, hi, lo);
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
        close = !(s.near > kFar * R + s.edge);  // NaN too
        if (!close) all8.take(s.ax, s.ay, s.az, s.bx, s.by, s.bz, s.cx, s.cy, s.cz, slack, s.area2, s.edge, R);
      }
      const uint64_t m = __ballot(close);
      if (close)
        queue[wave][queued + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] =
            t;
      queued += __popcll(m);
      if (queued >= 64) {
        queued -= 64;
        near(queued, 64);
      }
    }
    if (queued > 0) near(0, queued);
    const float half8 = all8.angle(), err8 = all8.bound();
    float half[8], e[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      half[c] = child[c].angle() + half8;
      e[c] = child[c].bound() + err8 + 1e-6f * (fabsf(half8) + 1.f);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)  // 16 permutes in flight
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        half[c] += __shfl_xor(half[c], d);
        e[c] += __shfl_xor(e[c], d);
      }
    uint32_t open = 0;  // children left open, uniform in the wave
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int32_t ci = 2 * bi + (c >> 2 & 1), cj = 2 * bj + (c >> 1 & 1), ck = 2 * bk + (c & 1);
      if (ci >= cnx || cj >= cny || ck >= cnz) continue;  // uniform in the wave
      if (!settled(half[c], e[c])) {
        open |= 1u << c;
        continue;
      }
      const int8_t in = inside(half[c]) ? 1 : 0;
      for (int q = lane; q < S * S * S; q += 64) {
        const int i = S * ci + q / (S * S), j = S * cj + q / S % S, k = S * ck + q % S;
        if (i < gr.nx && j < gr.ny && k < gr.nz) solid[((int64_t)i * gr.ny + j) * gr.nz + k] = in;
      }
    }
    if (open) {
      // one addition to the counter for a parent: one for each of its 8 children, at 12 ns, took
      // nearly all of a box of 12 triangles on 128^3 nodes (7.0 ms, 1.2 with one)
      int32_t at = 0;
      if (lane == 0) at = atomicAdd(next_count, __popc(open));
      at = __builtin_amdgcn_readfirstlane(at);
      if (lane < 8 && (open >> lane & 1u)) {
        const int32_t ci = 2 * bi + (lane >> 2), cj = 2 * bj + (lane >> 1 & 1), ck = 2 * bk + (lane & 1);
        next[at + __popc(open & ((1u << lane) - 1u))] = (ci * cny + cj) * cnz + ck;
      }
    }
  }
}

__device__ __forceinline__ void node_point(const VoxGrid &gr, int32_t id, double &px, double &py, double &pz) {
  const int32_t k = id % gr.nz, t = id / gr.nz, j = t % gr.ny, i = t / gr.ny;
  px = gr.x0 + gr.dx * (double)i, py = gr.y0 + gr.dx * (double)j, pz = gr.z0 + gr.dx * (double)k;
}

// The bounded FP32 sum of all triangles at a node, by a wave: Omega / 2 and its bound.
__device__ __forceinline__ void node_sum(const float *__restrict__ tris, const VoxGrid &gr, double px, double py,
                                         double pz, int lane, float &half, float &e) {
  const float inv = (float)(1.0 / gr.dx), slack = point_slack(gr.eta);
  float3 hi, lo;
  split_point(px, py, pz, hi, lo);
  Product p;
  for (int32_t t = lane; t < gr.n_tris; t += 64) {
    const Corners s(tris, t, hi, lo, inv);
    p.take(s.ax, s.ay, s.az, s.bx, s.by, s.bz, s.cx, s.cy, s.cz, slack, 0.f, 0.f, 0.f);
  }
  half = p.angle(), e = p.bound();
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    half += __shfl_xor(half, d);
    e += __shfl_xor(e, d);
  }
}

// How many of kSamples nodes spread over the grid that sum leaves open.
constexpr int kSamples = 256;

__global__ void __launch_bounds__(256)
    k_winding_sample(const float *__restrict__ tris, const VoxGrid gr, int32_t *__restrict__ count) {
  const int64_t it = blockIdx.x * 4 + (threadIdx.x >> 6), nodes = (int64_t)gr.nx * gr.ny * gr.nz;
  const int32_t id = __builtin_amdgcn_readfirstlane((int32_t)((2 * it + 1) * nodes / (2 * kSamples)));
  double px, py, pz;
  node_point(gr, id, px, py, pz);
  float half, e;
  node_sum(tris, gr, px, py, pz, threadIdx.x & 63, half, e);
  if ((threadIdx.x & 63) == 0 && !settled(half, e)) atomicAdd(count, 1);
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Nodes left open by the blocks, up to kGroup a wave (one while there are no more nodes
// than waves).  First the bounded FP32 sum at the node itself, without the far triangles'
// bound, which grows with every layer of surface around: 32 overlapping boxes left nearly
// all of 128^3 nodes open, whose FP64 sums took 42 ms.  Then, for the nodes that this leaves
// open, the FP64 sum bit for bit as k_winding takes it: the lanes form the triangles'
// angles for one node after another, and lane j adds node j's in triangle order.  With 8
// nodes the adding is a tenth of the angles' time.
constexpr int kGroup = 8;

__global__ void __launch_bounds__(256)
    k_winding_nodes(const float *__restrict__ tris, const VoxGrid gr, const int32_t *__restrict__ list,
                    const int32_t *__restrict__ count, int8_t *__restrict__ solid) {
  __shared__ double terms[4][kGroup][65];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n = *count, waves = (int64_t)gridDim.x * 4;
  const int g = (int)(n >= kGroup * waves ? kGroup : (n + waves - 1) / waves);
  for (int64_t it = (blockIdx.x * 4 + wave) * (int64_t)g; it < n; it += waves * g) {
    const int m = (int)(n - it < g ? n - it : g);  // nodes of this round, one a lane
    const int32_t id = list[it + (lane < m ? lane : 0)];
    double px, py, pz, omega = 0.0;
    node_point(gr, id, px, py, pz);
    uint32_t open = 0;  // uniform in the wave
#pragma unroll 1
    for (int j = 0; j < m; ++j) {
      float half, e;
      node_sum(tris, gr, lane_value(px, j), lane_value(py, j), lane_value(pz, j), lane, half, e);
      if (!settled(half, e)) open |= 1u << j;
      else if (lane == j) solid[id] = inside(half) ? 1 : 0;
    }
    if (!open) continue;
    const bool mine = lane < m && (open >> lane & 1u);
    for (int32_t base = 0; base < gr.n_tris; base += 64) {
      const int cnt = gr.n_tris - base < 64 ? gr.n_tris - base : 64;
      float v[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) v[k] = tris[(int64_t)(base + (lane < cnt ? lane : 0)) * 9 + k];
#pragma unroll 1
      for (uint32_t left = open; left; left &= left - 1u) {
        const int j = __builtin_amdgcn_readfirstlane(__ffs((int)left) - 1);
        terms[wave][j][lane] = triangle_angle(v, lane_value(px, j), lane_value(py, j), lane_value(pz, j));
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (mine)
        for (int q = 0; q < cnt; ++q) omega += terms[wave][lane][q];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (mine) solid[id] = winding_flag(omega);
  }
}

__global__ void k_clear_counts(int32_t *counts) {
  if (threadIdx.x < 4) counts[threadIdx.x] = 0;
}

// list places of a workspace, in int32: the counts, then the undecided blocks of 4,
// of 2 and the open nodes
int64_t vox_list(int32_t nx, int32_t ny, int32_t nz, int level) {
  int64_t at = 64;
  if (level > 0) at += (int64_t)blocks_of(nx, 4) * blocks_of(ny, 4) * blocks_of(nz, 4);
  if (level > 1) at += (int64_t)blocks_of(nx, 2) * blocks_of(ny, 2) * blocks_of(nz, 2);
  if (level > 2) at += (int64_t)nx * ny * nz;
  return at;
}

int launch_winding(hipStream_t s, const float *tris, const VoxGrid &gr, int8_t *solid, const Gate &gate) {
  const int64_t n = (int64_t)gr.nx * gr.ny * gr.nz;
  k_winding<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(tris, gr.n_tris, gr.x0, gr.y0, gr.z0, gr.dx, gr.nx, gr.ny,
                                                       gr.nz, solid, gate);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return iofail(LBM3D_EHIP, "lbm3d_voxelize: ", hipGetErrorString(e));
  return LBM3D_OK;
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
  const int64_t n = (int64_t)nx * ny * nz;
  const int32_t all = blocks_of(nx, 8) * blocks_of(ny, 8) * blocks_of(nz, 8);
  const int32_t blocks4 = blocks_of(nx, 4) * blocks_of(ny, 4) * blocks_of(nz, 4);
  constexpr unsigned kMost = 2048;  // workgroups of 4 waves: 8 per CU
  // When every node should take k_winding after all, which costs 4.6 ps a node and
  // triangle, or 0.39 us a triangle below about 85,000 nodes (launches that do not fill
  // the GPU):
  //  - It is over before the blocks' launches are (35 us at least).  80 triangles on 32^3
  //    nodes 36 us against 44, 160 67 against 47.
  //  - Few triangles, large ones, leave most blocks of 4 open, and waves that hold them on
  //    a few of their 64 lanes: against k_winding a block then costs about 0.85 + 85 /
  //    n_tris.  A box of 12 on 128^3 132 us against 1,165, 8 of them 1.0 ms against 2.7,
  //    32 3.8 against 5.4; 4 spheres of 80, which leave a quarter open, 3.1 ms against 0.3.
  //  - From 65,536 triangles the bound of the FP32 sums, about 5e-6 each, is a third of a
  //    radian: a closed surface stays clear of it (327,680 triangles on 48^3 221 ms against
  //    34), any other mesh may not.  256 nodes are tried first, and past a quarter of them
  //    left open (or all, with a NaN among the corners) k_winding takes over.
  const double work = std::fmax((double)n, 85000.0) / (double)n;
  const double share = work / (0.85 + 85.0 / std::max(n_tris, 1));  // of blocks left open, where both cost the same
  const Gate none{nullptr, 0}, few{ws, (int32_t)std::fmin(share * blocks4, 2e9)}, many{ws + 3, kSamples / 4};
  const Gate gate = n_tris > 65536 ? many : (few.most < blocks4 ? few : none);
  if (work * (double)n * n_tris < 9e6) return launch_winding(s, tris, gr, solid, none);
  k_clear_counts<<<1, 64, 0, s>>>(ws);
  if (n_tris > 65536) k_winding_sample<<<kSamples / 4, 256, 0, s>>>(tris, gr, ws + 3);
  k_winding_blocks<4><<<std::min<unsigned>(kMost, (unsigned)(all + 3) / 4), 256, 0, s>>>(
      tris, gr, nullptr, nullptr, all, list4, ws, solid, n_tris > 65536 ? many : none);
  if (gate.count)
    if (int rc = launch_winding(s, tris, gr, solid, gate)) return rc;
  // no more waves than blocks or nodes there can be: launches that find nothing are short
  const auto grid = [&](int64_t items) { return (unsigned)std::min<int64_t>(kMost, (items + 3) / 4); };
  const int64_t blocks2 = (int64_t)blocks_of(nx, 2) * blocks_of(ny, 2) * blocks_of(nz, 2);
  k_winding_blocks<2><<<grid(blocks4), 256, 0, s>>>(tris, gr, list4, ws, 0, list2, ws + 1, solid, gate);
  k_winding_blocks<1><<<grid(blocks2), 256, 0, s>>>(tris, gr, list2, ws + 1, 0, list1, ws + 2, solid, none);
  k_winding_nodes<<<grid(n), 256, 0, s>>>(tris, gr, list1, ws + 2, solid);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return iofail(LBM3D_EHIP, "lbm3d_voxelize_blocks: ", hipGetErrorString(e));
  return LBM3D_OK;
}

int lbm3d_voxelize(void *stream, const float *tris, int32_t n_tris, double x0, double y0, double z0, double dx,
                   int32_t nx, int32_t ny, int32_t nz, int8_t *solid) {
  if (nx < 1 || ny < 1 || nz < 1 || n_tris < 0 || !(dx > 0)) return iofail(LBM3D_EINVAL, "bad grid or mesh size");
  if ((n_tris > 0 && !tris) || !solid) return iofail(LBM3D_EINVAL, "NULL mesh or output");
  if ((int64_t)nx * ny * nz > INT32_MAX) return iofail(LBM3D_ESIZE, "grid has more than 2^31-1 nodes");
  return launch_winding((hipStream_t)stream, tris, VoxGrid{x0, y0, z0, dx, nx, ny, nz, n_tris, 0.f}, solid,
                        Gate{nullptr, 0});
}

}  // extern "C"
