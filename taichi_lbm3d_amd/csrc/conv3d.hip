// 3-D "same" convolutions for the warm-start surrogate: BF16 implicit GEMM on
// the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16), FP32 accumulation.  The C
// ABI is declared in include/lbm3d_conv.h.
//
// Forward (and data gradient, which is a forward convolution of the output
// gradient with flipped weights): GEMM with M = output channels, N = voxels,
// K = taps x input channels.  Activations are channels-last, so the 8
// consecutive K values a lane feeds to one MFMA are 8 consecutive channels of
// one (shifted) voxel: a single 16-byte LDS read.  k_conv3z marches along z
// (few input channels), k_conv3 walks bricks (many).
//
// Weight gradient: GEMM with M = output channels, N = input channels, K =
// voxels, the operands transposed by the LDS reads.  Workgroups write partial
// sums; k_fold_sets adds them in a fixed order.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <type_traits>

#include "lbm3d.h"
#include "lbm3d_conv.h"
#include "xcd.h"

#ifndef LBM3D_CONV_XCD_CHUNK
#define LBM3D_CONV_XCD_CHUNK 64  // tiled forward: runs of consecutive bricks per XCD (shared halos hit L2)
#endif
#ifndef LBM3D_CONVZ_XCD_CHUNK
#define LBM3D_CONVZ_XCD_CHUNK 32  // marching forward: runs of consecutive columns per XCD
#endif
#ifndef LBM3D_CONV_WGRAD_XCD_CHUNK
#define LBM3D_CONV_WGRAD_XCD_CHUNK 64  // weight gradient: runs of consecutive jobs per XCD (16 or 256: the same to 1 %)
#endif

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

thread_local char c_err[256] = "";

int cfail(int code, const char *msg) {
  snprintf(c_err, sizeof(c_err), "%s", msg);
  return code;
}

int ccheck(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    snprintf(c_err, sizeof(c_err), "%s: %s", what, hipGetErrorString(e));
    return LBM3D_EHIP;
  }
  return LBM3D_OK;
}

// exact c / d for c < 2^31: (c * m) >> s
struct Div {
  uint32_t d, m, s;
};
Div make_div(uint32_t d) {
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  Div r;
  r.d = d;
  r.m = (uint32_t)(((1ull << (31 + l)) + d - 1) / d);
  r.s = 31 + l;
  return r;
}
__device__ __forceinline__ uint32_t qdiv(uint32_t c, const Div &v) { return (uint32_t)(((uint64_t)c * v.m) >> v.s); }

struct Vol {
  int32_t n, d, h, w;
  Div dw, dh, dd;
  uint32_t vox;      // n*d*h*w
  int32_t periodic;  // 1: taps past a face wrap to the opposite face; 0: zero padding
};

Vol make_vol(int32_t n, int32_t d, int32_t h, int32_t w, int32_t periodic = 0) {
  Vol v;
  v.periodic = periodic;
  v.n = n;
  v.d = d;
  v.h = h;
  v.w = w;
  v.dw = make_div((uint32_t)w);
  v.dh = make_div((uint32_t)h);
  v.dd = make_div((uint32_t)d);
  v.vox = (uint32_t)((int64_t)n * d * h * w);
  return v;
}

// voxel index -> (b, z, y, x)
__device__ __forceinline__ void decode(const Vol &v, uint32_t m, int &b, int &z, int &y, int &x) {
  const uint32_t t = qdiv(m, v.dw);
  x = (int)(m - t * (uint32_t)v.w);
  const uint32_t t2 = qdiv(t, v.dh);
  y = (int)(t - t2 * (uint32_t)v.h);
  const uint32_t bb = qdiv(t2, v.dd);
  z = (int)(t2 - bb * (uint32_t)v.d);
  b = (int)bb;
}

// a coordinate one step outside [0, n) wrapped back in
__device__ __forceinline__ int wrap1(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }

__device__ __forceinline__ u32x4 ld16(const uint16_t *p) { return *reinterpret_cast<const u32x4 *>(p); }

__device__ __forceinline__ uint16_t to_bf16(float f) {
  const __hip_bfloat16 h = __float2bfloat16(f);  // round to nearest even
  return *reinterpret_cast<const uint16_t *>(&h);
}

// ---------------------------------------------------------------------------
// Forward: y[v][co] = act(sum_{tap, ci} x[v + off(tap)][ci] * w[co][tap*cin + ci] + bias[co])
// MFMA 16x16x32 lane layout: A (16 x 32): lane l holds row l%16, k = 8*(l/16) .. +7;
// B (32 x 16): column l%16, the same k; C (16 x 16): column l%16, rows 4*(l/16) .. +3.
//
// Forward 3x3x3 convolutions.  Both kernels below compute, per wave, fragments
// of 16 voxels (one x row) x 16 output channels.  K runs over chunks of 16
// input channels x 27 taps, 14 MFMA steps of two taps each (the 28th slot is
// zero): lane group g holds tap 2s + g/2, channels 8 (g%2) .. +7.  The weights
// are the MFMA's A operand (rows = output channels) and the voxels its B
// operand, so a lane ends up with 4 consecutive channels of one voxel and
// stores 8 bytes.  The order of the K steps is the same in both, so a result
// does not depend on which kernel computes it.
// ---------------------------------------------------------------------------
constexpr int kBz = 2, kBy = 8, kBx = 16;                  // brick
constexpr int kHz = kBz + 2, kHy = kBy + 2, kHx = kBx + 2;  // halo
constexpr int kHalo = kHz * kHy * kHx;                     // 720 voxels
constexpr int kSteps = 14;                                 // K steps per 16-channel chunk (28 tap slots)
constexpr int kHaloLoads = 6;                              // 16-byte halo loads per thread (6 x 256 >= 2 x 720)
constexpr int kHaloBuf = kHaloLoads * 256;                 // 16-byte entries of one LDS buffer
constexpr int kWRing = 7;                                  // weight fragments in flight (divides kSteps)

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

__device__ const uint32_t conv_zero[4] = {0u, 0u, 0u, 0u};  // what a halo voxel outside the volume reads

// halo-index offset of tap t from the halo voxel of its (-1, -1, -1) neighbour
__host__ __device__ constexpr int tap_halo_offset(int t) {
  return (t / 9) * kHy * kHx + ((t / 3) % 3) * kHx + (t % 3);
}

// A fragments of the weights: output channels 16 tile .. +15, a lane's row r16,
// 8 K values.  Packed weights hold [chunk][step][tile][lane] fragments, plain
// ones rows of kpad; both are a lane offset plus a uniform offset.  The 28th tap
// slot is zero: stored so when packed, read past the resource's end when not.
struct Weights {
  __amdgpu_buffer_rsrc_t r;
  int off, off_last, cin, cout, packed;
  __device__ __forceinline__ Weights(const uint16_t *w, int packed_, int cin_, int cout_, int kpad, int tile, int lane)
      : cin(cin_), cout(cout_), packed(packed_) {
    const int g = lane >> 4, second = g >> 1;
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w), (short)0,
                                          packed ? (cin / 16) * kSteps * cout * 64 : cout * kpad * 2, 0x00020000);
    off = packed ? (tile * 64 + lane) * 16
                 : 2 * ((16 * tile + (lane & 15)) * kpad + second * cin + 8 * (g & 1));
    off_last = !packed && second ? 0x7fffffff : off;
  }
  __device__ __forceinline__ u32x4 operator()(int c, int s) const {  // chunk c, step s
    const int so = packed ? (c * kSteps + s) * cout * 64 : 2 * (2 * s * cin + 16 * c);
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, s == kSteps - 1 ? off_last : off, so, 0);
    return u32x4{v[0], v[1], v[2], v[3]};
  }
};

// What a forward kernel reads and writes besides a plain input and output.
//   kUp    the input's first c_low channels are those of a volume of half the
//          extents, upsampled (each voxel read for its 2 x 2 x 2 block), the
//          others those of `x`: a concatenation that is never built
//   kPool  the 2 x 2 x 2 maximum of the output is written too (half extents)
//   kDown  of the output channels below c_split only the sum over 2 x 2 x 2 blocks
//          is written (half extents): the gradient of kUp's low part.  A
//          separate pass over the full extents took 84 us of a 2 x 128^3 training
//          step, and the 16 -> 48 convolution there takes 150 us where it took
//          193 with the store.
// c_split > 0: output channels below it go to `y` (c_split per voxel), the
// others to `y_hi`: the two parts of a concatenation's gradient.
// The copies and reductions these replace took 2.9 of 6.2 ms of a 2 x 192^3
// inference and 1.5 of 7.1 ms of a 2 x 128^3 training step; pooling in the
// epilogue adds nothing to the 250 us of a 16 -> 16 layer, and reading the
// upsampled part at half extents takes 96 -> 32 channels at 2 x 96^3 from 394 to
// 328 us.
enum ConvMode { kPlain = 0, kUp = 1, kPool = 2, kDown = 3 };

struct ConvExtra {
  const uint16_t *low;  // kUp
  int c_low;
  uint16_t *pool;       // kPool, kDown (c_split channels)
  int c_split;
  uint16_t *y_hi;
};

// bias and ReLU of 4 channels of one voxel
__device__ __forceinline__ f32x4 finish4(f32x4 v, const f32x4 b4, int relu) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] += b4[e];
    if (relu) v[e] = v[e] > 0.f ? v[e] : 0.f;
  }
  return v;
}

// 4 channels rounded and packed for one 8-byte store
__device__ __forceinline__ uint2 pack4(const f32x4 v) {
  return make_uint2((uint32_t)to_bf16(v[0]) | ((uint32_t)to_bf16(v[1]) << 16),
                    (uint32_t)to_bf16(v[2]) | ((uint32_t)to_bf16(v[3]) << 16));
}

// 1x1x1 convolutions: a matrix product of the voxels' channels, bound by its
// bytes.  A wave computes 4 fragments of 16 voxels x NT of 16 output channels with
// the weights as the A operand, so a lane has 4 channels of a voxel, and all of a
// chunk's loads are in flight together.  Two tiles' rows are interleaved by fours, so
// that a lane has 8 consecutive channels of both and a store takes 16 bytes, 64 of a
// voxel.  16 -> 16 channels at 2 x 128^3 (268 MB): 75 us with 2-byte stores and an
// address from coordinates per load -> 48 us (5.6 TB/s).  16 -> 128 at 2 x 96^3: 253 us
// with 2-byte stores, 337 with 8-byte ones of 32 bytes a voxel, 168 with 16-byte ones.
template <int NT>
__global__ void __launch_bounds__(256)
    k_conv1(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const float *__restrict__ bias,
            uint16_t *__restrict__ y, uint32_t vox, int cin, int cout, int kpad, int relu) {
  constexpr int H = NT > 1 ? 2 : 1;  // tiles whose rows are interleaved
  const int lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  const uint32_t m0 = blockIdx.x * 256u + (threadIdx.x & ~63u) + (uint32_t)r16;
  const int co0 = blockIdx.y * 16 * NT;
  // first of the 4 channels that rows 4 q .. 4 q + 3 of tile t stand for
  const auto channel = [&](int t, int q) { return co0 + 16 * H * (t / H) + 4 * H * q + 4 * (t % H); };
  f32x4 acc[4][NT];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kc = 0; kc < cin; kc += 32) {
    const int k = kc + 8 * g;
    u32x4 b[4], a[NT];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const uint32_t m = m0 + 16u * f;
      b[f] = m < vox && k < cin ? ld16(x + (size_t)m * cin + k) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)  // kpad: 32-multiple
      a[t] = ld16(w + (size_t)(channel(t, r16 >> 2) + (r16 & 3)) * kpad + k);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int f = 0; f < 4; ++f)
        acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[t]),
                                                            __builtin_bit_cast(bf16x8, b[f]), acc[f][t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < NT; t += H) {
    f32x4 b4[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int co = channel(t + h, g);
      b4[h] = bias ? f32x4{bias[co], bias[co + 1], bias[co + 2], bias[co + 3]} : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const uint32_t m = m0 + 16u * f;
      if (m >= vox) continue;
      uint16_t *const to = y + (size_t)m * cout + channel(t, g);
      const uint2 lo = pack4(finish4(acc[f][t], b4[0], relu));
      if constexpr (H == 2) {
        const uint2 hi = pack4(finish4(acc[f][t + 1], b4[1], relu));
        *reinterpret_cast<u32x4 *>(to) = u32x4{lo.x, lo.y, hi.x, hi.y};
      } else {
        *reinterpret_cast<uint2 *>(to) = lo;
      }
    }
  }
}

// The network's head: a 1x1x1 convolution whose first 4 of 16 output channels are
// used, rounded to BF16 and returned in FP32.  A wave takes 64 voxels: fragment f's
// weights stand in rows 4f .. 4f+3 of its A operand, so that lane group f ends
// with the 4 channels of fragment f's voxels, lane l with those of voxel l.
//
// kHeadOut writes the channels.  kHeadFields turns them into a warm start at once:
// v = channels 0-2 times scale_v, rho = 1 + channel 3 times scale_rho (or 1 with
// rho_one), both as a product with 1 on fluid voxels and 0 on solid ones, for the
// voxels of a box (core) of the volume, each step rounded on its own.  Per voxel
// of 16 channels 32 + 16 and 33 + 16 bytes, against 64 for the padded output and
// 56 more for the passes that read it: at 2 x 192^3 a convolution of 276 us and
// 400 us of passes -> 128 us (5.4 TB/s).
enum HeadMode { kHeadOut = 0, kHeadFields = 1 };

struct HeadFields {
  Vol core;             // one volume: the box
  int32_t h, w;         // extents of the volume it lies in
  int64_t first;        // the box's first voxel there
  const int8_t *solid;  // of the box
  float scale_v, scale_rho;
  int rho_one;
  float *rho, *v;
};

template <int MODE>
__global__ void __launch_bounds__(256)
    k_head(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, const float *__restrict__ bias,
           float *__restrict__ out, uint32_t vox, int cin, int kpad, const HeadFields hf) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  const uint32_t mw = blockIdx.x * 256u + (threadIdx.x & ~63u);
  if (mw >= vox) return;
  const uint16_t *src[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    uint32_t m = mw + 16u * f + (uint32_t)r16;
    if (m >= vox) m = vox - 1;
    int64_t at = m;
    if constexpr (MODE == kHeadFields) {
      int b, z, yy, xx;
      decode(hf.core, m, b, z, yy, xx);
      at = hf.first + ((int64_t)z * hf.h + yy) * hf.w + xx;
    }
    src[f] = x + at * cin;
  }
  f32x4 acc[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kc = 0; kc < cin; kc += 32) {
    const int k = kc + 8 * g;
    const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
    u32x4 b[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) b[f] = k < cin ? ld16(src[f] + k) : zero;
    const u32x4 row = ld16(w + (size_t)(r16 & 3) * kpad + k);  // the row of one of the 4 channels
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const u32x4 a = (r16 >> 2) == f ? row : zero;
      acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b[f]),
                                                       acc[f], 0, 0, 0);
    }
  }
  const uint32_t m = mw + (uint32_t)lane;
  if (m >= vox) return;
  float p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float lo = (g & 1) ? acc[1][e] : acc[0][e], hi = (g & 1) ? acc[3][e] : acc[2][e];
    p[e] = __uint_as_float((uint32_t)to_bf16(((g & 2) ? hi : lo) + (bias ? bias[e] : 0.f)) << 16);
  }
  if constexpr (MODE == kHeadOut) {
    *reinterpret_cast<float4 *>(out + (size_t)m * 4) = make_float4(p[0], p[1], p[2], p[3]);
  } else {
    const float fluid = hf.solid[m] ? 0.f : 1.f;
    float *const vm = hf.v + (size_t)m * 3;
#pragma unroll
    for (int e = 0; e < 3; ++e) vm[e] = p[e] * hf.scale_v * fluid;
    hf.rho[m] = hf.rho_one ? 1.f : 1.f + p[3] * hf.scale_rho * fluid;
  }
}

__device__ __forceinline__ f32x4 max4(const f32x4 a, const f32x4 b) {
  return f32x4{fmaxf(a[0], b[0]), fmaxf(a[1], b[1]), fmaxf(a[2], b[2]), fmaxf(a[3], b[3])};
}

// the value of the other voxel of an x pair (lanes r16 and r16 ^ 1)
__device__ __forceinline__ f32x4 other_x(f32x4 v) {
  f32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)  // quad_perm [1, 0, 3, 2]
    o[e] = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0xB1, 0xF, 0xF, true));
  return o;
}
// the maximum over the pair
__device__ __forceinline__ f32x4 max_xpair(f32x4 v) { return max4(v, other_x(v)); }

// The sum over a 2 x 2 x 2 block of voxels rounded to BF16, at its even x, in the
// order of torch's sum: z pairs, then the four (y, x) in turn.  a0, a1: this x, the
// even row, both planes; b0, b1: the odd row.
__device__ __forceinline__ f32x4 unpack4(uint2 v) {
  return f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xFFFF0000u), __uint_as_float(v.y << 16),
               __uint_as_float(v.y & 0xFFFF0000u)};
}
__device__ __forceinline__ f32x4 sum_block(uint2 a0, uint2 a1, uint2 b0, uint2 b1) {
  const f32x4 a = unpack4(a0) + unpack4(a1), b = unpack4(b0) + unpack4(b1);
  return ((a + other_x(a)) + b) + other_x(b);
}

// where a tile's output goes: base pointer and channels per voxel
struct OutPlace {
  uint16_t *y;
  int c, co;
  __device__ __forceinline__ OutPlace(uint16_t *y_, int cout, int tile, int g, const ConvExtra &ex) {
    const bool hi = ex.c_split > 0 && 16 * tile >= ex.c_split;
    y = hi ? ex.y_hi : y_;
    c = ex.c_split > 0 ? (hi ? cout - ex.c_split : ex.c_split) : cout;
    co = 16 * tile + 4 * g - (hi ? ex.c_split : 0);
  }
};

// Bricks of one launch: n volumes of nbz x nby x nbx bricks, x fastest.
struct Bricks {
  uint32_t n;
  Div dx, dy, dz;
};

Bricks make_bricks(int32_t n, int32_t d, int32_t h, int32_t w) {
  const uint32_t nbz = (uint32_t)(d + kBz - 1) / kBz, nby = (uint32_t)(h + kBy - 1) / kBy,
                 nbx = (uint32_t)(w + kBx - 1) / kBx;
  Bricks b;
  b.n = (uint32_t)n * nbz * nby * nbx;
  b.dx = make_div(nbx);
  b.dy = make_div(nby);
  b.dz = make_div(nbz);
  return b;
}

// brick -> volume and first voxel
__device__ __forceinline__ void brick_origin(const Bricks &bk, uint32_t bi, int &bb, int &z0, int &y0, int &x0) {
  const uint32_t t = qdiv(bi, bk.dx), u = qdiv(t, bk.dy), v = qdiv(u, bk.dz);
  x0 = (int)(bi - t * bk.dx.d) * kBx;
  y0 = (int)(t - u * bk.dy.d) * kBy;
  z0 = (int)(u - v * bk.dz.d) * kBz;
  bb = (int)v;
}

// Many input channels: workgroups loop over bricks of 2 x 8 x 16 output voxels
// (z, y, x) and compute 16 CT output channels.  Wave w takes channel tile w % CT
// and, of each brick, the rows y = YR (w / CT) .. +YR-1 (YR = 2 CT) of both
// planes, MF = 2 YR fragments.  Per chunk of 16 input channels the brick's halo
// (4 x 10 x 18 voxels) is staged in one of two LDS buffers, straight from
// memory; the next chunk's (or brick's) halo is loaded while the MFMAs of the
// current one run, so a chunk has one barrier and no exposed load.  Weight
// fragments are streamed kWRing - 1 steps ahead.  STAGE (weights as rows, one tile a
// workgroup): a fragment comes from 32 places, too many for each of four waves to
// fetch; they are staged with the halo, once for the workgroup (80 -> 80 channels at
// 2 x 64^3 467 -> 296 us, 64 -> 64 at 2 x 24^3 28 -> 25).
// Bound by the MFMAs (half the LDS reads, with two channel tiles a wave, 145 -> 143
// us for 192 -> 64, but 382 -> 400 for 96 -> 32 at 2 x 96^3): 192 -> 64 channels at
// 2 x 48^3 take 150 us (980 TFLOP/s) against 305 for one 16-channel tile per workgroup
// with its halo loaded behind a barrier.
template <int CT, int MODE, bool STAGE>
__global__ void __launch_bounds__(256, 2)
    k_conv3(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, int packed,
            const float *__restrict__ bias, uint16_t *__restrict__ y, const Vol vol, int cin, int cout, int kpad,
            int relu, const Bricks bk, const ConvExtra ex) {
  constexpr int YR = 2 * CT, MF = 2 * YR;
  // [voxel][16 channels as two 16-byte halves]; two arrays, so that a read of
  // one never waits for the loads into the other
  __shared__ u32x4 haloA[kHaloBuf], haloB[kHaloBuf];
  __shared__ u32x4 fragA[STAGE ? kSteps * 64 : 1], fragB[STAGE ? kSteps * 64 : 1];  // [step][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int half = g & 1, second = g >> 1;  // channel half and tap parity of this lane's K values
  const int tile = blockIdx.y * CT + wave % CT;
  const int yr0 = (wave / CT) * YR;  // the wave's first brick row
  const int nch = cin / 16;
  const int64_t vstride = (int64_t)vol.d * vol.h * vol.w;  // voxels per volume

  const Weights weight(w, packed, cin, cout, kpad, tile, lane);
  u32x4 wr[kWRing];
  if constexpr (!STAGE) {
#pragma unroll
    for (int s = 0; s < kWRing - 1; ++s) wr[s] = weight(0, s);
  }
  auto load_weights = [&](int c, u32x4 *frag) {
    const uint16_t *const row = w + ((size_t)(16 * tile + r16) * kpad + second * cin + 8 * half + 16 * c);
    for (int s = wave; s < kSteps; s += 4) {
      const uint16_t *const src = s == kSteps - 1 && second ? reinterpret_cast<const uint16_t *>(conv_zero)
                                                            : row + 2 * s * cin;
      __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(frag + 64 * s), 16, 0, 0);
    }
  };

  // halo loads of one brick: entry e = 256 q + thread is half e & 1 of halo
  // voxel e / 2; its voxel index in the volume, or -1 outside it
  int hvox[kHaloLoads], lvox[MODE == kUp ? kHaloLoads : 1];  // lvox: in the half-extent volume
  const uint16_t *xv = x, *lv = ex.low;
  const int c_skip = MODE == kUp ? cin - ex.c_low : cin, nlow = MODE == kUp ? ex.c_low / 16 : 0;
  auto locate = [&](uint32_t bi) {
    int bb, z0, y0, x0;
    brick_origin(bk, bi, bb, z0, y0, x0);
    xv = x + (size_t)bb * vstride * c_skip;
    if (MODE == kUp) lv = ex.low + (size_t)bb * (vstride >> 3) * ex.c_low;
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));  // decompose the entries here, not once into registers held across the loop
#pragma unroll
    for (int q = 0; q < kHaloLoads; ++q) {
      const int hv = (t >> 1) + 128 * q;
      const int hz = hv / (kHy * kHx), r = hv - hz * (kHy * kHx);
      const int hy = r / kHx, hx = r - hy * kHx;
      int zz = z0 + hz - 1, yy = y0 + hy - 1, xx = x0 + hx - 1;
      if (vol.periodic) {  // halo voxels past a face come from the opposite face
        zz = wrap1(zz, vol.d);
        yy = wrap1(yy, vol.h);
        xx = wrap1(xx, vol.w);
      }
      const bool in = hv < kHalo && (unsigned)zz < (unsigned)vol.d && (unsigned)yy < (unsigned)vol.h &&
                      (unsigned)xx < (unsigned)vol.w;
      hvox[q] = in ? (zz * vol.h + yy) * vol.w + xx : -1;
      if (MODE == kUp) lvox[q] = in ? ((zz >> 1) * (vol.h >> 1) + (yy >> 1)) * (vol.w >> 1) + (xx >> 1) : -1;
    }
  };
  auto load_halo = [&](int c, u32x4 *buf) {
    if constexpr (STAGE) load_weights(c, buf == haloA ? fragA : fragB);
#pragma unroll
    for (int q = 0; q < kHaloLoads; ++q) {
      const uint16_t *src = xv + ((int64_t)hvox[q] * c_skip + 16 * (c - nlow) + 8 * ((int)threadIdx.x & 1));
      if (MODE == kUp && c < nlow) src = lv + ((int64_t)lvox[q] * ex.c_low + 16 * c + 8 * ((int)threadIdx.x & 1));
      if (hvox[q] < 0) src = reinterpret_cast<const uint16_t *>(conv_zero);
      __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(buf + 256 * q + 64 * wave), 16, 0, 0);
    }
  };

  // B fragment f = (z, row), step s: halo byte address a0 + 32 (z kHy kHx + row
  // kHx + T(2s)), plus for the second half of the lanes 32 (T(2s+1) - T(2s)),
  // one of three values: the next voxel in x, the next row's or plane's first.
  const uint32_t a0 = (uint32_t)(16 * (2 * (yr0 * kHx + r16) + half));
  const uint32_t ax = a0 + (second ? 32u : 0u);
  const uint32_t ay = a0 + (second ? (uint32_t)(32 * (kHx - 2)) : 0u);
  const uint32_t az = a0 + (second ? (uint32_t)(32 * (kHy * kHx - 2 * kHx - 2)) : 0u);

  // one chunk's 14 steps from buffer `buf`
  auto multiply = [&](f32x4 *acc, const u32x4 *buf, int c) {
    // fragments in groups of 4 (group k: step k / GS, fragments 4 (k % GS) ..
    // +3), read one group ahead of their MFMAs; the scheduling barriers keep
    // the compiler from reading further ahead and spilling
    constexpr int GS = MF / 4, NG = kSteps * GS;
    const char *const hb = reinterpret_cast<const char *>(buf);
    u32x4 v[2][4];
    auto read_group = [&](int k) {
      const int s = k / GS, t0 = 2 * s, t1 = 2 * s + 1;
      const uint32_t al = t1 >= 27 ? a0 : (t1 % 9 == 0 ? az : (t1 % 3 == 0 ? ay : ax));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int f = 4 * (k % GS) + j;
        const uint32_t imm = (uint32_t)(32 * ((f / YR) * kHy * kHx + (f % YR) * kHx + tap_halo_offset(t0)));
        v[k & 1][j] = *reinterpret_cast<const u32x4 *>(hb + al + imm);
      }
    };
    read_group(0);
    if constexpr (STAGE) wr[0] = (buf == haloA ? fragA : fragB)[lane];
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      if (k + 1 < NG) read_group(k + 1);
      const int s = k / GS;
      if constexpr (STAGE) {
        if (k % GS == 0 && s + 1 < kSteps) wr[(s + 1) % kWRing] = (buf == haloA ? fragA : fragB)[64 * (s + 1) + lane];
      } else if (k % GS == 0) {  // the fragment kWRing - 1 steps on, of this, the next or the next brick's first chunk
        const int sn = s + kWRing - 1;
        const int cn = sn < kSteps ? c : (c + 1 < nch ? c + 1 : 0);
        wr[sn % kWRing] = weight(cn, sn % kSteps);
      }
      const bf16x8 av = __builtin_bit_cast(bf16x8, wr[s % kWRing]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int f = 4 * (k % GS) + j;
        u32x4 vv = v[k & 1][j];
        if (s == kSteps - 1 && second) vv = u32x4{0u, 0u, 0u, 0u};  // the 28th tap slot
        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, vv), acc[f], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const uint32_t per_xcd = gridDim.x >> 3;
  uint32_t it = blockIdx.x >> 3;
  uint32_t bi = xcd_block(LBM3D_CONV_XCD_CHUNK, blockIdx.x & 7u, it, bk.n);
  if (bi >= bk.n) return;  // uniform in the workgroup
  locate(bi);
  load_halo(0, haloA);
  while (bi < bk.n) {
    const uint32_t bcur = bi;
    f32x4 acc[MF];
#pragma unroll
    for (int f = 0; f < MF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto next_brick = [&](u32x4 *buf) {
      it += per_xcd;
      bi = xcd_block(LBM3D_CONV_XCD_CHUNK, blockIdx.x & 7u, it, bk.n);
      if (bi < bk.n) {
        locate(bi);
        load_halo(0, buf);
      }
    };
    // One chunk: wait for this thread's halo loads and (the barrier) everyone's;
    // all waves are then past their reads of the other buffer, so the next
    // chunk's (or brick's) loads into it can start.
    auto chunk = [&](int c, u32x4 *cur, u32x4 *other) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      __syncthreads();
      if (c + 1 < nch)
        load_halo(c + 1, other);
      else if (!(nch & 1))
        next_brick(other);
      __builtin_amdgcn_sched_barrier(0);
      multiply(acc, cur, c);
    };
    int c = 0;
    for (; c + 1 < nch; c += 2) {
      chunk(c, haloA, haloB);
      chunk(c + 1, haloB, haloA);
    }
    if (c < nch) {  // an odd chunk count: the next brick starts in the same buffer, once it has been read
      chunk(c, haloA, haloB);
      __syncthreads();
      next_brick(haloA);
    }
    // C layout: lane holds rows (channels) 4g .. 4g+3, column (voxel x) r16
    int bb, z0, y0, x0;
    brick_origin(bk, bcur, bb, z0, y0, x0);
    const OutPlace op(y, cout, tile, g, ex);
    f32x4 b4 = f32x4{0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) b4[e] = bias[16 * tile + 4 * g + e];
    }
    const int oy0 = y0 + yr0, ox = x0 + r16;
    const bool down = MODE == kDown && 16 * tile < ex.c_split;  // uniform in the wave
    uint16_t *yv = op.y + ((size_t)bb * vstride + ((int64_t)z0 * vol.h + oy0) * vol.w + ox) * op.c + op.co;
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      const int fz = f / YR, fy = f % YR;
      acc[f] = finish4(acc[f], b4, relu);
      if (!down && z0 + fz < vol.d && oy0 + fy < vol.h && ox < vol.w)
        *reinterpret_cast<uint2 *>(yv + ((int64_t)fz * vol.h + fy) * vol.w * op.c) = pack4(acc[f]);
    }
    if constexpr (MODE == kPool) {  // even extents: a block is inside whole or not at all
#pragma unroll
      for (int fy = 0; fy < YR; fy += 2) {
        const f32x4 m = max_xpair(max4(max4(acc[fy], acc[fy + 1]), max4(acc[YR + fy], acc[YR + fy + 1])));
        if (!(r16 & 1) && z0 < vol.d && oy0 + fy < vol.h && ox < vol.w)
          *reinterpret_cast<uint2 *>(
              ex.pool + ((size_t)bb * (vstride >> 3) +
                         ((int64_t)(z0 >> 1) * (vol.h >> 1) + ((oy0 + fy) >> 1)) * (vol.w >> 1) + (ox >> 1)) * cout +
              op.co) = pack4(m);
      }
    }
    if (MODE == kDown && down) {
#pragma unroll
      for (int fy = 0; fy < YR; fy += 2) {
        const f32x4 m = sum_block(pack4(acc[fy]), pack4(acc[YR + fy]), pack4(acc[fy + 1]), pack4(acc[YR + fy + 1]));
        if (!(r16 & 1) && z0 < vol.d && oy0 + fy < vol.h && ox < vol.w)
          *reinterpret_cast<uint2 *>(
              ex.pool + ((size_t)bb * (vstride >> 3) +
                         ((int64_t)(z0 >> 1) * (vol.h >> 1) + ((oy0 + fy) >> 1)) * (vol.w >> 1) + (ox >> 1)) *
                            ex.c_split + op.co) = pack4(m);
      }
    }
  }
}

// Few input channels (16 WCH, WCH <= 3): a march along z.  A workgroup owns a
// column of TY x 16 output voxels (y, x), 16 CT output channels and a run of
// planes.  The input planes it needs, with their one-voxel border and all
// channels, go through a ring of 4 LDS slots: while output plane z is computed
// from slots z-1, z, z+1, plane z+2 is loaded into the fourth, straight to LDS.
// Every input plane is read once per column, in whole rows of all channels (the
// bricks of k_conv3 read each plane twice, 32 bytes of a voxel at a time), and
// the weights stay in registers.
// Bound by HBM for 16 -> 16 channels (2 x 192^3: 250 us, 3.6 TB/s of
// activations, against 480 us before and 360 us in bricks) and by the MFMAs for
// 48 -> 16 (624 us, 940 TFLOP/s, against 1,225 and 841; a quarter of the LDS reads
// saved 12 %, by sharing a fragment between three output planes, which changes the
// order of the sums).
constexpr int kRing = 4;

// Columns of one launch: n volumes of nby x nbx columns (x fastest), each cut
// into segs runs of zl planes (the slowest index).
struct Columns {
  uint32_t n;  // workgroups
  Div dx, dy, dn;
  int32_t zl;
};

template <int WCH, int CT, int TY, int MODE>
__global__ void __launch_bounds__(256, 2)
    k_conv3z(const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, int packed,
             const float *__restrict__ bias, uint16_t *__restrict__ y, const Vol vol, int cout, int kpad, int relu,
             const Columns ck, const ConvExtra ex) {
  constexpr int cin = 16 * WCH, P = 2 * WCH;          // 16-byte pieces of a voxel
  constexpr int MF = TY * CT / 4;                     // rows (fragments) of a wave
  constexpr int E = (TY + 2) * kHx * P;               // pieces of one slot
  constexpr int NQ = (E + 255) / 256;                 // loads per thread and plane
  constexpr int VB = 16 * P, RB = kHx * VB;           // bytes of a voxel and of a halo row
  __shared__ u32x4 ring[kRing * E + P];               // one voxel of slack: the 28th tap slot reads past the end
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int half = g & 1, second = g >> 1;
  const int tile = blockIdx.y * CT + wave % CT;
  const int row0 = (wave / CT) * MF;

  const uint32_t b = xcd_block(LBM3D_CONVZ_XCD_CHUNK, blockIdx.x & 7u, blockIdx.x >> 3, ck.n);
  if (b >= ck.n) return;  // padding block of the grid
  const uint32_t t1_ = qdiv(b, ck.dx), t2_ = qdiv(t1_, ck.dy), seg = qdiv(t2_, ck.dn);
  const int x0 = (int)(b - t1_ * ck.dx.d) * 16, y0 = (int)(t1_ - t2_ * ck.dy.d) * TY, bb = (int)(t2_ - seg * ck.dn.d);
  const int z_begin = (int)seg * ck.zl, z_end = z_begin + ck.zl < vol.d ? z_begin + ck.zl : vol.d;
  const int64_t vstride = (int64_t)vol.d * vol.h * vol.w, pstride = (int64_t)vol.h * vol.w;
  const int c_skip = MODE == kUp ? cin - ex.c_low : cin;
  const uint16_t *const xv = x + (size_t)bb * vstride * c_skip;
  const uint16_t *const lv = MODE == kUp ? ex.low + (size_t)bb * (vstride >> 3) * ex.c_low : nullptr;

  // this thread's pieces of a plane: entry e = 256 q + thread is piece e % P of
  // halo voxel e / P; its byte offset in the plane, the same for every plane
  uint32_t off[NQ];
  uint32_t valid = 0, from_low = 0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int e = 256 * q + (int)threadIdx.x;
    const int hv = e / P, pc = e % P, hy = hv / kHx, hx = hv % kHx;
    int yy = y0 + hy - 1, xx = x0 + hx - 1;
    if (vol.periodic) {
      yy = wrap1(yy, vol.h);
      xx = wrap1(xx, vol.w);
    }
    const bool in = e < E && (unsigned)yy < (unsigned)vol.h && (unsigned)xx < (unsigned)vol.w;
    off[q] = in ? 2u * ((uint32_t)(yy * vol.w + xx) * (uint32_t)c_skip + 8u * (uint32_t)pc) : 0u;
    if (MODE == kUp) {
      if (8 * pc < ex.c_low) {
        from_low |= 1u << q;
        if (in) off[q] = 2u * ((uint32_t)((yy >> 1) * (vol.w >> 1) + (xx >> 1)) * (uint32_t)ex.c_low + 8u * (uint32_t)pc);
      } else {
        off[q] -= 2u * (uint32_t)ex.c_low;  // the skip volume's own channel
      }
    }
    valid |= (in ? 1u : 0u) << q;
    if (e < E && !in)  // never loaded: zero in every slot
      for (int sl = 0; sl < kRing; ++sl) ring[sl * E + e] = u32x4{0u, 0u, 0u, 0u};
  }
  auto load_plane = [&](int z, int slot) {
    if (vol.periodic) z = wrap1(z, vol.d);
    if ((unsigned)z < (unsigned)vol.d) {
      const char *base = reinterpret_cast<const char *>(xv + z * pstride * c_skip);
      const char *low = MODE == kUp ? reinterpret_cast<const char *>(lv + (z >> 1) * (pstride >> 2) * ex.c_low) : base;
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if ((valid >> q) & 1u)
          __builtin_amdgcn_global_load_lds((gptr_t)((MODE == kUp && ((from_low >> q) & 1u) ? low : base) + off[q]),
                                           (lptr_t)(ring + (slot * E + 256 * q + 64 * wave)), 16, 0, 0);
    } else {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if (256 * q + (int)threadIdx.x < E) ring[slot * E + 256 * q + threadIdx.x] = u32x4{0u, 0u, 0u, 0u};
    }
  };
  load_plane(z_begin - 1, 0);
  load_plane(z_begin, 1);
  load_plane(z_begin + 1, 2);

  const Weights weight(w, packed, cin, cout, kpad, tile, lane);
  u32x4 wr[WCH * kSteps];
#pragma unroll
  for (int i = 0; i < WCH * kSteps; ++i) wr[i] = weight(i / kSteps, i % kSteps);
  const OutPlace op(y, cout, tile, g, ex);
  f32x4 b4 = f32x4{0.f, 0.f, 0.f, 0.f};
  if (bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) b4[e] = bias[16 * tile + 4 * g + e];
  }

  // B fragment f (row row0 + f), step s, chunk c: byte address l0 + slot of the
  // tap's plane + RB (f + dy) + VB dx + 32 c; the second half of the lanes is one
  // voxel on, or one row less two voxels on (steps whose second tap starts a
  // row), or in the next plane (step 4)
  const uint32_t l0 = (uint32_t)((row0 * kHx + r16) * VB + 16 * half);
  const uint32_t dx1 = second ? (uint32_t)VB : 0u, dy1 = second ? (uint32_t)(RB - 2 * VB) : 0u;
  const char *const lds = reinterpret_cast<const char *>(ring);
  const int oy0 = y0 + row0, ox = x0 + r16;
  uint16_t *yv = op.y + ((size_t)bb * vstride + ((int64_t)z_begin * vol.h + oy0) * vol.w + ox) * op.c + op.co;
  f32x4 even[MODE == kPool ? MF / 2 : 1];  // the even plane's row-pair maxima (runs start on even planes)
  uint2 evenb[MODE == kDown ? MF : 1];     // the even plane's rounded values
  const bool down = MODE == kDown && 16 * tile < ex.c_split;  // uniform in the wave
  int slot = 0;                            // of plane z - 1
  for (int z = z_begin; z < z_end; ++z) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this thread's loads of plane z + 1
    __syncthreads();                     // everyone's; and plane z - 2 has been read by all
    if (z + 1 < z_end) load_plane(z + 2, (slot + 3) & 3);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t sA = (uint32_t)slot * (E * 16), sB = (uint32_t)((slot + 1) & 3) * (E * 16),
                   sC = (uint32_t)((slot + 2) & 3) * (E * 16);
    const uint32_t ax = l0 + sA + dx1, ay = l0 + sA + dy1, a4 = l0 + (second ? sB : sA + (uint32_t)(2 * RB + 2 * VB));
    const uint32_t bx = l0 + sB + dx1, by = l0 + sB + dy1, cx = l0 + sC + dx1, cy = l0 + sC + dy1;
    f32x4 acc[MF];
#pragma unroll
    for (int f = 0; f < MF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int NI = WCH * kSteps * MF, NG = NI / 4;  // MFMAs, in groups of 4
    static_assert(NI % 4 == 0, "whole groups");
    u32x4 v[2][4];
    auto read_group = [&](int k) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * k + j, f = i % MF, s = (i / MF) % kSteps, c = i / (MF * kSteps);
        const int t = 2 * s, r = t % 9, dy = r / 3, dx = r % 3;  // first tap, in its plane
        const bool row = (2 * s + 1) % 3 == 0;                    // the second tap starts a row
        const uint32_t a = s == 4 ? a4 : (t < 9 ? (row ? ay : ax) : (t < 18 ? (row ? by : bx) : (row && s < 13 ? cy : cx)));
        const uint32_t imm = (uint32_t)((s == 4 ? f * RB : (f + dy) * RB + dx * VB) + 32 * c);
        v[k & 1][j] = *reinterpret_cast<const u32x4 *>(lds + a + imm);
      }
    };
    read_group(0);
#pragma unroll
    for (int k = 0; k < NG; ++k) {
      if (k + 1 < NG) read_group(k + 1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * k + j, f = i % MF, s = (i / MF) % kSteps;
        u32x4 vv = v[k & 1][j];
        if (s == kSteps - 1 && second) vv = u32x4{0u, 0u, 0u, 0u};  // the 28th tap slot
        acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[i / MF]),
                                                         __builtin_bit_cast(bf16x8, vv), acc[f], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // C layout: lane holds rows (channels) 4g .. 4g+3, column (voxel x) r16
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      acc[f] = finish4(acc[f], b4, relu);
      if (!down && oy0 + f < vol.h && ox < vol.w)
        *reinterpret_cast<uint2 *>(yv + (int64_t)f * vol.w * op.c) = pack4(acc[f]);
    }
    if constexpr (MODE == kPool) {
#pragma unroll
      for (int f = 0; f < MF; f += 2) {
        const f32x4 m = max4(acc[f], acc[f + 1]);
        if (!(z & 1)) {
          even[f / 2] = m;
        } else {
          const f32x4 p = max_xpair(max4(even[f / 2], m));
          if (!(r16 & 1) && oy0 + f < vol.h && ox < vol.w)
            *reinterpret_cast<uint2 *>(
                ex.pool + ((size_t)bb * (vstride >> 3) +
                           ((int64_t)(z >> 1) * (vol.h >> 1) + ((oy0 + f) >> 1)) * (vol.w >> 1) + (ox >> 1)) * cout +
                op.co) = pack4(p);
        }
      }
    }
    if (MODE == kDown && down) {
#pragma unroll
      for (int f = 0; f < MF; f += 2) {
        const uint2 lo = pack4(acc[f]), hi = pack4(acc[f + 1]);
        if (!(z & 1)) {
          evenb[f] = lo;
          evenb[f + 1] = hi;
        } else {
          const f32x4 p = sum_block(evenb[f], lo, evenb[f + 1], hi);
          if (!(r16 & 1) && oy0 + f < vol.h && ox < vol.w)
            *reinterpret_cast<uint2 *>(
                ex.pool + ((size_t)bb * (vstride >> 3) +
                           ((int64_t)(z >> 1) * (vol.h >> 1) + ((oy0 + f) >> 1)) * (vol.w >> 1) + (ox >> 1)) *
                              ex.c_split + op.co) = pack4(p);
        }
      }
    }
    yv += pstride * op.c;
    slot = (slot + 1) & 3;
  }
}

// wt[ci][tap'*cout + co] = w[co][tap*cin + ci], tap' = taps-1-tap; zero padding columns
__global__ void k_wflip(const uint16_t *__restrict__ w, uint16_t *__restrict__ wt, int cin, int cout, int taps,
                        int kpad_in, int kpad_out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)cin * kpad_out;
  if (i >= total) return;
  const int ci = (int)(i / kpad_out), k = (int)(i % kpad_out);
  uint16_t val = 0;
  if (k < taps * cout) {
    const int tp = k / cout, co = k % cout;
    const int tap = taps - 1 - tp;
    val = w[(size_t)co * kpad_in + tap * cin + ci];
  }
  wt[i] = val;
}

// FP32 weights w[cout][kpad] (3x3x3) to BF16 MFMA fragments: wp in k_conv3's
// packed order, [chunk][step][tile][lane][8], and, when wt is not null, the
// flipped weights of the data gradient (k_wflip's) in the same order.  One
// thread per lane of a fragment; the 28th tap slot is zero.  A launch takes up to
// kPackItems layers: one is 4 to 6 us of latency, so the network's 14 layers take
// 9 us together and 66 one by one.  W: float, or the bits of BF16 weights.
constexpr int kPackItems = 16;

struct PackItem {
  const void *w;
  uint16_t *wp, *wt;
  int32_t cin, cout, kpad;
  uint32_t first;  // block
};
struct PackList {
  int n;
  PackItem item[kPackItems];
};

__device__ __forceinline__ uint32_t bf16_bits(float f) { return to_bf16(f); }
__device__ __forceinline__ uint32_t bf16_bits(uint16_t h) { return h; }

template <typename W>
__global__ void __launch_bounds__(256) k_wpack(const PackList list) {
  int k = 0;
  while (k + 1 < list.n && blockIdx.x >= list.item[k + 1].first) ++k;  // uniform
  const PackItem &it = list.item[k];
  const W *const w = static_cast<const W *>(it.w);
  const int cin = it.cin, cout = it.cout, kpad = it.kpad;
  const int frags = kSteps * (cin / 16) * (cout / 16);  // the same for both
  int i = (int)((blockIdx.x - it.first) * 256 + threadIdx.x);
  const bool flip = i >= frags * 64;
  if (flip) i -= frags * 64;
  if (i >= frags * 64 || (flip && !it.wt)) return;
  const int ci_n = flip ? cout : cin, co_n = flip ? cin : cout;  // of the convolution the fragments are for
  const int lane = i & 63, fr = i >> 6;
  const int tile = fr % (co_n / 16), cs = fr / (co_n / 16);
  const int s = cs % kSteps, c = cs / kSteps;
  const int co = 16 * tile + (lane & 15), g = lane >> 4;
  const int tap = 2 * s + (g >> 1), ci = 16 * c + 8 * (g & 1);
  u32x4 v = u32x4{0u, 0u, 0u, 0u};
  if (tap < 27) {
    W f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      f[e] = flip ? w[(size_t)(ci + e) * kpad + (26 - tap) * cin + co] : w[(size_t)co * kpad + tap * cin + ci + e];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bf16_bits(f[2 * e]) | (bf16_bits(f[2 * e + 1]) << 16);
  }
  *reinterpret_cast<u32x4 *>((flip ? it.wt : it.wp) + (size_t)i * 8) = v;
}

// ---------------------------------------------------------------------------
// Weight gradients,
//   dw[co][tap*cin + ci] = sum over voxels v of dy[v][co] * x[v + off(tap)][ci]:
// MFMAs with M = 16 output channels (A = dy), N = 16 input channels (B = x) and
// K = 32 voxels.  Both operands need 8 consecutive voxels of one channel per
// lane from channels-last data: ds_read_b64_tr_b16 transposes a block of 4
// voxels x 16 channels on the way out of LDS, so dy and x are staged as they
// are, straight from memory.
//
// 3x3x3: a workgroup takes 16 input and 16 WCO output channels and a run of
// bricks (2 x 8 x 16 voxels, as the forward kernel's), which it stages one at a time.  A K chunk
// is two rows of the brick.  A wave owns one channel tile and one dx, that is 9
// taps: it keeps the brick's 8 A fragments in registers and reads each of the 36
// B fragments that its taps share (halo plane, first halo row) once, for 72
// MFMAs.  Every tap sees the chunks of a brick in order, and the bricks in
// order, so a set's sums do not depend on how the fragments are shared.
// Bound by HBM and the L2 misses of the halos at 16 -> 16 channels (2 x 128^3: 118
// us with the fold, 190 us with the operands transposed by 2-byte LDS writes and
// each B fragment read for one MFMA), by the LDS reads (0.6 fragments per MFMA)
// at more (96 -> 32 at 2 x 64^3: 130 us, 388 before), and by writing and folding
// the sets where voxels are few (128 -> 128 at 2 x 16^3: 31 us, 43 before).
// ---------------------------------------------------------------------------
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short bf16x8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) bf16x4 *ltr_t;

// 8 voxels of one channel: a 4-voxel transposed read and the next
__device__ __forceinline__ bf16x8 read_tr(const char *p, int next) {
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)p);
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(p + next));
  return __builtin_bit_cast(bf16x8, (bf16x8s)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int WCO, bool UP>
__global__ void __launch_bounds__(192 * WCO)
    k_wgrad3(const uint16_t *__restrict__ x, const uint16_t *__restrict__ dy, float *__restrict__ part, const Vol vol,
             int cin, int cout, int kpad, const Bricks bk, uint32_t per_block, uint32_t n, Div tiles,
             const uint16_t *__restrict__ low, int c_low) {
  constexpr int T = 192 * WCO;                                // threads
  constexpr int PX = 2, PD = 2 * WCO;                         // 16-byte pieces of a voxel of x and of dy
  constexpr int VX = 16 * PX, VD = 16 * PD;                   // bytes
  constexpr int EX = kHalo * PX, ED = 256 * PD;               // pieces of x's halo and of dy
  constexpr int NX = (EX + T - 1) / T, ND = (ED + T - 1) / T;  // loads per thread
  __shared__ u32x4 tile[EX + ED];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int dx = wave % 3, wco = wave / 3;
  // (set, channel tiles) with the tiles fastest, in runs per XCD: the workgroups
  // that read the same bricks, and their halos, run together on one L2 (48 -> 16
  // channels at 2 x 128^3: 295 us, 552 in plain order)
  const uint32_t job = xcd_block(LBM3D_CONV_WGRAD_XCD_CHUNK, blockIdx.x & 7u, blockIdx.x >> 3, n);
  if (job >= n) return;  // padding block of the grid
  const uint32_t set = qdiv(job, tiles), ct = job - set * tiles.d;
  const uint32_t nci = (uint32_t)cin / 16u;
  const int co0 = (int)(ct / nci) * 16 * WCO, c0 = (int)(ct % nci) * 16;
  // UP: x's channels below c_low come from `low`, a volume of half the extents, upsampled
  const bool from_low = UP && c0 < c_low;
  const int sh = from_low ? 1 : 0, xd = vol.d >> sh, xh = vol.h >> sh, xw = vol.w >> sh;
  const int xc = from_low ? c_low : (UP ? cin - c_low : cin), xc0 = UP && !from_low ? c0 - c_low : c0;
  const uint16_t *const xsrc = from_low ? low : x;
  const int64_t vstride = (int64_t)vol.d * vol.h * vol.w;

  int hpos[NX];  // halo coordinates of this thread's pieces of x: hz << 10 | hy << 5 | hx
#pragma unroll
  for (int q = 0; q < NX; ++q) {
    const int hv = (T * q + (int)threadIdx.x) / PX;
    hpos[q] = hv / (kHy * kHx) << 10 | hv / kHx % kHy << 5 | hv % kHx;
  }
  auto load = [&](uint32_t brick) {
    const uint16_t *const zero = reinterpret_cast<const uint16_t *>(conv_zero);
    int bb, z0, y0, x0;
    brick_origin(bk, brick, bb, z0, y0, x0);
    const uint16_t *const xv = xsrc + (size_t)bb * xd * xh * xw * xc + xc0;
    const uint16_t *const dv = dy + (size_t)bb * vstride * cout + co0;
#pragma unroll
    for (int q = 0; q < NX; ++q) {
      const int e = T * q + (int)threadIdx.x;
      const int zz = z0 - 1 + (hpos[q] >> 10), yy = y0 - 1 + (hpos[q] >> 5 & 31), xx = x0 - 1 + (hpos[q] & 31);
      const bool in = (unsigned)zz < (unsigned)vol.d && (unsigned)yy < (unsigned)vol.h && (unsigned)xx < (unsigned)vol.w;
      const uint16_t *src = xv + ((int64_t)(((zz >> sh) * xh + (yy >> sh)) * xw + (xx >> sh)) * xc + 8 * (e % PX));
      if (NX * T == EX || e < EX)
        __builtin_amdgcn_global_load_lds((gptr_t)(in ? src : zero), (lptr_t)(tile + T * q + 64 * wave), 16, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < ND; ++q) {
      const int e = T * q + (int)threadIdx.x, v = e / PD;
      const int zz = z0 + (v >> 7), yy = y0 + (v >> 4 & 7), xx = x0 + (v & 15);
      const bool in = zz < vol.d && yy < vol.h && xx < vol.w;
      const uint16_t *src = dv + ((int64_t)((zz * vol.h + yy) * vol.w + xx) * cout + 8 * (e % PD));
      if (ND * T == ED || e < ED)
        __builtin_amdgcn_global_load_lds((gptr_t)(in ? src : zero), (lptr_t)(tile + EX + T * q + 64 * wave), 16, 0, 0);
    }
  };

  // transposed reads: lane 16 g + i takes 4 channels of voxel i / 4 of the 4
  // (then the next 4) of row g / 2 of the pair, x half g % 2
  const char *const xb = reinterpret_cast<const char *>(tile) +
                         (((g >> 1) * kHx + dx + 8 * (g & 1) + (r16 >> 2)) * VX + 8 * (r16 & 3));
  const char *const db =
      reinterpret_cast<const char *>(tile) + EX * 16 + ((8 * g + (r16 >> 2)) * VD + 32 * wco + 8 * (r16 & 3));
  f32x4 acc[9];  // taps (tz, ty) of this dx
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const uint32_t b0 = set * per_block, b1 = b0 + per_block < bk.n ? b0 + per_block : bk.n;
  for (uint32_t br = b0; br < b1; ++br) {
    if (br != b0) __syncthreads();  // the previous brick's reads are done
    load(br);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    bf16x8 a[8];
#pragma unroll
    for (int kc = 0; kc < 8; ++kc) a[kc] = read_tr(db + 32 * kc * VD, 4 * VD);
    // B fragment n = (halo plane hz, first halo row hy), two read ahead; the
    // scheduling barriers keep the compiler from reading further ahead
    bf16x8 b[3];
    auto read_b = [&](int n) { b[n % 3] = read_tr(xb + ((n / 9) * kHy + n % 9) * kHx * VX, 4 * VX); };
    read_b(0);
    read_b(1);
#pragma unroll
    for (int n = 0; n < 36; ++n) {
      const int hz = n / 9, hy = n % 9;
      if (n + 2 < 36) read_b(n + 2);
#pragma unroll
      for (int tz = 0; tz < 3; ++tz)
#pragma unroll
        for (int ty = 0; ty < 3; ++ty) {
          const int z = hz - tz, y2 = hy - ty;  // the chunk's plane and first row
          if (z >= 0 && z < 2 && y2 >= 0 && y2 < 8 && !(y2 & 1))
            acc[3 * tz + ty] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[4 * z + y2 / 2], b[n % 3], acc[3 * tz + ty],
                                                                     0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // C layout: lane holds rows (co) 4g .. 4g+3, column (ci) r16; part[set][co][kpad]
  float *dst = part + (size_t)set * cout * kpad + (size_t)(co0 + 16 * wco + 4 * g) * kpad + c0 + r16;
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[(size_t)e * kpad + (3 * t + dx) * cin] = acc[t][e];
}

// 1x1x1: workgroup (p, channel tiles): a run of bricks, staged one at a time in
// 16 KB, so that eight workgroups' loads are in flight on a CU; wave w takes K
// chunks 2w and 2w + 1 of each.  Partial sets: one per wave, part[4 p +
// wave][co][kpad].  Bound by HBM.  Jobs in the order of k_wgrad3's: 32 -> 32 at 2 x 128^3
// 338 us with the tiles slowest, 139 with them fastest.
__global__ void __launch_bounds__(256)
    k_wgrad1(const uint16_t *__restrict__ x, const uint16_t *__restrict__ dy, float *__restrict__ part, const Vol vol,
             int cin, int cout, int kpad, const Bricks bk, uint32_t per_block, uint32_t n, Div tiles) {
  __shared__ u32x4 tile[1024];  // 256 voxels x 16 channels of x, then of dy
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const uint32_t job = xcd_block(LBM3D_CONV_WGRAD_XCD_CHUNK, blockIdx.x & 7u, blockIdx.x >> 3, n);
  if (job >= n) return;  // padding block of the grid
  const uint32_t set = qdiv(job, tiles), ct = job - set * tiles.d, nci = (uint32_t)cin / 16u;
  const int co0 = (int)(ct / nci) * 16, c0 = (int)(ct % nci) * 16;
  auto load = [&](uint32_t brick) {
    const uint16_t *const zero = reinterpret_cast<const uint16_t *>(conv_zero);
    int bb, z0, y0, x0;
    brick_origin(bk, brick, bb, z0, y0, x0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int e = 256 * q + (int)threadIdx.x, v = e >> 1;
      const int zz = z0 + (v >> 7), yy = y0 + (v >> 4 & 7), xx = x0 + (v & 15);
      const bool in = zz < vol.d && yy < vol.h && xx < vol.w;
      const int64_t vx = (((int64_t)bb * vol.d + zz) * vol.h + yy) * vol.w + xx;
      const uint16_t *const xs = x + (vx * cin + c0 + 8 * (e & 1)), *const ds = dy + (vx * cout + co0 + 8 * (e & 1));
      __builtin_amdgcn_global_load_lds((gptr_t)(in ? xs : zero), (lptr_t)(tile + 256 * q + 64 * wave), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gptr_t)(in ? ds : zero), (lptr_t)(tile + 512 + 256 * q + 64 * wave), 16, 0, 0);
    }
  };
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  const int off = (64 * wave + 8 * g + (r16 >> 2)) * 32 + 8 * (r16 & 3);
  const uint32_t b0 = set * per_block, b1 = b0 + per_block < bk.n ? b0 + per_block : bk.n;
  const char *const p = reinterpret_cast<const char *>(tile) + off;
  for (uint32_t br = b0; br < b1; ++br) {
    if (br != b0) __syncthreads();  // the previous brick's reads are done
    load(br);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(read_tr(p + 8192 + 1024 * c, 128), read_tr(p + 1024 * c, 128), acc,
                                                    0, 0, 0);
  }
  float *dst = part + ((size_t)set * 4 + wave) * cout * kpad + (size_t)(co0 + 4 * g) * kpad + c0 + r16;
#pragma unroll
  for (int e = 0; e < 4; ++e) dst[(size_t)e * kpad] = acc[e];
}

// v[0] = ((v0 + v8) + (v4 + v12)) + ...: the sum of 16 terms, halves first
__device__ __forceinline__ float tree16(float v[16]) {
#pragma unroll
  for (int w = 8; w >= 1; w >>= 1)
#pragma unroll
    for (int j = 0; j < w; ++j) v[j] += v[j + w];
  return v[0];
}

// dst[e] = sum of the terms part[q step + e] of nsets <= 4096 sets (step: the size
// of a set, or of 16 after a first level), in an order fixed by nsets alone:
// groups of 16 consecutive sets by tree16 while more than 16 terms remain, the
// last (at most 16) terms one after another.  A block takes E elements and sums
// G = 1024 / E groups at a time, a group a thread, in one launch.  Elements whose
// column (e % kpad) is past `used` are padding: 0.
template <int E>
__global__ void __launch_bounds__(1024)
    k_fold_sets(const float *__restrict__ part, float *__restrict__ dst, uint32_t size, uint32_t step, int nsets,
                int kpad, int used) {
  constexpr int G = 1024 / E, T = G / 16;  // groups, and groups of groups, of a round
  __shared__ float red[G][E], top[T][E];
  const int col = threadIdx.x % E, row = threadIdx.x / E;
  const uint32_t e = blockIdx.x * E + col;
  const bool live = e < size && e % (uint32_t)kpad < (uint32_t)used, last = row == 0 && e < size;
  const float *const p = part + (e < size ? e : size - 1);  // terms past the end: clamped loads, then 0
  float s = 0.f;
  if (nsets <= 16) {  // one term a set
    red[row][col] = live && row < nsets ? p[row * (int64_t)step] : 0.f;
    __syncthreads();
    if (last) {
      for (int q = 0; q < nsets; ++q) s += red[q][col];
      dst[e] = s;
    }
    return;
  }
  const int groups = (nsets + 15) / 16;
  for (int q0 = 0; q0 < groups; q0 += G) {  // uniform in the block
    const int first = (q0 + row) * 16;
    float v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = p[(int64_t)(first + j < nsets ? first + j : nsets - 1) * step];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = live && first + j < nsets ? v[j] : 0.f;
    red[row][col] = tree16(v);  // the round before has read its rows: see the barrier below
    __syncthreads();
    if (groups <= 16) {  // at most 16 terms: one after another
      if (last)
        for (int q = 0; q < groups; ++q) s += red[q][col];
      break;
    }
    if (row < T) {
      float u[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) u[j] = red[16 * row + j][col];
      top[row][col] = tree16(u);
    }
    __syncthreads();
    if (last)
      for (int t = 0; t < T && q0 + 16 * t < groups; ++t) s += top[t][col];
  }
  if (last) dst[e] = s;
}

// The same for at most 256 sets of many elements: one thread an element.
__global__ void __launch_bounds__(256)
    k_fold_few(const float *__restrict__ part, float *__restrict__ dst, int64_t size, int nsets, int kpad, int used) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= size) return;
  float s = 0.f;
  if ((int)(e % kpad) < used) {
    const float *const p = part + e;
    if (nsets <= 16) {
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = j < nsets ? p[(int64_t)j * size] : 0.f;
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (j < nsets) s += v[j];
    } else {
      for (int first = 0; first < nsets; first += 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = first + j < nsets ? p[(int64_t)(first + j) * size] : 0.f;
        s += tree16(v);
      }
    }
  }
  dst[e] = s;
}

// One level of the fold for more sets: part[16 q] = tree16 of sets 16 q .. +15, in place.
__global__ void __launch_bounds__(256)
    k_fold_level(float *__restrict__ part, int64_t size, int nsets) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)((nsets + 15) / 16) * size) return;
  const int64_t q = i / size, e = i - q * size;
  float v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = 16 * q + j < nsets ? part[(16 * q + j) * size + e] : 0.f;
  part[16 * q * size + e] = tree16(v);
}

// Elements a block of k_fold_sets takes: whole lines of 64 elements where there are
// blocks for every CU, 32 for the two smallest weight gradients (13,824 of 2048
// sets: 38 us with the gradient, 47 with 16, 64 with 8; 7,168: 102-111 with any of
// 16, 32, 64), and 4 for a layer's bias gradient (16 of 2048 sets: 88 us with the
// pass over 2 x 128^3 voxels before it, 97 with 64, where one block walks them in
// eight rounds).
void fold_block(hipStream_t s, const float *part, float *dst, uint32_t size, uint32_t step, int nsets, int kpad,
                int used) {
  if (size >= 16384)
    k_fold_sets<64><<<(size + 63) / 64, 1024, 0, s>>>(part, dst, size, step, nsets, kpad, used);
  else if (size >= 1024)
    k_fold_sets<32><<<(size + 31) / 32, 1024, 0, s>>>(part, dst, size, step, nsets, kpad, used);
  else
    k_fold_sets<4><<<(size + 3) / 4, 1024, 0, s>>>(part, dst, size, step, nsets, kpad, used);
}

int fold_sets(hipStream_t s, float *part, float *dst, int64_t size, int nsets, int kpad, int used) {
  // a thread an element where there are enough elements to fill the GPU: 32 sets of
  // 442 k (the gradient of 128 -> 128 channels, 2 x 16^3, takes 30 us in all; 60
  // with a block of 16 waves for 64 elements), but 128 sets of 57 k 29 us with
  // the block and 35 with the thread
  if (nsets <= 256 && size >= 100000) {
    k_fold_few<<<(unsigned)((size + 255) / 256), 256, 0, s>>>(part, dst, size, nsets, kpad, used);
  } else if (nsets <= 4096) {
    fold_block(s, part, dst, (uint32_t)size, (uint32_t)size, nsets, kpad, used);
  } else {
    const int64_t n = (int64_t)((nsets + 15) / 16) * size;
    k_fold_level<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(part, size, nsets);
    if (int rc = ccheck("fold of partial sums")) return rc;
    fold_block(s, part, dst, (uint32_t)size, (uint32_t)(16 * size), (nsets + 15) / 16, kpad, used);
  }
  return ccheck("fold of partial sums");
}

int check_conv(int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks) {
  if (n < 1 || d < 1 || h < 1 || wd < 1) return cfail(LBM3D_EINVAL, "volume extents must be >= 1");
  if (ks != 1 && ks != 3) return cfail(LBM3D_EINVAL, "kernel size must be 1 or 3");
  if (cin < 16 || cin > 256 || cin % 16 || cout < 16 || cout > 256 || cout % 16)
    return cfail(LBM3D_EINVAL, "channel counts must be multiples of 16 in [16, 256]");
  // voxel indices are 32-bit (exact magic division below 2^31); element offsets are 64-bit
  if ((int64_t)n * d * h * wd >= ((int64_t)1 << 31)) return cfail(LBM3D_ESIZE, "more than 2^31-1 voxels");
  return LBM3D_OK;
}

// Kernels that load 16-byte pieces straight to LDS, or through buffer resources, take
// tensors that start on 16 bytes.
int check_start(const void *a, const void *b = nullptr, const void *c = nullptr) {
  if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) return cfail(LBM3D_EINVAL, "tensors must start on 16 bytes");
  return LBM3D_OK;
}

constexpr int kWgTargetBlocks = 2048;

// Weight gradient: bricks per set of partial sums and sets, about kWgTargetBlocks
// (set, channel tile) pairs in all.  A set's bricks and the number of sets fix
// the order of the sums.
int wgrad_plan(const Bricks &bk, int32_t cin, int32_t cout, uint32_t &per) {
  const int64_t nb = bk.n;
  const int64_t tiles = (int64_t)(cout / 16) * (cin / 16);
  int64_t P = (kWgTargetBlocks + tiles - 1) / tiles;
  if (P > nb) P = nb;
  if (P < 1) P = 1;
  const int64_t pb = (nb + P - 1) / P;
  per = (uint32_t)pb;
  return (int)((nb + pb - 1) / pb);
}

constexpr int wgrad_sets(int ks) { return ks == 3 ? 1 : 4; }  // partial sets of a workgroup

// ---------------------------------------------------------------------------
// Periodic distance to solid (the surrogate's second input channel): the
// separable squared-distance transform as three min-plus passes,
//   g(v) = min over |o| <= M of f(v + o e_axis) + o^2  (coordinates wrapped),
// starting from f = 0 on solid cells and 3M^2 + 1 elsewhere, then
// dist = min(sqrt(f), M).  Exact for distances up to M; larger ones are capped.
// f >= 0, so an offset with o^2 >= the best value so far cannot improve it: a
// thread searches outwards, two offsets a round, and stops there: in a porous
// medium after a few offsets instead of 2M + 1.  Threads run along the innermost
// axis, so every pass reads coalesced rows.
//
// k_dist_lines keeps the lines of 64 neighbouring voxels along the searched axis in
// LDS (256 bytes a coordinate), so a line is read from memory once instead of once
// per offset tried, and the innermost pass is part of the middle one (ballots,
// dist_row).  Longer lines than 256 and margins from 64 take k_dist_rows and
// k_dist_axis, one pass an axis.  Bound by the rounds of LDS reads where a wave's 128
// voxels have one far from any solid.  M = 24:
//   157 x 149 x 160                         26 + 26 + 16 us -> 24 + 20 us
//   2 x 192^3, 16 BF16 channels written     40 + 90 + 148 us -> 55 + 96 us
//   100 x 110 x 66, whole call 25 -> 22 us; 192 x 192 x 20 the same (lanes past
//   the row's end idle); 8 waves a block and one voxel at a time 52 us for the first
// ---------------------------------------------------------------------------
// what the last pass writes: the distance; {mask, distance / scale} in FP32; or
// 16 BF16 channels of which those are the first two and the others zero
enum DistOut { kDistPlain = 0, kDistPair = 1, kDistNet = 2 };

struct DistGeo {
  int64_t total;
  int32_t d0, d1, d2;
  Div div0, div1, div2;  // by the extents, for totals below 2^31
  int32_t margin;
  float inv_scale;       // a power of two
};

// The outward search along a line of n values, from coordinates c and d at a time.
// An offset of m + 1 (the last round of an odd m) gives more than m^2, which the
// last pass caps.
template <class At>
__device__ __forceinline__ float2 dist_search2(const At &at, int c, int d, int n, int m) {
  float best_c = at(c), best_d = at(d);
  int lo_c = c, hi_c = c, lo_d = d, hi_d = d;
  float near = 1.f, far = 4.f;  // o^2, (o + 1)^2
  const auto below = [&](int i) { return i == 0 ? n - 1 : i - 1; };
  const auto above = [&](int i) { return i == n - 1 ? 0 : i + 1; };
  for (int o = 1; o <= m && near < fmaxf(best_c, best_d); o += 2) {
    const int lo_c1 = below(lo_c), hi_c1 = above(hi_c), lo_d1 = below(lo_d), hi_d1 = above(hi_d);
    lo_c = below(lo_c1), hi_c = above(hi_c1), lo_d = below(lo_d1), hi_d = above(hi_d1);
    best_c = fminf(best_c, fminf(fminf(at(lo_c1), at(hi_c1)) + near, fminf(at(lo_c), at(hi_c)) + far));
    best_d = fminf(best_d, fminf(fminf(at(lo_d1), at(hi_d1)) + near, fminf(at(lo_d), at(hi_d)) + far));
    near = far + (float)(2 * o + 3);
    far = near + (float)(2 * o + 5);
  }
  return make_float2(best_c, best_d);
}

// The innermost pass for margins below 64, without a search, for the 64 voxels of a
// wave: the solid bits of the row's coordinates z0 - 64 .. z0 + 127 (wrapped); each
// lane finds its nearest set bit on either side.
__device__ __forceinline__ float dist_row(uint64_t before, uint64_t here, uint64_t after, int lane, int m) {
  // bit i of up: solid at distance i above (0 .. 63); bit 63 - i of down: below
  const uint64_t up = lane ? (here >> lane) | (after << (64 - lane)) : here;
  const uint64_t down = lane < 63 ? (here << (63 - lane)) | (before >> (lane + 1)) : here;
  const int du = up ? __ffsll((unsigned long long)up) - 1 : 64, dd = down ? __clzll((long long)down) : 64;
  const int dmin = du < dd ? du : dd;
  return (float)(dmin <= m ? dmin * dmin : 3 * m * m + 1);
}

// mask and scaled distance as the first two of 16 BF16 channels, in one word
__device__ __forceinline__ uint32_t net_word(float mask, float scaled) {
  return (uint32_t)to_bf16(mask) | ((uint32_t)to_bf16(scaled) << 16);
}

// The middle (AXIS 1: with the innermost pass before it) or the outer axis (AXIS 0)
// of the lines through 64 voxels z0 .. z0 + 63 of a row; 16 waves.  LDS is filled
// first, 8 values per lane in flight; a row's three bytes give its distances.  Then
// every wave searches two of the line's rows at a time.  A voxel is solid where the
// squared distance is 0, so the last pass needs no mask.
constexpr int kDistWaves = 16, kDistAhead = 8;
constexpr int kDistLine = 256;  // longest line: 64 KB of LDS

template <int AXIS, int OUT>
__global__ void __launch_bounds__(64 * kDistWaves)
    k_dist_lines(const int8_t *__restrict__ solid, const float *__restrict__ f, void *__restrict__ out,
                 const DistGeo gm, const Div segs) {
  extern __shared__ float lines[];  // [coordinate][64]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = AXIS == 1 ? gm.d1 : gm.d0, m = gm.margin;
  const uint32_t t = qdiv(blockIdx.x, segs);
  const int z0 = (int)(blockIdx.x - t * segs.d) * 64;
  const int64_t plane = (int64_t)gm.d1 * gm.d2, stride = AXIS == 1 ? gm.d2 : plane;
  int64_t first = t * plane;  // of coordinate 0
  if (AXIS == 0) {
    const uint32_t vol = qdiv(t, gm.div1);
    first = (int64_t)vol * gm.d0 * plane + (int64_t)(t - vol * (uint32_t)gm.d1) * gm.d2;
  }
  const bool in = z0 + lane < gm.d2;
  const int z = in ? z0 + lane : gm.d2 - 1;
  const auto last = [&](int c) { return c < n ? c : n - 1; };
  if constexpr (AXIS == 1) {
    // coordinates z0 + lane - 64, + 0, + 64, each wrapped into the row
    const int zw = (z0 + lane) % gm.d2, step = 64 % gm.d2;
    const int zm = zw < step ? zw - step + gm.d2 : zw - step, zp = zw + step >= gm.d2 ? zw + step - gm.d2 : zw + step;
    for (int c0 = wave; c0 < n; c0 += kDistWaves * kDistAhead) {
      int8_t a[kDistAhead], b[kDistAhead], c[kDistAhead];
#pragma unroll
      for (int i = 0; i < kDistAhead; ++i) {
        const int8_t *const row = solid + first + (int64_t)last(c0 + kDistWaves * i) * stride;
        a[i] = row[zm];
        b[i] = row[zw];
        c[i] = row[zp];
      }
#pragma unroll
      for (int i = 0; i < kDistAhead; ++i) {
        const float v = dist_row(__ballot(a[i] != 0), __ballot(b[i] != 0), __ballot(c[i] != 0), lane, m);
        if (c0 + kDistWaves * i < n) lines[(c0 + kDistWaves * i) * 64 + lane] = v;
      }
    }
  } else {
    for (int c0 = wave; c0 < n; c0 += kDistWaves * kDistAhead) {
      float v[kDistAhead];
#pragma unroll
      for (int i = 0; i < kDistAhead; ++i) v[i] = f[first + last(c0 + kDistWaves * i) * stride + z];
#pragma unroll
      for (int i = 0; i < kDistAhead; ++i)
        if (c0 + kDistWaves * i < n) lines[(c0 + kDistWaves * i) * 64 + lane] = v[i];
    }
  }
  __syncthreads();
  auto put = [&](int c, float best) {
    const int64_t v = first + c * stride + z;
    if constexpr (AXIS == 1) {
      if (in) static_cast<float *>(out)[v] = best;
    } else {
      // correctly rounded: the distance an exact EDT (FP64) reports, cast to FP32
      const float dist = fminf(sqrtf(best), (float)m), mask = best == 0.f ? 1.f : 0.f, scaled = dist * gm.inv_scale;
      if constexpr (OUT == kDistPlain) {
        if (in) static_cast<float *>(out)[v] = dist;
      } else if constexpr (OUT == kDistPair) {
        if (in) static_cast<float2 *>(out)[v] = make_float2(mask, scaled);
      } else {
        // 32 bytes a voxel: a store takes 32 voxels, whole lines
        const uint32_t word = net_word(mask, scaled);
        u32x4 *const o4 = static_cast<u32x4 *>(out) + 2 * (first + c * stride + z0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t other = (uint32_t)__shfl((int)word, 32 * h + (lane >> 1));
          if (z0 + 32 * h + (lane >> 1) < gm.d2) o4[64 * h + lane] = u32x4{lane & 1 ? 0u : other, 0u, 0u, 0u};
        }
      }
    }
  };
  const auto at = [&](int c) { return lines[c * 64 + lane]; };
  for (int c = wave; c < n; c += 2 * kDistWaves) {
    const int d = c + kDistWaves < n ? c + kDistWaves : c;
    const float2 best = dist_search2(at, c, d, n, m);
    put(c, best.x);
    if (d != c) put(d, best.y);
  }
}

// the innermost pass by itself, one wave per 64 voxels of a row
__global__ void __launch_bounds__(256)
    k_dist_rows(const int8_t *__restrict__ solid, float *__restrict__ out, const DistGeo gm, Div segs, int64_t waves) {
  const int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wv >= waves) return;  // whole waves
  const int lane = threadIdx.x & 63, n = gm.d2;
  const int64_t row = waves < ((int64_t)1 << 31) ? (int64_t)qdiv((uint32_t)wv, segs) : wv / segs.d;
  const int z0 = (int)(wv - row * segs.d) * 64;
  const int8_t *line = solid + row * n;
  const int z = (z0 + lane) % n, step = 64 % n;
  const int zm = z < step ? z - step + n : z - step, zp = z + step >= n ? z + step - n : z + step;
  const float v = dist_row(__ballot(line[zm] != 0), __ballot(line[z] != 0), __ballot(line[zp] != 0), lane, gm.margin);
  if (z0 + lane < n) out[row * n + z0 + lane] = v;
}

template <int AXIS, int OUT>
__global__ void __launch_bounds__(256)
    k_dist_axis(const int8_t *__restrict__ solid, const float *__restrict__ f, void *__restrict__ out,
                const DistGeo gm) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= gm.total) return;
  const bool narrow = gm.total < ((int64_t)1 << 31);
  const int64_t row = narrow ? (int64_t)qdiv((uint32_t)v, gm.div2) : v / gm.d2;
  const int m = gm.margin;
  const float big = (float)(3 * m * m + 1);
  int n = gm.d2, c = (int)(v - row * gm.d2);
  int64_t stride = 1;
  if constexpr (AXIS != 2) {
    const int64_t plane = narrow ? (int64_t)qdiv((uint32_t)row, gm.div1) : row / gm.d1;
    if constexpr (AXIS == 1) {
      n = gm.d1;
      c = (int)(row - plane * gm.d1);
      stride = gm.d2;
    } else {
      const int64_t vol = narrow ? (int64_t)qdiv((uint32_t)plane, gm.div0) : plane / gm.d0;
      n = gm.d0;
      c = (int)(plane - vol * gm.d0);
      stride = (int64_t)gm.d1 * gm.d2;
    }
  }
  const int64_t line = v - (int64_t)c * stride;  // this voxel's line at coordinate 0
  auto at = [&](int cc) -> float {
    const int64_t u = line + (int64_t)cc * stride;
    if constexpr (AXIS == 2) return solid[u] != 0 ? 0.f : big;
    else return f[u];
  };
  float best = at(c);
  int lo = c, hi = c;
  for (int o = 1; o <= m && (float)(o * o) < best; o += 2) {
    const int lo1 = lo == 0 ? n - 1 : lo - 1, hi1 = hi == n - 1 ? 0 : hi + 1;
    lo = lo1 == 0 ? n - 1 : lo1 - 1;
    hi = hi1 == n - 1 ? 0 : hi1 + 1;
    const float near = fminf(at(lo1), at(hi1)) + (float)(o * o);
    const float far = fminf(at(lo), at(hi)) + (float)((o + 1) * (o + 1));
    best = fminf(best, o < m ? fminf(near, far) : near);
  }
  if constexpr (AXIS != 0) {
    static_cast<float *>(out)[v] = best;
  } else {
    // correctly rounded: the distance an exact EDT (FP64) reports, cast to FP32
    const float dist = fminf(sqrtf(best), (float)m);
    if constexpr (OUT == kDistPlain) {
      static_cast<float *>(out)[v] = dist;
    } else {
      const float mask = solid[v] != 0 ? 1.f : 0.f, scaled = dist * gm.inv_scale;
      if constexpr (OUT == kDistPair) {
        static_cast<float2 *>(out)[v] = make_float2(mask, scaled);
      } else {
        u32x4 *o4 = static_cast<u32x4 *>(out) + 2 * v;
        o4[0] = u32x4{net_word(mask, scaled), 0u, 0u, 0u};
        o4[1] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  }
}

// bf16 y > 0 (false for -0, negatives and NaN)
__device__ __forceinline__ bool bf16_positive(uint32_t h) {
  return !(h & 0x8000u) && h != 0u && !((h & 0x7F80u) == 0x7F80u && (h & 0x7Fu));
}

__device__ __forceinline__ float bf16_to_f32(uint32_t h) { return __uint_as_float(h << 16); }

// Backward of y = relu(z): dz = g * (y > 0) (a masked element is g * 0.0 in
// FP32, rounded to bf16: a zero with g's sign, or NaN), stored to dz; with
// y == nullptr dz = g.  Each block also sums dz per channel over its voxels
// in FP32: part[block][c].  Data are [voxels][C] bf16, C dividing 2048, so a
// thread's 8-element chunks (chunk q covers elements 8q .. 8q+7) always hold
// the same 8 channels when the blocks' chunk ranges start on multiples of C/8.
//
// kGradPool: g has a second part, the gradient of y's 2 x 2 x 2 maximum: at the
// voxels that attain it, `share` (its gradient over their number, k_pool_share);
// the sum is rounded to BF16 first, as two accumulated gradients are.
struct PoolGrad {
  const uint16_t *pooled, *share;
  Vol vol;
  Div pieces;  // by C / 8
};

// kGradHead: g is the FP32 gradient of k_head's 4 channels; dz is it in BF16 as the
// first 4 of 16 channels (the others zero), and there is no ReLU.
enum GradMode { kGradPlain = 0, kGradPool = 1, kGradHead = 2 };

template <int MODE>
__global__ void __launch_bounds__(256)
    k_relu_bias_grad(const uint16_t *g, const uint16_t *__restrict__ y, uint16_t *dz,  // dz may be g
                     float *__restrict__ part, int64_t chunks, int C, int64_t per_block, const PoolGrad pg) {
  __shared__ float red[256][9];
  const int t = (int)threadIdx.x;
  const int64_t q0 = (int64_t)blockIdx.x * per_block;
  const int64_t q1 = q0 + per_block < chunks ? q0 + per_block : chunks;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  for (int64_t q = q0 + t; q < q1; q += 256) {
    u32x4 a = u32x4{0u, 0u, 0u, 0u};
    if constexpr (MODE != kGradHead) {
      a = ld16(g + q * 8);
    } else if (!(q & 1)) {
      const float4 p = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(g) + q * 2);
      const uint2 r = pack4(f32x4{p.x, p.y, p.z, p.w});
      a = u32x4{r.x, r.y, 0u, 0u};
    }
    if (MODE != kGradHead && y) {
      const u32x4 m = ld16(y + q * 8);
      if constexpr (MODE == kGradPool) {
        int b, z, yy, x;
        const uint32_t v = chunks < ((int64_t)1 << 31) ? qdiv((uint32_t)q, pg.pieces) : (uint32_t)(q / pg.pieces.d);
        decode(pg.vol, v, b, z, yy, x);
        const int64_t o = ((((int64_t)b * (pg.vol.d >> 1) + (z >> 1)) * (pg.vol.h >> 1) + (yy >> 1)) * (pg.vol.w >> 1) +
                           (x >> 1)) * C + 8 * (q - (int64_t)v * pg.pieces.d);
        const u32x4 top = ld16(pg.pooled + o), share = ld16(pg.share + o);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t r[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const uint32_t yk = (m[w] >> (16 * k)) & 0xFFFFu, tk = (top[w] >> (16 * k)) & 0xFFFFu;
            const float sk = bf16_to_f32((share[w] >> (16 * k)) & 0xFFFFu);
            const float gk = bf16_to_f32((a[w] >> (16 * k)) & 0xFFFFu);
            r[k] = to_bf16(gk + (yk == tk ? sk : sk * 0.0f));
          }
          a[w] = r[0] | (r[1] << 16);
        }
      }
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        uint32_t lo = a[w] & 0xFFFFu, hi = a[w] >> 16;
        if (!bf16_positive(m[w] & 0xFFFFu))
          lo = __bfloat16_as_ushort(__float2bfloat16(bf16_to_f32(lo) * 0.0f));
        if (!bf16_positive(m[w] >> 16))
          hi = __bfloat16_as_ushort(__float2bfloat16(bf16_to_f32(hi) * 0.0f));
        a[w] = lo | (hi << 16);
      }
    }
    *reinterpret_cast<u32x4 *>(dz + q * 8) = a;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      acc[2 * w] += bf16_to_f32(a[w] & 0xFFFFu);
      acc[2 * w + 1] += bf16_to_f32(a[w] >> 16);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[t][e] = acc[e];
  __syncthreads();
  if (t < C) {  // channel t: threads r, r + C/8, ... hold it in slot t % 8 (r = t / 8)
    const int groups = C / 8;
    float sum = 0.f;
    for (int u = t / 8; u < 256; u += groups) sum += red[u][t % 8];
    part[(int64_t)blockIdx.x * C + t] = sum;
  }
}

// The gradient of a 2 x 2 x 2 maximum, shared among the voxels that attain it:
// share = BF16(gp / count), one 16-byte piece (8 channels) per thread.  y >= 0
// (a ReLU output), so equal values have equal bits.
__global__ void __launch_bounds__(256)
    k_pool_share(const uint16_t *__restrict__ y, const uint16_t *__restrict__ pooled, const uint16_t *__restrict__ gp,
                 uint16_t *__restrict__ share, const Vol low, Div pieces, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const uint32_t v = total < ((int64_t)1 << 31) ? qdiv((uint32_t)i, pieces) : (uint32_t)(i / pieces.d);
  const int pc = (int)(i - (int64_t)v * pieces.d), c = 8 * (int)pieces.d;
  int b, z, yy, x;
  decode(low, v, b, z, yy, x);
  const int64_t h2 = 2 * low.h, w2 = 2 * low.w;
  const uint16_t *src = y + ((((int64_t)b * low.d + z) * 2 * h2 + 2 * yy) * w2 + 2 * x) * c + 8 * pc;
  const u32x4 top = ld16(pooled + i * 8), g = ld16(gp + i * 8);
  int cnt[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) cnt[e] = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const u32x4 a = ld16(src + (((k >> 2) * h2 + ((k >> 1) & 1)) * w2 + (k & 1)) * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      cnt[2 * e] += (a[e] & 0xFFFFu) == (top[e] & 0xFFFFu);
      cnt[2 * e + 1] += (a[e] >> 16) == (top[e] >> 16);
    }
  }
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = (uint32_t)to_bf16(bf16_to_f32(g[e] & 0xFFFFu) / (float)cnt[2 * e]) |
           ((uint32_t)to_bf16(bf16_to_f32(g[e] >> 16) / (float)cnt[2 * e + 1]) << 16);
  *reinterpret_cast<u32x4 *>(share + i * 8) = o;
}

// One forward convolution, as the launchers pass it on.
struct ConvCall {
  const uint16_t *x, *w;
  int packed;
  const float *bias;
  uint16_t *y;
  Vol vol;
  int cin, cout, kpad, relu;
  ConvExtra ex;
};

template <int CT, int MODE, bool STAGE = false>
void launch_conv3_bricks(hipStream_t s, const ConvCall &a, const Bricks &bk) {
  const unsigned gy = (unsigned)(a.cout / (16 * CT));
  // persistent workgroups: as many as are resident (3 per CU by LDS, 2 with staged
  // weights or where the kernel takes more than 168 VGPRs), in whole groups of 8 XCDs
  const int64_t resident = ((CT == 1 && !STAGE) || (CT == 2 && MODE != kUp) ? 768 : 512) / gy;
  int64_t gx = xcd_grid(bk.n, LBM3D_CONV_XCD_CHUNK);
  if (gx > resident) gx = resident & ~int64_t(7);
  if (gx < 8) gx = 8;
  k_conv3<CT, MODE, STAGE><<<dim3((unsigned)gx, gy), 256, 0, s>>>(a.x, a.w, a.packed, a.bias, a.y, a.vol, a.cin, a.cout,
                                                           a.kpad, a.relu, bk, a.ex);
}

template <int WCH, int CT, int TY, int MODE>
void launch_conv3z(hipStream_t s, const ConvCall &a) {
  const Vol &vol = a.vol;
  const int64_t nbx = (vol.w + 15) / 16, nby = (vol.h + TY - 1) / TY, gy = a.cout / (16 * CT);
  const int64_t cols = nbx * nby * vol.n;
  // planes per workgroup: the cut that takes the fewest rounds of resident
  // workgroups times planes (3 extra planes of border and start-up per run);
  // an even number with pooling and block sums
  const int64_t slots = 256 * (WCH == 1 ? 3 : 2);
  int64_t best = vol.d, best_cost = INT64_MAX;
  for (int64_t segs = 1; segs <= vol.d; ++segs) {
    int64_t zl = (vol.d + segs - 1) / segs;
    if (MODE == kPool || MODE == kDown) zl = (zl + 1) & ~int64_t(1);
    const int64_t runs = (vol.d + zl - 1) / zl;
    const int64_t cost = ((cols * runs * gy + slots - 1) / slots) * (zl + 3);
    if (cost < best_cost) best = zl, best_cost = cost;
    if (cols * segs * gy > 32 * slots) break;
  }
  Columns ck;
  ck.zl = (int32_t)best;
  const int64_t segs = (vol.d + ck.zl - 1) / ck.zl;
  ck.n = (uint32_t)(cols * segs);
  ck.dx = make_div((uint32_t)nbx);
  ck.dy = make_div((uint32_t)nby);
  ck.dn = make_div((uint32_t)vol.n);
  const dim3 grid((unsigned)xcd_grid(ck.n, LBM3D_CONVZ_XCD_CHUNK), (unsigned)gy);
  k_conv3z<WCH, CT, TY, MODE><<<grid, 256, 0, s>>>(a.x, a.w, a.packed, a.bias, a.y, vol, a.cout, a.kpad, a.relu, ck,
                                                   a.ex);
}

template <int MODE>
int launch_conv3(hipStream_t s, const ConvCall &a) {
  const Vol &vol = a.vol;
  const int tiles = a.cout / 16, cin = a.cin;
  const Bricks bk = make_bricks(vol.n, vol.d, vol.h, vol.w);
  if (xcd_grid(bk.n, LBM3D_CONV_XCD_CHUNK) > (int64_t)(UINT32_MAX / 256u))
    return cfail(LBM3D_ESIZE, "too many bricks for one launch");
  // March along z where the weights of all input channels fit the registers
  // (16 channels, or up to 48 for at most two channel tiles per workgroup) and a
  // plane's byte offsets fit 32 bits; bricks else.  Where both fit: 32 -> 32 at
  // 2 x 96^3 119-123 us either way, 32 -> 64 at 2 x 48^3 35 us either way, 16 -> 32
  // at 2 x 96^3 65 us marching and 79 in bricks.
  if ((cin == 16 || (cin <= 48 && tiles % 4 != 0)) && (int64_t)vol.h * vol.w * cin < ((int64_t)1 << 31)) {
    if (cin == 16) {
      if constexpr (MODE != kUp) {  // an upsampled and a skip part take 32 channels at least
        if (tiles % 4 == 0) launch_conv3z<1, 4, 8, MODE>(s, a);
        else if (tiles % 2 == 0) launch_conv3z<1, 2, 8, MODE>(s, a);
        else launch_conv3z<1, 1, 16, MODE>(s, a);
      }
    } else if (cin == 32) {
      if (tiles % 2 == 0) launch_conv3z<2, 2, 8, MODE>(s, a);
      else launch_conv3z<2, 1, 8, MODE>(s, a);
    } else {
      constexpr bool kTwo = MODE == kPlain || MODE == kUp;  // the even plane's values would spill
      if (kTwo && tiles % 2 == 0)
        launch_conv3z<3, 2, 8, kTwo ? MODE : kPlain>(s, a);
      else
        launch_conv3z<3, 1, 8, MODE>(s, a);
    }
    return ccheck("lbm3d_conv3d_fwd");
  }
  // as many channel tiles per workgroup (the halo is loaded once per workgroup)
  // as leave 2 workgroups per CU: 128 -> 128 channels at 2 x 16^3 take 17 us with
  // 256 workgroups of one tile, 32 us with 64 of four
  int ct = tiles % 4 == 0 ? 4 : (tiles % 2 == 0 ? 2 : 1);
  while (ct > 1 && (int64_t)bk.n * (tiles / ct) < 512) ct >>= 1;
  if (ct == 4) launch_conv3_bricks<4, MODE>(s, a, bk);
  else if (ct == 2) launch_conv3_bricks<2, MODE>(s, a, bk);
  else if (MODE == kPlain && !a.packed) launch_conv3_bricks<1, MODE, MODE == kPlain>(s, a, bk);
  else launch_conv3_bricks<1, MODE>(s, a, bk);
  return ccheck("lbm3d_conv3d_fwd");
}

int relu_bias_plan(int64_t voxels, int C, int64_t &chunks, int64_t &per_block) {
  chunks = voxels * C / 8;
  int64_t blocks = (chunks + 256 * 8 - 1) / (256 * 8);  // about 8 chunks per thread
  if (blocks > 2048) blocks = 2048;
  if (blocks < 1) blocks = 1;
  const int64_t unit = C / 8;
  per_block = (chunks + blocks - 1) / blocks;
  per_block = (per_block + unit - 1) / unit * unit;
  return (int)((chunks + per_block - 1) / per_block);
}

template <typename W>
int wpack(void *stream, int32_t count, const lbm3d_conv_pack *layers) {
  if (count < 0 || (count > 0 && !layers)) return cfail(LBM3D_EINVAL, "no layers");
  for (int32_t k = 0; k < count; ++k) {
    if (int rc = check_conv(1, 1, 1, 1, layers[k].cin, layers[k].cout, 3)) return rc;
    if (!layers[k].w || !layers[k].wp) return cfail(LBM3D_EINVAL, "NULL tensor");
  }
  for (int32_t k0 = 0; k0 < count; k0 += kPackItems) {
    PackList list{};
    uint32_t blocks = 0;
    for (int32_t k = k0; k < count && k < k0 + kPackItems; ++k) {
      const lbm3d_conv_pack &l = layers[k];
      list.item[list.n++] = PackItem{l.w, l.wp, l.wt, l.cin, l.cout, lbm3d_conv_kpad(l.cin, 3), blocks};
      blocks += (uint32_t)(kSteps * (l.cin / 16) * (l.cout / 16) * 64 * (l.wt ? 2 : 1) + 255) / 256;
    }
    k_wpack<W><<<blocks, 256, 0, (hipStream_t)stream>>>(list);
    if (int rc = ccheck("lbm3d_conv3d_wpack")) return rc;
  }
  return LBM3D_OK;
}

}  // namespace

extern "C" {

const char *lbm3d_conv_last_error(void) { return c_err; }

int32_t lbm3d_conv_kpad(int32_t cin, int32_t ks) {
  if (cin < 1 || (ks != 1 && ks != 3)) return 0;
  const int32_t k = ks * ks * ks * cin;
  return (k + 31) / 32 * 32;
}

int lbm3d_conv3d_fwd(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, uint16_t *y, int32_t n,
                     int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks, int32_t flags) {
  int rc = check_conv(n, d, h, wd, cin, cout, ks);
  if (rc) return rc;
  if (!x || !w || !y) return cfail(LBM3D_EINVAL, "NULL tensor");
  if (flags & ~(LBM3D_CONV_RELU | LBM3D_CONV_PERIODIC)) return cfail(LBM3D_EINVAL, "unknown flag bits");
  const int relu = (flags & LBM3D_CONV_RELU) ? 1 : 0;
  const Vol vol = make_vol(n, d, h, wd, (flags & LBM3D_CONV_PERIODIC) ? 1 : 0);
  const int kpad = lbm3d_conv_kpad(cin, ks);
  hipStream_t s = (hipStream_t)stream;
  if (ks == 3) {
    if ((rc = check_start(x, w))) return rc;
    return launch_conv3<kPlain>(s, ConvCall{x, w, 0, bias, y, vol, cin, cout, kpad, relu, ConvExtra{}});
  }
  const unsigned gx = (vol.vox + 255u) / 256u;
  if (cout % 64 == 0)
    k_conv1<4><<<dim3(gx, cout / 64), 256, 0, s>>>(x, w, bias, y, vol.vox, cin, cout, kpad, relu);
  else if (cout % 32 == 0)
    k_conv1<2><<<dim3(gx, cout / 32), 256, 0, s>>>(x, w, bias, y, vol.vox, cin, cout, kpad, relu);
  else
    k_conv1<1><<<dim3(gx, cout / 16), 256, 0, s>>>(x, w, bias, y, vol.vox, cin, cout, kpad, relu);
  return ccheck("lbm3d_conv3d_fwd");
}

int64_t lbm3d_conv3d_packed_elements(int32_t cin, int32_t cout) {
  if (check_conv(1, 1, 1, 1, cin, cout, 3)) return 0;
  return (int64_t)kSteps * 2 * cin * cout;
}

int lbm3d_conv3d_wpack_many(void *stream, int32_t count, const lbm3d_conv_pack *layers) {
  return wpack<float>(stream, count, layers);
}

int lbm3d_conv3d_wpack(void *stream, const float *w, uint16_t *wp, uint16_t *wt, int32_t cin, int32_t cout) {
  const lbm3d_conv_pack one{w, wp, wt, cin, cout};
  return wpack<float>(stream, 1, &one);
}

int lbm3d_conv3d_wpack_bf16(void *stream, const uint16_t *w, uint16_t *wp, uint16_t *wt, int32_t cin, int32_t cout) {
  const lbm3d_conv_pack one{reinterpret_cast<const float *>(w), wp, wt, cin, cout};  // read as the BF16 it is
  return wpack<uint16_t>(stream, 1, &one);
}

static int packed_call(const uint16_t *x, const uint16_t *wp, const float *bias, uint16_t *y, int32_t n, int32_t d,
                       int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t flags, ConvCall &a) {
  int rc = check_conv(n, d, h, wd, cin, cout, 3);
  if (rc) return rc;
  if (!x || !wp || !y) return cfail(LBM3D_EINVAL, "NULL tensor");
  if ((rc = check_start(x))) return rc;
  if (flags & ~(LBM3D_CONV_RELU | LBM3D_CONV_PERIODIC)) return cfail(LBM3D_EINVAL, "unknown flag bits");
  a = ConvCall{x,   wp,   1, bias, y, make_vol(n, d, h, wd, (flags & LBM3D_CONV_PERIODIC) ? 1 : 0), cin, cout,
               lbm3d_conv_kpad(cin, 3), (flags & LBM3D_CONV_RELU) ? 1 : 0, ConvExtra{}};
  return LBM3D_OK;
}

int lbm3d_conv3d_fwd_packed(void *stream, const uint16_t *x, const uint16_t *wp, const float *bias, uint16_t *y,
                            int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t flags) {
  ConvCall a;
  if (int rc = packed_call(x, wp, bias, y, n, d, h, wd, cin, cout, flags, a)) return rc;
  return launch_conv3<kPlain>((hipStream_t)stream, a);
}

int lbm3d_conv3d_fwd_pool(void *stream, const uint16_t *x, const uint16_t *wp, const float *bias, uint16_t *y,
                          uint16_t *pool, int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout,
                          int32_t flags) {
  ConvCall a;
  if (int rc = packed_call(x, wp, bias, y, n, d, h, wd, cin, cout, flags, a)) return rc;
  if (!pool) return cfail(LBM3D_EINVAL, "NULL tensor");
  if (!a.relu) return cfail(LBM3D_EINVAL, "pooling goes with LBM3D_CONV_RELU");
  if ((d | h | wd) & 1) return cfail(LBM3D_EINVAL, "pooling needs even extents");
  a.ex.pool = pool;
  return launch_conv3<kPool>((hipStream_t)stream, a);
}

int lbm3d_conv3d_fwd_up(void *stream, const uint16_t *low, const uint16_t *skip, const uint16_t *wp,
                        const float *bias, uint16_t *y, int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low,
                        int32_t c_skip, int32_t cout, int32_t flags) {
  if (c_low < 16 || c_low % 16 || c_skip < 16 || c_skip % 16 || c_low > 240 || c_skip > 240)
    return cfail(LBM3D_EINVAL, "channel counts must be multiples of 16, together at most 256");
  ConvCall a;
  if (int rc = packed_call(skip, wp, bias, y, n, d, h, wd, c_low + c_skip, cout, flags, a)) return rc;
  if (!low) return cfail(LBM3D_EINVAL, "NULL tensor");
  if (int rc = check_start(low)) return rc;
  if ((d | h | wd) & 1) return cfail(LBM3D_EINVAL, "upsampling needs even extents");
  a.ex.low = low;
  a.ex.c_low = c_low;
  return launch_conv3<kUp>((hipStream_t)stream, a);
}

int lbm3d_conv3d_dgrad_up(void *stream, const uint16_t *dy, const uint16_t *wt, uint16_t *d_low, uint16_t *d_skip,
                          int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low, int32_t c_skip, int32_t cout) {
  if (c_low < 16 || c_low % 16 || c_skip < 16 || c_skip % 16 || c_low > 240 || c_skip > 240)
    return cfail(LBM3D_EINVAL, "channel counts must be multiples of 16, together at most 256");
  ConvCall a;
  if (int rc = packed_call(dy, wt, nullptr, d_skip, n, d, h, wd, cout, c_low + c_skip, 0, a)) return rc;
  if (!d_low) return cfail(LBM3D_EINVAL, "NULL tensor");
  if ((d | h | wd) & 1) return cfail(LBM3D_EINVAL, "upsampling needs even extents");
  a.ex.c_split = c_low;
  a.ex.y_hi = d_skip;
  a.ex.pool = d_low;
  return launch_conv3<kDown>((hipStream_t)stream, a);
}

int lbm3d_conv3d_wflip(void *stream, const uint16_t *w, uint16_t *wt, int32_t cin, int32_t cout, int32_t ks) {
  int rc = check_conv(1, 1, 1, 1, cin, cout, ks);
  if (rc) return rc;
  if (!w || !wt) return cfail(LBM3D_EINVAL, "NULL tensor");
  const int taps = ks * ks * ks;
  const int kin = lbm3d_conv_kpad(cin, ks), kout = lbm3d_conv_kpad(cout, ks);
  const int64_t total = (int64_t)cin * kout;
  k_wflip<<<(unsigned)((total + 255) / 256), 256, 0, (hipStream_t)stream>>>(w, wt, cin, cout, taps, kin, kout);
  return ccheck("lbm3d_conv3d_wflip");
}

int lbm3d_conv3d_dgrad(void *stream, const uint16_t *dy, const uint16_t *wt, uint16_t *dx, int32_t n, int32_t d,
                       int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks) {
  // a forward convolution from cout to cin channels with the flipped weights
  return lbm3d_conv3d_fwd(stream, dy, wt, nullptr, dx, n, d, h, wd, cout, cin, ks, 0);
}

size_t lbm3d_conv3d_wgrad_workspace_bytes(int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout,
                                          int32_t ks) {
  if (check_conv(n, d, h, wd, cin, cout, ks)) return 0;
  uint32_t per;
  return (size_t)wgrad_plan(make_bricks(n, d, h, wd), cin, cout, per) * wgrad_sets(ks) * cout *
         lbm3d_conv_kpad(cin, ks) * sizeof(float);
}

// a weight gradient and its fold; low / c_low: the upsampled part of x, if any
static int wgrad_run(void *stream, const uint16_t *x, const uint16_t *dy, float *dw, int32_t n, int32_t d, int32_t h,
                     int32_t wd, int32_t cin, int32_t cout, int32_t ks, void *workspace, size_t workspace_bytes,
                     const uint16_t *low, int c_low) {
  int rc = check_conv(n, d, h, wd, cin, cout, ks);
  if (rc) return rc;
  if (!x || !dy || !dw || !workspace || (c_low > 0 && !low)) return cfail(LBM3D_EINVAL, "NULL tensor or workspace");
  if ((rc = check_start(x, dy, low))) return rc;
  if (workspace_bytes < lbm3d_conv3d_wgrad_workspace_bytes(n, d, h, wd, cin, cout, ks))
    return cfail(LBM3D_EINVAL, "wgrad workspace too small");
  const Vol vol = make_vol(n, d, h, wd);
  hipStream_t s = (hipStream_t)stream;
  const Bricks bk = make_bricks(n, d, h, wd);
  uint32_t per;
  const int sets = wgrad_plan(bk, cin, cout, per), kpad = lbm3d_conv_kpad(cin, ks);
  float *part = (float *)workspace;
  if (ks == 1) {
    const uint32_t tiles = (uint32_t)((cout / 16) * (cin / 16)), jobs = (uint32_t)sets * tiles;
    k_wgrad1<<<(unsigned)xcd_grid(jobs, LBM3D_CONV_WGRAD_XCD_CHUNK), 256, 0, s>>>(x, dy, part, vol, cin, cout, kpad, bk,
                                                                              per, jobs, make_div(tiles));
  } else {
    // two output channel tiles a workgroup where there are, which share the staged x
    const int wco = cout % 32 == 0 ? 2 : 1;
    const uint32_t tiles = (uint32_t)((cout / (16 * wco)) * (cin / 16)), jobs = (uint32_t)sets * tiles;
    const unsigned grid = (unsigned)xcd_grid(jobs, LBM3D_CONV_WGRAD_XCD_CHUNK);
    const Div td = make_div(tiles);
#define LBM3D_WGRAD3(O, U) \
  k_wgrad3<O, U><<<grid, 192 * (O), 0, s>>>(x, dy, part, vol, cin, cout, kpad, bk, per, jobs, td, low, c_low)
    if (wco == 2) {
      if (c_low > 0) LBM3D_WGRAD3(2, true);
      else LBM3D_WGRAD3(2, false);
    } else {
      if (c_low > 0) LBM3D_WGRAD3(1, true);
      else LBM3D_WGRAD3(1, false);
    }
#undef LBM3D_WGRAD3
  }
  if ((rc = ccheck("lbm3d_conv3d_wgrad"))) return rc;
  return fold_sets(s, part, dw, (int64_t)cout * kpad, sets * wgrad_sets(ks), kpad, ks * ks * ks * cin);
}

int lbm3d_conv3d_wgrad(void *stream, const uint16_t *x, const uint16_t *dy, float *dw, int32_t n, int32_t d, int32_t h,
                       int32_t wd, int32_t cin, int32_t cout, int32_t ks, void *workspace, size_t workspace_bytes) {
  return wgrad_run(stream, x, dy, dw, n, d, h, wd, cin, cout, ks, workspace, workspace_bytes, nullptr, 0);
}

int lbm3d_conv3d_wgrad_up(void *stream, const uint16_t *low, const uint16_t *skip, const uint16_t *dy, float *dw,
                          int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low, int32_t c_skip, int32_t cout,
                          void *workspace, size_t workspace_bytes) {
  if (c_low < 16 || c_low % 16 || c_skip < 16 || c_skip % 16 || c_low > 240 || c_skip > 240)
    return cfail(LBM3D_EINVAL, "channel counts must be multiples of 16, together at most 256");
  if ((d | h | wd) & 1) return cfail(LBM3D_EINVAL, "upsampling needs even extents");
  return wgrad_run(stream, skip, dy, dw, n, d, h, wd, c_low + c_skip, cout, 3, workspace, workspace_bytes, low, c_low);
}

size_t lbm3d_relu_bias_grad_workspace_bytes(int64_t voxels, int32_t c) {
  if (voxels < 1 || c < 8 || c > 256 || 2048 % c) return 0;
  int64_t chunks, per;
  return (size_t)relu_bias_plan(voxels, c, chunks, per) * c * sizeof(float);
}

int lbm3d_relu_bias_grad(void *stream, const uint16_t *g, const uint16_t *y, uint16_t *dz, float *db, int64_t voxels,
                         int32_t c, void *workspace, size_t workspace_bytes) {
  if (voxels < 1) return cfail(LBM3D_EINVAL, "no voxels");
  if (c < 8 || c > 256 || 2048 % c) return cfail(LBM3D_EINVAL, "channels must divide 2048, 8..256");
  if (!g || !dz || !db || !workspace) return cfail(LBM3D_EINVAL, "NULL tensor or workspace");
  if (workspace_bytes < lbm3d_relu_bias_grad_workspace_bytes(voxels, c))
    return cfail(LBM3D_EINVAL, "relu/bias workspace too small");
  int64_t chunks, per;
  const int blocks = relu_bias_plan(voxels, c, chunks, per);
  hipStream_t s = (hipStream_t)stream;
  k_relu_bias_grad<kGradPlain><<<(unsigned)blocks, 256, 0, s>>>(g, y, dz, (float *)workspace, chunks, c, per, PoolGrad{});
  if (int rc = ccheck("lbm3d_relu_bias_grad")) return rc;
  return fold_sets(s, (float *)workspace, db, c, blocks, c, c);
}

int lbm3d_conv_head_fwd(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, float *out,
                        int64_t voxels, int32_t cin) {
  if (voxels < 1 || cin < 16 || cin > 256 || cin % 16) return cfail(LBM3D_EINVAL, "bad head shape");
  if (voxels >= ((int64_t)1 << 31)) return cfail(LBM3D_ESIZE, "more than 2^31-1 voxels");
  if (!x || !w || !out) return cfail(LBM3D_EINVAL, "NULL tensor");
  k_head<kHeadOut><<<(unsigned)((voxels + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      x, w, bias, out, (uint32_t)voxels, cin, lbm3d_conv_kpad(cin, 1), HeadFields{});
  return ccheck("lbm3d_conv_head_fwd");
}

int lbm3d_conv_head_fields(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, const int8_t *solid,
                           float *rho, float *v, const int32_t extents[3], const int32_t origin[3],
                           const int32_t core[3], int32_t cin, float scale_v, float scale_rho, int rho_one) {
  if (!x || !w || !solid || !rho || !v || !extents || !origin || !core) return cfail(LBM3D_EINVAL, "NULL tensor");
  if (cin < 16 || cin > 256 || cin % 16) return cfail(LBM3D_EINVAL, "bad head shape");
  for (int a = 0; a < 3; ++a)
    if (core[a] < 1 || origin[a] < 0 || extents[a] < 1 || origin[a] > extents[a] - core[a])
      return cfail(LBM3D_EINVAL, "the box does not lie in the volume");
  const int64_t vox = (int64_t)core[0] * core[1] * core[2];
  if (vox >= ((int64_t)1 << 31)) return cfail(LBM3D_ESIZE, "more than 2^31-1 voxels");
  const int64_t first = ((int64_t)origin[0] * extents[1] + origin[1]) * extents[2] + origin[2];
  const HeadFields hf{make_vol(1, core[0], core[1], core[2]), extents[1], extents[2], first, solid, scale_v, scale_rho,
                      rho_one, rho, v};
  k_head<kHeadFields><<<(unsigned)((vox + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      x, w, bias, nullptr, (uint32_t)vox, cin, lbm3d_conv_kpad(cin, 1), hf);
  return ccheck("lbm3d_conv_head_fields");
}

int lbm3d_conv_head_grad(void *stream, const float *g, uint16_t *dz, float *db, int64_t voxels, void *workspace,
                         size_t workspace_bytes) {
  if (voxels < 1) return cfail(LBM3D_EINVAL, "no voxels");
  if (!g || !dz || !db || !workspace) return cfail(LBM3D_EINVAL, "NULL tensor or workspace");
  if (workspace_bytes < lbm3d_relu_bias_grad_workspace_bytes(voxels, 16))
    return cfail(LBM3D_EINVAL, "head gradient workspace too small");
  int64_t chunks, per;
  const int blocks = relu_bias_plan(voxels, 16, chunks, per);
  hipStream_t s = (hipStream_t)stream;
  k_relu_bias_grad<kGradHead><<<(unsigned)blocks, 256, 0, s>>>(reinterpret_cast<const uint16_t *>(g), nullptr, dz,
                                                               (float *)workspace, chunks, 16, per, PoolGrad{});
  if (int rc = ccheck("lbm3d_conv_head_grad")) return rc;
  return fold_sets(s, (float *)workspace, db, 16, blocks, 16, 16);
}

int lbm3d_relu_pool_grad(void *stream, const uint16_t *g, const uint16_t *y, const uint16_t *pooled,
                         const uint16_t *g_pool, uint16_t *dz, float *db, int32_t n, int32_t d, int32_t h, int32_t w,
                         int32_t c, uint16_t *share, void *workspace, size_t workspace_bytes) {
  if (n < 1 || d < 1 || h < 1 || w < 1 || ((d | h | w) & 1)) return cfail(LBM3D_EINVAL, "extents must be even");
  if (c < 8 || c > 256 || 2048 % c) return cfail(LBM3D_EINVAL, "channels must divide 2048, 8..256");
  if (!g || !y || !pooled || !g_pool || !dz || !db || !share || !workspace)
    return cfail(LBM3D_EINVAL, "NULL tensor or workspace");
  const int64_t voxels = (int64_t)n * d * h * w;
  if (voxels >= ((int64_t)1 << 31)) return cfail(LBM3D_ESIZE, "more than 2^31-1 voxels");
  if (workspace_bytes < lbm3d_relu_bias_grad_workspace_bytes(voxels, c))
    return cfail(LBM3D_EINVAL, "relu/bias workspace too small");
  hipStream_t s = (hipStream_t)stream;
  const Div pieces = make_div((uint32_t)c / 8);
  const int64_t low = voxels / 8 * (c / 8);
  k_pool_share<<<(unsigned)((low + 255) / 256), 256, 0, s>>>(y, pooled, g_pool, share,
                                                            make_vol(n, d / 2, h / 2, w / 2), pieces, low);
  if (int rc = ccheck("lbm3d_relu_pool_grad")) return rc;
  int64_t chunks, per;
  const int blocks = relu_bias_plan(voxels, c, chunks, per);
  k_relu_bias_grad<kGradPool><<<(unsigned)blocks, 256, 0, s>>>(g, y, dz, (float *)workspace, chunks, c, per,
                                                         PoolGrad{pooled, share, make_vol(n, d, h, w), pieces});
  if (int rc = ccheck("lbm3d_relu_pool_grad")) return rc;
  return fold_sets(s, (float *)workspace, db, c, blocks, c, c);
}

static int distance_passes(void *stream, const int8_t *solid, void *out, int mode, float *work, int32_t n, int32_t d,
                           int32_t h, int32_t w, int32_t margin, float inv_scale, float *second) {
  if (n < 1 || d < 1 || h < 1 || w < 1) return cfail(LBM3D_EINVAL, "empty volume");
  if (margin < 1 || margin > 1024) return cfail(LBM3D_EINVAL, "margin must be 1..1024");
  if (!solid || !out || !work || !second) return cfail(LBM3D_EINVAL, "NULL tensor");
  DistGeo gm;
  gm.total = (int64_t)n * d * h * w;
  gm.d0 = d;
  gm.d1 = h;
  gm.d2 = w;
  gm.div0 = make_div((uint32_t)d);
  gm.div1 = make_div((uint32_t)h);
  gm.div2 = make_div((uint32_t)w);
  gm.margin = margin;
  gm.inv_scale = inv_scale;
  hipStream_t s = (hipStream_t)stream;
  const unsigned grid = (unsigned)((gm.total + 255) / 256);
  const int64_t segs = ((int64_t)w + 63) / 64, most = (int64_t)(UINT32_MAX / (64u * kDistWaves));
  const Div dsegs = make_div((uint32_t)segs);
  // a pass cannot run in place: it reads values that other threads overwrite
  if (margin < 64 && h <= kDistLine && (int64_t)n * d * segs <= most) {
    k_dist_lines<1, 0><<<(unsigned)(n * d * segs), 64 * kDistWaves, 256 * h, s>>>(solid, nullptr, work, gm, dsegs);
  } else {
    const int64_t rows = (int64_t)n * d * h, blocks = (rows * segs + 3) / 4;
    if (margin < 64 && blocks <= (int64_t)(UINT32_MAX / 256u))
      k_dist_rows<<<(unsigned)blocks, 256, 0, s>>>(solid, second, gm, dsegs, rows * segs);
    else
      k_dist_axis<2, 0><<<grid, 256, 0, s>>>(solid, nullptr, second, gm);
    k_dist_axis<1, 0><<<grid, 256, 0, s>>>(solid, second, work, gm);
  }
  if (int rc = ccheck("lbm3d_distance_periodic")) return rc;
  const bool lines = d <= kDistLine && (int64_t)n * h * segs <= most;
  auto outer = [&](auto m) {
    constexpr int kOut = decltype(m)::value;
    if (lines)
      k_dist_lines<0, kOut><<<(unsigned)(n * h * segs), 64 * kDistWaves, 256 * d, s>>>(solid, work, out, gm, dsegs);
    else
      k_dist_axis<0, kOut><<<grid, 256, 0, s>>>(solid, work, out, gm);
  };
  if (mode == kDistNet) outer(std::integral_constant<int, kDistNet>{});
  else if (mode == kDistPair) outer(std::integral_constant<int, kDistPair>{});
  else outer(std::integral_constant<int, kDistPlain>{});
  return ccheck("lbm3d_distance_periodic");
}

int lbm3d_distance_periodic(void *stream, const int8_t *solid, float *dist, float *work, int32_t n, int32_t d,
                            int32_t h, int32_t w, int32_t margin) {
  return distance_passes(stream, solid, dist, kDistPlain, work, n, d, h, w, margin, 1.f, dist);
}

int lbm3d_surrogate_inputs(void *stream, const int8_t *solid, void *out, int network, float scale, float *work,
                           int32_t n, int32_t d, int32_t h, int32_t w, int32_t margin) {
  int e = 0;
  if (!(scale > 0.f) || frexpf(scale, &e) != 0.5f) return cfail(LBM3D_EINVAL, "scale must be a power of two");
  if (!out || !work) return cfail(LBM3D_EINVAL, "NULL tensor");
  // the first pass's result goes to the second half of work
  float *second = work + (int64_t)n * d * h * w;
  return distance_passes(stream, solid, out, network ? kDistNet : kDistPair, work, n, d, h, w, margin, 1.f / scale,
                         second);
}

}  // extern "C"
