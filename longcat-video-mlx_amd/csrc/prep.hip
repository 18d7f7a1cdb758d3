// Pre-BSA preparation of q and k in one pass: per-head RMSNorm (fp32 math),
// 3D RoPE, and the block means the routing needs.
//
// Follows the attention layer ahead of BSA (longcat_video/models/attention.py:
// 191-201):
//   q = RMSNorm_FP32(q)  -- blocks.py:55-72: x_f32 * rsqrt(mean(x_f32^2) + eps),
//                           rounded to the input dtype, times the weight in
//                           that dtype;
//   q = rope_3d(q)       -- rope_3d.py:107-128: widened to fp32,
//                           x*cos + rotate_half(x)*sin, rounded back;
// (the same for k), followed by mean_pool_blocks_3d of the result
// (block_sparse_attention.py:67-104).  The reference runs these as separate
// full-tensor passes; here one wave reads each row of a block once, writes
// the prepared row and accumulates the block mean of the written values.
//
// RoPE angles come from a per-axis table built by the caller (cos and sin of
// position * inverse frequency for the t, h and w parts of the head dim),
// staged in LDS once per (persistent) workgroup.  The RoPE grid is the latent grid; the
// BSA blocks may be a different view of the same tokens (e.g. contiguous
// 64-token blocks), so the two geometries are separate arguments.
#include <algorithm>

#include "norm_common.h"

namespace lcv {
namespace {

constexpr int kPrepWaves = 4;

struct PrepArgs {
  Tensor4 in[2];
  Tensor4 out[2];
  const void* weight[2];  // [D] in the tensor dtype, or null (weight 1)
  float* mean[2];         // [B, H, nb, D] fp32
  const float* table;     // cos_t, sin_t, cos_h, sin_h, cos_w, sin_w
  int32_t H, D, nb;
  int32_t rT, rH, rW;     // RoPE grid
  int32_t dt, dh;         // RoPE dims of the t and h parts (w takes the rest)
  int32_t table_len;
  int32_t total_items;
  float eps;
  float rcp_plane, rcp_w;  // 1 / (rH * rW), 1 / rW
  float neg_zero, one;     // -0.0f and 1.0f (FMA operands the compiler cannot fold)
  Geom g;
  FastDiv per_block;      // 2 * B * H: items per BSA block index
  FastDiv heads;          // H
};

// The cached form (prep_cached_kernel): k and v continue a cache of earlier
// tokens, already normed and not yet rotated.
struct CachedArgs {
  PrepArgs p;             // in / out / weight / mean of q (0) and new k (1); g is q's geometry
  Tensor4 cache[2];       // k, v of the cached tokens
  Tensor4 v_in, v_out;    // new v, and cached + new v (null: v is not gathered)
  Tensor4 k_norm;         // new k after its norm, before RoPE (null: not wanted)
  int32_t cached;         // tokens in the cache
  int32_t nk;             // blocks of k / v (cached + new)
  int32_t head_items;     // items before the first q-block's
  FastDiv head_per_block, bh;  // items per block among those, B * H
  Geom gk;
};

// Quotient of n by d for n < 2^22 from an fp32 reciprocal: (n + 1/2) / d is
// at least 1/(2d) away from an integer, more than the rounding error of
// (n + 1/2) * fl(1/d) (under 2^-23 relative) can cover for n < 2^22.
__device__ __forceinline__ uint32_t small_div(uint32_t n, float rcp) {
  return (uint32_t)__builtin_fmaf((float)n, rcp, 0.5f * rcp);
}

// The table as staged in LDS: per axis, (cos, sin) interleaved per column, so
// a pair's two factors are one 8-byte read.  Axis a's region starts where its
// cos part starts in the caller's layout (the regions have the same sizes).
__device__ __forceinline__ int lds_slot(const PrepArgs& a, int i) {
  const int ht = a.dt / 2, hh = a.dh / 2, hw = (a.D - a.dt - a.dh) / 2;
  const int nt = a.rT * ht, nh = a.rH * hh, nw = a.rW * hw;
  int base = 0, n = nt;
  if (i >= 2 * nt + 2 * nh) {
    base = 2 * nt + 2 * nh;
    n = nw;
  } else if (i >= 2 * nt) {
    base = 2 * nt;
    n = nh;
  }
  const int j = i - base;
  return j < n ? base + 2 * j : base + 2 * (j - n) + 1;
}

// What a lane needs to turn rows: per pair p (dims 8c + 2p, +1) its axis and its
// column's byte offset in that axis' LDS row.
template <int D>
struct RopeLane {
  int axis[4], col[4];
  __device__ RopeLane(const PrepArgs& a, int c) {
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      const int d = 8 * c + 2 * pp;
      axis[pp] = d < a.dt ? 0 : (d < a.dt + a.dh ? 1 : 2);
      col[pp] = 4 * (axis[pp] == 0 ? d : (axis[pp] == 1 ? d - a.dt : d - a.dt - a.dh));
    }
  }
};

// Where the LDS rows of grid position `tok` start, per axis, in (cos, sin) pairs
// (below kMaxRopeTable / 2).  One lane per row of a block computes it, for the D / 8
// lanes that turn the row (each of them for itself, and with unpacked bf16
// rounding, a step was 215 to 269 instructions, now 156 to 164, and the VALU the
// bound beside HBM): filling a cache of 28,800 tokens x 32 heads x 128 263 -> 230 us
// (5.1 TB/s); D = 64, 20,480 x 16: q and k 40.3 -> 35.0 us, around a cache 79 -> 67.
struct RopePos {
  uint16_t slot[4];
};
__device__ __forceinline__ RopePos rope_pos(const PrepArgs& a, uint32_t tok) {
  const uint32_t ht = (uint32_t)a.dt / 2, hh = (uint32_t)a.dh / 2, hw = (uint32_t)(a.D - a.dt - a.dh) / 2;
  const uint32_t pt = small_div(tok, a.rcp_plane);
  const uint32_t prem = tok - __umul24(pt, (uint32_t)(a.rH * a.rW));
  const uint32_t ph = small_div(prem, a.rcp_w);
  const uint32_t pw = prem - __umul24(ph, (uint32_t)a.rW);
  const uint32_t reg_h = (uint32_t)a.rT * ht, reg_w = reg_h + (uint32_t)a.rH * hh;
  return RopePos{{(uint16_t)__umul24(pt, ht), (uint16_t)(reg_h + __umul24(ph, hh)),
                  (uint16_t)(reg_w + __umul24(pw, hw)), 0}};
}

template <typename T>
__device__ __forceinline__ u32x4 load_weight(const void* w, int c) {
  if (w) return *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(w) + 8 * c);
  const uint32_t one = bits16(from_f32<T>(1.0f));
  return u32x4{one | (one << 16), one | (one << 16), one | (one << 16), one | (one << 16)};
}

// RMSNorm of a row held 8 elements a lane over D / 8 lanes.
template <typename T, int D>
__device__ __forceinline__ void norm_row(const float (&x)[8], const u32x4& wr, float eps, float nz, float (&y)[8]) {
  float ss = 0.0f;
#pragma unroll
  // x*x of a 16-bit value is exact in fp32, so the fused form rounds the
  // sum exactly as square-then-add does.
  for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(x[e], x[e], ss);
  ss = group_sum<D / 8>(ss);
  const float rs = rsqrtf(ss * (1.0f / D) + eps);
  norm_scale<T>(x, rs, wr, nz, y);
}

// RoPE of y at the position whose slots are `pos`; the rounded row is packed and
// added to acc.
template <typename T, int D>
__device__ __forceinline__ u32x4 rope_row(const PrepArgs& a, const RopeLane<D>& L, const float* tab,
                                          const RopePos& pos, const float (&y)[8], float (&acc)[8]) {
  const float nz = a.neg_zero, one = a.one;
  uint32_t packed[4];
#pragma unroll
  for (int pp = 0; pp < 4; ++pp) {
    const float2 f = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(tab) +
                                                      (8 * (int)pos.slot[L.axis[pp]] + L.col[pp]));
    const float cs = f.x, sn = f.y;
    const float u = y[2 * pp], v = y[2 * pp + 1];
    // x*cos + rotate_half(x)*sin, rounded per product and sum.
    packed[pp] = round_pair<T>(mul1(u, cs, nz) - mul1(v, sn, nz), mul1(v, cs, nz) + mul1(u, sn, nz));
    const T o0 = __builtin_bit_cast(T, (uint16_t)(packed[pp] & 0xffffu));
    const T o1 = __builtin_bit_cast(T, (uint16_t)(packed[pp] >> 16));
    acc[2 * pp] = __builtin_fmaf(to_f32(o0), one, acc[2 * pp]);
    acc[2 * pp + 1] = __builtin_fmaf(to_f32(o1), one, acc[2 * pp + 1]);
  }
  return u32x4{packed[0], packed[1], packed[2], packed[3]};
}

// Block mean: combine the row groups (lanes c, c + LPR, ...) in a fixed
// butterfly order; the lanes of group 0 store the D means.
template <int D>
__device__ __forceinline__ void store_mean(float (&acc)[8], float* mean, int lane) {
  constexpr int LPR = D / 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
#pragma unroll
    for (int m = LPR; m < 64; m <<= 1) acc[e] += __shfl_xor(acc[e], m);
  }
  if (lane < LPR) {
    float* mp = mean + 8 * lane;
    constexpr float inv = 1.0f / 64.0f;
    *reinterpret_cast<float4*>(mp) = float4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    *reinterpret_cast<float4*>(mp + 4) = float4{acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv};
  }
}

// Row loads in flight per lane and waves per SIMD at least.  D = 128: 2 and 6 (4 and 4
// gave 380 against 380 us for q, k of 57,600 tokens x 32 heads, 198 / 194 us at
// 28,800, 398 / 387 us around a cache); D = 64: 4 and 4 (34.5 against 35.8 us at
// 20,480 x 16, 67 / 73 us around a cache).
template <int D>
struct PrepTune {
  static constexpr int kBatch = D == 128 ? 2 : 4, kWaves = D == 128 ? 6 : 4;
};

// Lane l's slots to row l of this wave's table.  LDS operations of one wave complete
// in order; the fences keep the compiler from moving reads across.
__device__ __forceinline__ void set_pos(RopePos* pos, int lane, const RopePos& v) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  pos[lane] = v;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <typename T, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PrepTune<D>::kWaves))) void prep_kernel(PrepArgs a) {
  constexpr int LPR = D / 8;       // lanes per row (8 elements per lane)
  constexpr int RPS = 64 / LPR;    // rows per step
  constexpr int kPrepBatch = PrepTune<D>::kBatch;
  extern __shared__ float tab[];  // table_len floats (dynamic)
  __shared__ int64_t row_in[2][64], row_out[2][64];  // element offset of each block row
  __shared__ RopePos pos[kPrepWaves][64];            // of a wave's block rows

  // The workgroup is persistent: the table and the row offsets are staged
  // once and its waves then walk the (block, tensor, b, h) items with a
  // grid-wide stride.
  for (int i = threadIdx.x; i < a.table_len; i += 256) tab[lds_slot(a, i)] = a.table[i];
  if (threadIdx.x < 64) {
    const int32_t t = voxel_row_offset(a.g, threadIdx.x);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      row_in[k][threadIdx.x] = (int64_t)t * a.in[k].ss;
      row_out[k][threadIdx.x] = (int64_t)t * a.out[k].ss;
    }
  }
  __syncthreads();

  const int wave = uniform_i32(threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  const int c = lane % LPR;  // this lane's 8 dims: 8c .. 8c+7
  const RopeLane<D> L(a, c);
  const uint32_t lane_tok = (uint32_t)voxel_row_offset(a.g, lane);
  const int stride = gridDim.x * kPrepWaves;

  for (int item = blockIdx.x * kPrepWaves + wave; item < a.total_items; item += stride) {
    // Items run head-fastest, so the waves resident together read the q and k
    // heads of the same tokens (adjacent in a fused QKV buffer).
    const uint32_t n = fast_div((uint32_t)item, a.per_block);
    const uint32_t r = (uint32_t)item - n * a.per_block.d;
    const uint32_t bt = fast_div(r, a.heads);
    const int h = (int)(r - bt * a.heads.d);
    const int tensor = (int)(bt & 1u);
    const int b = (int)(bt >> 1);
    const int bh = b * a.H + h;
    const int32_t tok0 = block_base_token(a.g, (int32_t)n);
    const Tensor4 xi = a.in[tensor];
    const Tensor4 xo = a.out[tensor];
    const T* src = reinterpret_cast<const T*>(xi.ptr) + (int64_t)b * xi.sb + (int64_t)h * xi.sh +
                   (int64_t)tok0 * xi.ss + 8 * c;
    T* dst = reinterpret_cast<T*>(const_cast<void*>(xo.ptr)) + (int64_t)b * xo.sb + (int64_t)h * xo.sh +
             (int64_t)tok0 * xo.ss + 8 * c;
    const u32x4 wr = load_weight<T>(a.weight[tensor], c);
    set_pos(pos[wave], lane, rope_pos(a, (uint32_t)tok0 + lane_tok));

    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
#pragma unroll 1
    for (int s0 = 0; s0 < 64 / RPS; s0 += kPrepBatch) {
      // q / k are streamed once: non-temporal loads and stores.
      u32x4 raw[kPrepBatch];
#pragma unroll
      for (int u = 0; u < kPrepBatch; ++u)
        raw[u] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4*>(src + row_in[tensor][(s0 + u) * RPS + lane / LPR]));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kPrepBatch; ++u) {
        const int row = (s0 + u) * RPS + lane / LPR;
        float x[8], y[8];
        widen8<T>(raw[u], x);
        norm_row<T, D>(x, wr, a.eps, a.neg_zero, y);
        const u32x4 packed = rope_row<T, D>(a, L, tab, pos[wave][row], y, acc);
        __builtin_nontemporal_store(packed, reinterpret_cast<u32x4*>(dst + row_out[tensor][row]));
      }
    }
    store_mean<D>(acc, a.mean[tensor] + ((int64_t)bh * a.nb + n) * D, lane);
  }
}

// prep_kernel with q and k of different lengths: k (and v) rows below `cached`
// come from the cache, k's un-normed; RoPE positions run over cached + new
// tokens, so new row r of q and k sits at cached + r.  q is read once, cached and
// new k once, and nothing is padded, concatenated or rotated in between.  Items
// run k-block (v-block) by k-block; the last nb of the nk k-blocks go with the
// q-blocks, so that the rows of a token that q, k and v share are read together.
// HBM bound, as prep_kernel.  Measured at 32 heads of 128, bf16, 3,600 tokens a
// frame: 8 frames after 4 cached ones 1.89 GB in 0.39 ms, 4.9 TB/s (the torch
// norms, concatenations and RoPE it replaces: 7.3 ms); filling a cache of 4
// frames 0.59 GB in 0.14 ms (2.3 ms).
template <typename T, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PrepTune<D>::kWaves))) void prep_cached_kernel(CachedArgs ca) {
  constexpr int LPR = D / 8;
  constexpr int RPS = 64 / LPR;
  constexpr int kPrepBatch = PrepTune<D>::kBatch;
  extern __shared__ float tab[];
  __shared__ int32_t row_tok[2][64];       // token offset of each block row: q's geometry, k's
  __shared__ RopePos pos[kPrepWaves][64];  // of a wave's block rows
  const PrepArgs& a = ca.p;
  for (int i = threadIdx.x; i < a.table_len; i += 256) tab[lds_slot(a, i)] = a.table[i];
  if (threadIdx.x < 64) {
    row_tok[0][threadIdx.x] = voxel_row_offset(a.g, threadIdx.x);
    row_tok[1][threadIdx.x] = voxel_row_offset(ca.gk, threadIdx.x);
  }
  __syncthreads();
  const int wave = uniform_i32(threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  const int c = lane % LPR;
  const RopeLane<D> L(a, c);
  const int stride = gridDim.x * kPrepWaves;

  for (int item = blockIdx.x * kPrepWaves + wave; item < a.total_items; item += stride) {
    int tensor, n;   // 0 q, 1 k, 2 v; its block
    uint32_t r;
    if (item < ca.head_items) {
      n = (int)fast_div((uint32_t)item, ca.head_per_block);
      r = (uint32_t)item - (uint32_t)n * ca.head_per_block.d;
      tensor = 1 + (int)fast_div(r, ca.bh);
      r -= (uint32_t)(tensor - 1) * ca.bh.d;
    } else {
      const uint32_t it = (uint32_t)(item - ca.head_items);
      n = (int)fast_div(it, a.per_block);
      r = it - (uint32_t)n * a.per_block.d;
      tensor = (int)fast_div(r, ca.bh);
      r -= (uint32_t)tensor * ca.bh.d;
      if (tensor) n += ca.nk - a.nb;
    }
    const int bh = (int)r;
    const int b = (int)fast_div(r, a.heads);
    const int h = bh - b * (int)a.heads.d;
    const int32_t tok0 = block_base_token(tensor ? ca.gk : a.g, n);
    const Tensor4 xi = tensor == 2 ? ca.v_in : a.in[tensor];
    const Tensor4 xo = tensor == 2 ? ca.v_out : a.out[tensor];
    const Tensor4 xc = ca.cache[tensor == 2 ? 1 : 0];
    const int first_new = tensor ? ca.cached : 0;  // rows below come from the cache
    const T* src = reinterpret_cast<const T*>(xi.ptr) + (int64_t)b * xi.sb + (int64_t)h * xi.sh + 8 * c;
    const T* old = reinterpret_cast<const T*>(xc.ptr) + (int64_t)b * xc.sb + (int64_t)h * xc.sh + 8 * c;
    T* dst = reinterpret_cast<T*>(const_cast<void*>(xo.ptr)) + (int64_t)b * xo.sb + (int64_t)h * xo.sh + 8 * c;
    const int32_t* rows = row_tok[tensor ? 1 : 0];
    if (tensor == 2) {
#pragma unroll 4
      for (int st = 0; st < 64 / RPS; ++st) {
        const int32_t t = tok0 + rows[st * RPS + lane / LPR];
        const T* from = t < first_new ? old + (int64_t)t * xc.ss : src + (int64_t)(t - first_new) * xi.ss;
        __builtin_nontemporal_store(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(from)),
                                    reinterpret_cast<u32x4*>(dst + (int64_t)t * xo.ss));
      }
      continue;
    }
    T* kn = tensor && ca.k_norm.ptr ? reinterpret_cast<T*>(const_cast<void*>(ca.k_norm.ptr)) +
                                          (int64_t)b * ca.k_norm.sb + (int64_t)h * ca.k_norm.sh + 8 * c
                                    : nullptr;
    const u32x4 wr = load_weight<T>(a.weight[tensor], c);
    set_pos(pos[wave], lane, rope_pos(a, (uint32_t)(tok0 + rows[lane] + (tensor ? 0 : ca.cached))));
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
#pragma unroll 1
    for (int s0 = 0; s0 < 64 / RPS; s0 += kPrepBatch) {
      u32x4 raw[kPrepBatch];
#pragma unroll
      for (int u = 0; u < kPrepBatch; ++u) {
        const int32_t t = tok0 + rows[(s0 + u) * RPS + lane / LPR];
        const T* from = t >= first_new ? src + (int64_t)(t - first_new) * xi.ss : old + (int64_t)t * xc.ss;
        raw[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(from));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kPrepBatch; ++u) {
        const int row = (s0 + u) * RPS + lane / LPR;
        const int32_t t = tok0 + rows[row];
        const bool is_new = t >= first_new;
        float x[8], y[8];
        widen8<T>(raw[u], x);
        norm_row<T, D>(x, wr, a.eps, a.neg_zero, y);
        if (kn && is_new) {
          uint32_t w[4];
#pragma unroll
          for (int m = 0; m < 4; ++m)  // exact: y holds T values
            w[m] = bits16(from_f32<T>(y[2 * m])) | (bits16(from_f32<T>(y[2 * m + 1])) << 16);
          *reinterpret_cast<u32x4*>(kn + (int64_t)(t - first_new) * ca.k_norm.ss) = u32x4{w[0], w[1], w[2], w[3]};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = is_new ? y[e] : x[e];
        const u32x4 packed = rope_row<T, D>(a, L, tab, pos[wave][row], y, acc);
        __builtin_nontemporal_store(packed, reinterpret_cast<u32x4*>(dst + (int64_t)t * xo.ss));
      }
    }
    store_mean<D>(acc, a.mean[tensor] + ((int64_t)bh * (tensor ? ca.nk : a.nb) + n) * D, lane);
  }
}

// As many workgroups as are resident at once (each stages the table once).
template <typename Args>
hipError_t launch_resident(void (*kernel)(Args), const Args& args, int table_len, int items, hipStream_t stream) {
  const size_t shmem = (size_t)table_len * sizeof(float);
  int dev = 0, cus = 0, per_cu = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, shmem);
  if (e != hipSuccess) return e;
  const int want = (items + kPrepWaves - 1) / kPrepWaves;
  const int grid = std::max(1, std::min(want, cus * std::max(per_cu, 1)));
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), shmem, stream, args);
  return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_prep_t(const PrepArgs& a, hipStream_t stream) {
  return launch_resident(&prep_kernel<T, D>, a, a.table_len, a.total_items, stream);
}

template <typename T, int D>
hipError_t launch_cached_t(const CachedArgs& a, hipStream_t stream) {
  return launch_resident(&prep_cached_kernel<T, D>, a, a.p.table_len, a.p.total_items, stream);
}

PrepArgs prep_args(const Tensor4* in, const Tensor4* out, const void* const* weight, float* const* mean, int H, int D,
                   int nb, const Geom& g, const int32_t* rope_grid, const int32_t* rope_dims, const float* table,
                   int table_len, float eps) {
  PrepArgs a{};
  for (int t = 0; t < 2; ++t) {
    a.in[t] = in[t];
    a.out[t] = out[t];
    a.weight[t] = weight[t];
    a.mean[t] = mean[t];
  }
  a.table = table;
  a.H = H;
  a.D = D;
  a.nb = nb;
  a.rT = rope_grid[0];
  a.rH = rope_grid[1];
  a.rW = rope_grid[2];
  a.dt = rope_dims[0];
  a.dh = rope_dims[1];
  a.table_len = table_len;
  a.eps = eps;
  a.g = g;
  a.heads = make_fastdiv((uint32_t)H);
  a.rcp_plane = (float)(1.0 / ((double)a.rH * a.rW));
  a.rcp_w = (float)(1.0 / (double)a.rW);
  a.neg_zero = -0.0f;
  a.one = 1.0f;
  return a;
}

}  // namespace

bool prep_supported(int dtype, int D) { return dtype != 2 && (D == 64 || D == 128); }

hipError_t launch_prep(const Tensor4* in, const Tensor4* out, const void* const* weight,
                       float* const* mean, int dtype, int B, int H, int D, int nb, const Geom& g,
                       const int32_t* rope_grid, const int32_t* rope_dims, const float* table,
                       int table_len, float eps, hipStream_t stream) {
  PrepArgs a = prep_args(in, out, weight, mean, H, D, nb, g, rope_grid, rope_dims, table, table_len, eps);
  a.total_items = 2 * B * H * nb;
  a.per_block = make_fastdiv((uint32_t)(2 * B * H));
  if (dtype == 0) return D == 128 ? launch_prep_t<f16, 128>(a, stream) : launch_prep_t<f16, 64>(a, stream);
  return D == 128 ? launch_prep_t<bf16, 128>(a, stream) : launch_prep_t<bf16, 64>(a, stream);
}

hipError_t launch_prep_cached(const PrepCached& x, int dtype, int B, int H, int D, int nb, int nk, const Geom& g,
                              const Geom& gk, const int32_t* rope_grid, const int32_t* rope_dims, const float* table,
                              int table_len, float eps, hipStream_t stream) {
  CachedArgs c{};
  c.p = prep_args(x.in, x.out, x.weight, x.mean, H, D, nb, g, rope_grid, rope_dims, table, table_len, eps);
  c.cache[0] = x.k_cache;
  c.cache[1] = x.v_cache;
  c.v_in = x.v_in;
  c.v_out = x.v_out;
  c.k_norm = x.k_norm;
  c.cached = x.cached;
  c.nk = nk;
  c.gk = gk;
  const int kv = x.v_out.ptr ? 2 : 1;  // tensors over the k-blocks
  c.head_items = (nk - nb) * kv * B * H;
  c.head_per_block = make_fastdiv((uint32_t)(kv * B * H));
  c.bh = make_fastdiv((uint32_t)(B * H));
  c.p.per_block = make_fastdiv((uint32_t)((kv + 1) * B * H));
  c.p.total_items = c.head_items + (kv + 1) * B * H * nb;
  if (dtype == 0) return D == 128 ? launch_cached_t<f16, 128>(c, stream) : launch_cached_t<f16, 64>(c, stream);
  return D == 128 ? launch_cached_t<bf16, 128>(c, stream) : launch_cached_t<bf16, 64>(c, stream);
}

}  // namespace lcv
