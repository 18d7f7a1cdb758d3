// Row operations of the DiT block around the attention, each one HBM pass:
//
//  * residual + LayerNorm: r = x, x + a, or x + gate * a (fp32, per-frame
//    gate), rounded to the tensor dtype; optionally written out; then
//    LayerNorm_FP32(r) with either the affine weight / bias or the AdaLN
//    modulation (* (scale + 1) + shift, per frame), rounded to the dtype
//    (longcat_video_dit.py:107-136 with blocks.py:79-119);
//  * SwiGLU gate: silu(a) * b over the two halves of the fused w1 / w3
//    projection (blocks.py:50-51);
//  * AdaLN modulation: silu(t) W^T + b in fp32 from the half-precision weight,
//    written chunk by chunk (longcat_video_dit.py:80-138);
//  * per-head RMSNorm_FP32 (blocks.py:55-72) from one layout to another, for
//    the cross-attention's q and k (attention.py:325-326).
//
// The reference runs each of these as several full-tensor passes in fp32.
#include <algorithm>

#include "norm_common.h"

namespace lcv {
namespace {

constexpr int kRowWaves = 4;

struct RowArgs {
  const void* x;
  const void* a;          // [rows, C] or null
  const float* gate;      // [B, T, C] or null: r = x + gate * a
  const float* shift;     // [B, T, C] or null: AdaLN modulation
  const float* scale;
  const void* ln_w;       // [C] in the tensor dtype or null: affine LayerNorm
  const void* ln_b;
  void* x_out;            // r, or null
  void* n_out;            // the normalised row, or null
  int32_t rows, C, rows_per_batch, tokens_per_frame, frames;
  float eps;
};

template <typename T>
__device__ __forceinline__ void load8(const T* p, float* v) {
  const u32x4 raw = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    v[2 * m] = to_f32(__builtin_bit_cast(T, (uint16_t)(raw[m] & 0xffffu)));
    v[2 * m + 1] = to_f32(__builtin_bit_cast(T, (uint16_t)(raw[m] >> 16)));
  }
}

template <typename T>
__device__ __forceinline__ void store8(T* p, const float* v) {
  uint32_t w[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
    w[m] = bits16(round_from_f32<T>(v[2 * m])) | (bits16(round_from_f32<T>(v[2 * m + 1])) << 16);
  *reinterpret_cast<u32x4*>(p) = u32x4{w[0], w[1], w[2], w[3]};
}

__device__ __forceinline__ void load8f(const float* p, float* v) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
  v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// One wave per row; lane l holds the 8-element chunks l, l + 64, ... of the
// row (NMAX chunks at most, so C <= 512 * NMAX).  HBM bound: all of a row's x and a
// are loaded before the first use, and nothing in the kernel branches per lane
// (a chunk past the row re-reads the lane's first one and counts for nothing), so
// that no load waits for another.  28,800 x 4096, fp16, before (a wait per chunk and
// tensor) and now: gated residual + norm 192 -> 179 us (5.3 TB/s), residual +
// modulation 196 -> 178, modulation alone 115 -> 104, gated residual alone 131 -> 126;
// at C = 8192 451 -> 345, 440 -> 352, 265 -> 232 and 306 -> 251 us.
enum RowMode { kNoAdd = 0, kAdd = 1, kGatedAdd = 2 };

template <typename T, int NMAX, int MODE>
__global__ __launch_bounds__(256) void rows_kernel(RowArgs p) {
  const int wave = uniform_i32(threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  const int row = blockIdx.x * kRowWaves + wave;
  if (row >= p.rows) return;  // wave-uniform
  const int b = row / p.rows_per_batch;
  const int t = (row - b * p.rows_per_batch) / p.tokens_per_frame;
  const int64_t frame = ((int64_t)b * p.frames + t) * p.C;
  const int64_t base = (int64_t)row * p.C;
  const int nch = p.C / 8;
  const int first = lane < nch ? lane : 0;
  auto chunk = [&](int i) { return lane + 64 * i < nch ? lane + 64 * i : first; };
  auto live = [&](int i) { return lane + 64 * i < nch; };

  u32x4 xr[NMAX], ar[NMAX];
#pragma unroll
  for (int i = 0; i < NMAX; ++i)
    xr[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(p.x) + base + 8 * chunk(i));
  if constexpr (MODE != kNoAdd) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i)
      ar[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(p.a) + base + 8 * chunk(i));
  }
  float r[NMAX][8];
#pragma unroll
  for (int i = 0; i < NMAX; ++i) {
    widen8<T>(xr[i], r[i]);
    if constexpr (MODE != kNoAdd) {
      float av[8];
      widen8<T>(ar[i], av);
      if constexpr (MODE == kGatedAdd) {
        float g[8];
        load8f(p.gate + frame + 8 * chunk(i), g);
#pragma unroll
        for (int e = 0; e < 8; ++e) r[i][e] = to_f32(round_from_f32<T>(r[i][e] + g[e] * av[e]));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) r[i][e] = to_f32(round_from_f32<T>(r[i][e] + av[e]));
      }
    }
  }
  if constexpr (MODE != kNoAdd) {
    if (p.x_out) {
#pragma unroll
      for (int i = 0; i < NMAX; ++i)
        if (live(i)) store8(reinterpret_cast<T*>(p.x_out) + base + 8 * chunk(i), r[i]);
    }
  }
  if (!p.n_out) return;

  // LayerNorm in fp32: mean, then the mean of squared deviations.
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NMAX; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += live(i) ? r[i][e] : 0.0f;
  const float mean = wave_sum(s) / (float)p.C;
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < NMAX; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = live(i) ? r[i][e] - mean : 0.0f;
      q += d * d;
    }
  const float rstd = rsqrtf(wave_sum(q) / (float)p.C + p.eps);
#pragma unroll
  for (int i = 0; i < NMAX; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) r[i][e] = (r[i][e] - mean) * rstd;
  if (p.ln_w) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      float w[8], bb[8];
      load8(reinterpret_cast<const T*>(p.ln_w) + 8 * chunk(i), w);
      load8(reinterpret_cast<const T*>(p.ln_b) + 8 * chunk(i), bb);
#pragma unroll
      for (int e = 0; e < 8; ++e) r[i][e] = r[i][e] * w[e] + bb[e];
    }
  }
  if (p.scale) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      float sc[8], sh[8];
      load8f(p.scale + frame + 8 * chunk(i), sc);
      load8f(p.shift + frame + 8 * chunk(i), sh);
#pragma unroll
      for (int e = 0; e < 8; ++e) r[i][e] = r[i][e] * (sc[e] + 1.0f) + sh[e];
    }
  }
#pragma unroll
  for (int i = 0; i < NMAX; ++i)
    if (live(i)) store8(reinterpret_cast<T*>(p.n_out) + base + 8 * chunk(i), r[i]);
}

template <typename T, int NMAX, int MODE>
hipError_t launch_rows_m(const RowArgs& a, hipStream_t stream) {
  const int grid = (a.rows + kRowWaves - 1) / kRowWaves;
  hipLaunchKernelGGL((rows_kernel<T, NMAX, MODE>), dim3(grid), dim3(64 * kRowWaves), 0, stream, a);
  return hipGetLastError();
}

template <typename T, int NMAX>
hipError_t launch_rows_t(const RowArgs& a, hipStream_t stream) {
  if (!a.a) return launch_rows_m<T, NMAX, kNoAdd>(a, stream);
  return a.gate ? launch_rows_m<T, NMAX, kGatedAdd>(a, stream) : launch_rows_m<T, NMAX, kAdd>(a, stream);
}

// silu(a) * b, each rounded to the dtype (torch's silu computes x / (1 +
// exp(-x)) in fp32; the product of two dtype values is exact in fp32).
// Inside |x| < 80 the division runs as a reciprocal, a product and one residual
// correction, the quotient that IEEE division gives (checked for every fp16 and
// bf16 x), without its scaling of extreme operands; waves with larger x divide.
// With a 64-bit division per thread for its row the kernel was bound by the VALU:
// 28,800 x 11,008, fp16, 384 -> 343 us (5.5 TB/s, the rate of a copy).
__device__ __forceinline__ float silu_near(float x) {
  const float d = 1.0f + expf(-x);
  const float rc = __builtin_amdgcn_rcpf(d);
  const float y = x * rc;
  return __builtin_fmaf(-__builtin_fmaf(d, y, -x), rc, y);  // this order of signs keeps -0
}

constexpr int kGatePer = 2;  // 8-element chunks per thread

template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* h, T* out, uint32_t n8, FastDiv per_row) {
  u32x4 ar[kGatePer], br[kGatePer];
#pragma unroll
  for (int u = 0; u < kGatePer; ++u) {
    const uint32_t i = (blockIdx.x * kGatePer + u) * 256u + threadIdx.x;
    const uint32_t j = i < n8 ? i : n8 - 1;
    const uint32_t row = fast_div(j, per_row);
    const T* src = h + 8 * ((int64_t)row * per_row.d + j);
    ar[u] = *reinterpret_cast<const u32x4*>(src);
    br[u] = *reinterpret_cast<const u32x4*>(src + 8 * (int64_t)per_row.d);
  }
#pragma unroll
  for (int u = 0; u < kGatePer; ++u) {
    const uint32_t i = (blockIdx.x * kGatePer + u) * 256u + threadIdx.x;
    float a[8], bv[8], y[8];
    widen8<T>(ar[u], a);
    widen8<T>(br[u], bv);
    float m = 0.0f;  // a NaN is no maximum: silu_near keeps it
#pragma unroll
    for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(a[e]));
    if (__ballot(!(m < 80.0f))) {
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = a[e] / (1.0f + expf(-a[e]));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = silu_near(a[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = to_f32(round_from_f32<T>(y[e])) * bv[e];
    if (i < n8) store8(out + 8 * (int64_t)i, y);
  }
}

// RMSNorm_FP32 of rows of D elements: (b, n, h) -> out[b, h, n, :] (any
// strides), D / 8 lanes per row.
struct HeadNormArgs {
  const void* x;
  int64_t x_sb, x_sn, x_sh;
  void* out;
  int64_t o_sb, o_sn, o_sh;
  const void* w;  // [D] or null
  int32_t B, N, H, rows;
  float eps, neg_zero;
};

template <typename T, int D>
__global__ __launch_bounds__(256) void head_norm_kernel(HeadNormArgs p) {
  constexpr int LPR = D / 8;
  constexpr int RPW = 64 / LPR;  // rows per wave
  const int lane = threadIdx.x % 64;
  const int row = (blockIdx.x * 4 + (int)(threadIdx.x / 64)) * RPW + lane / LPR;
  const bool ok = row < p.rows;
  const int rr = ok ? row : 0;
  const int h = rr % p.H;
  const int bn = rr / p.H;
  const int n = bn % p.N;
  const int b = bn / p.N;
  const int c = lane % LPR;
  float x[8];
  load8(reinterpret_cast<const T*>(p.x) + b * p.x_sb + n * p.x_sn + h * p.x_sh + 8 * c, x);
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(x[e], x[e], ss);  // x*x exact in fp32
  ss = group_sum<LPR>(ss);
  const float rs = rsqrtf(ss * (1.0f / D) + p.eps);
  u32x4 wr;
  if (p.w) {
    wr = *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(p.w) + 8 * c);
  } else {
    const uint32_t one = bits16(from_f32<T>(1.0f));
    wr = u32x4{one | (one << 16), one | (one << 16), one | (one << 16), one | (one << 16)};
  }
  float y[8];
  norm_scale<T>(x, rs, wr, p.neg_zero, y);
  if (ok) store8(reinterpret_cast<T*>(p.out) + b * p.o_sb + n * p.o_sn + h * p.o_sh + 8 * c, y);
}

// out[j][r][c] = b[j C + c] + sum_k silu(t[r][k]) W[j C + c][k], all in fp32.
// Reading W (25 MB at 6 x 4096 x 512) is the floor, 5 us; what is left is the
// latency of one load, one silu phase and one reduction after the other, in a
// single round of waves.  silu(t) of eight rows is formed once per workgroup; a
// wave keeps it in registers (lane l: columns 8 l .. 8 l + 7 of each 512) and walks
// over rows of W, kAdaRows of them loaded before the first is used; the eight sums
// of a W row are reduced over the 64 lanes by halving first the sums a lane holds,
// then the lanes.  8 frames, fp16: 23 us (34 us with a wait per loaded row), for
// torch's conversions, GEMM and copies of the chunks 75 us and ten launches.
constexpr int kAdaRows = 8;
constexpr int kAdaWaves = 3072;  // three per SIMD

struct AdaArgs {
  const float* t;   // [R, K]
  const void* w;    // [M, K]
  const void* b;    // [M]
  float* out;       // [M / C, R, C]
  int32_t R, K, M, C;
};

template <typename T, int NC>
__global__ __launch_bounds__(256) void adaln_kernel(AdaArgs p) {
  const int wave = uniform_i32(blockIdx.x * 4 + threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  const int r0 = blockIdx.y * 8;
  __shared__ __attribute__((aligned(16))) float silu[8][512 * NC];  // zero past R and K
  {
    constexpr int n = 512 * NC / 256;  // 256-column strips per row
    float x[8 * n];
#pragma unroll
    for (int i = 0; i < 8 * n; ++i) {  // in-range loads, all before the first use
      const int r = r0 + i / n, k = 256 * (i % n) + (int)threadIdx.x;
      x[i] = p.t[(int64_t)(r < p.R ? r : 0) * p.K + (k < p.K ? k : 0)];
    }
#pragma unroll
    for (int i = 0; i < 8 * n; ++i) {
      const int r = i / n, k = 256 * (i % n) + (int)threadIdx.x;
      const float v = r0 + r < p.R && k < p.K ? x[i] : 0.0f;
      silu[r][k] = v / (1.0f + expf(-v));
    }
  }
  __syncthreads();
  float s[NC][8][8];
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int r = 0; r < 8; ++r) load8f(&silu[r][512 * n + 8 * lane], s[n][r]);
  const int waves = gridDim.x * 4;
  for (int m0 = wave * kAdaRows; m0 < p.M; m0 += waves * kAdaRows) {  // M % kAdaRows == 0
    u32x4 raw[kAdaRows][NC];  // every load before the first use; zero past K
#pragma unroll
    for (int i = 0; i < kAdaRows; ++i)
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int k = 512 * n + 8 * lane;
        raw[i][n] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(p.w) + (int64_t)(m0 + i) * p.K +
                                                    (k < p.K ? k : 0));
      }
    __builtin_amdgcn_sched_barrier(0);
    float w[kAdaRows][NC][8];
#pragma unroll
    for (int i = 0; i < kAdaRows; ++i)
#pragma unroll
      for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t u = 512 * n + 8 * lane < p.K ? raw[i][n][e] : 0u;
          w[i][n][2 * e] = to_f32(__builtin_bit_cast(T, (uint16_t)(u & 0xffffu)));
          w[i][n][2 * e + 1] = to_f32(__builtin_bit_cast(T, (uint16_t)(u >> 16)));
        }
#pragma unroll
    for (int i = 0; i < kAdaRows; ++i) {
      float a[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        a[r] = 0.0f;
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int e = 0; e < 8; ++e) a[r] = __builtin_fmaf(s[n][r][e], w[i][n][e], a[r]);
      }
      // Lane bit 5 picks sums 0..3 or 4..7, bit 4 the pair, bit 3 the sum: lane l
      // ends with sum (l / 8) over all lanes' columns.
#pragma unroll
      for (int h = 4, bit = 32; h >= 1; h /= 2, bit /= 2)
#pragma unroll
        for (int r = 0; r < h; ++r) {
          const bool up = lane & bit;
          const float mine = up ? a[r + h] : a[r], other = up ? a[r] : a[r + h];
          a[r] = mine + __shfl_xor(other, bit);
        }
      const float sum = group_sum<8>(a[0]);
      const int r = r0 + lane / 8;
      const int m = m0 + i;
      if (lane % 8 == 0 && r < p.R) {
        const int j = m / p.C;
        p.out[((int64_t)j * p.R + r) * p.C + (m - j * p.C)] = sum + to_f32(reinterpret_cast<const T*>(p.b)[m]);
      }
    }
  }
}

}  // namespace

bool rows_supported(int dtype, int C) { return dtype != 2 && C > 0 && C % 8 == 0 && C <= 8192; }

hipError_t launch_rows(const void* x, const void* a, const float* gate, const float* shift,
                       const float* scale, const void* ln_w, const void* ln_b, void* x_out,
                       void* n_out, int dtype, int rows, int C, int rows_per_batch,
                       int tokens_per_frame, int frames, float eps, hipStream_t stream) {
  RowArgs p{x, a, gate, shift, scale, ln_w, ln_b, x_out, n_out,
            rows, C, rows_per_batch, tokens_per_frame, frames, eps};
  const int nmax = (C / 8 + 63) / 64;
  if (dtype == 0) {
    if (nmax <= 2) return launch_rows_t<f16, 2>(p, stream);
    if (nmax <= 4) return launch_rows_t<f16, 4>(p, stream);
    if (nmax <= 8) return launch_rows_t<f16, 8>(p, stream);
    return launch_rows_t<f16, 16>(p, stream);
  }
  if (nmax <= 2) return launch_rows_t<bf16, 2>(p, stream);
  if (nmax <= 4) return launch_rows_t<bf16, 4>(p, stream);
  if (nmax <= 8) return launch_rows_t<bf16, 8>(p, stream);
  return launch_rows_t<bf16, 16>(p, stream);
}

hipError_t launch_swiglu(const void* h, void* out, int dtype, int64_t rows, int hidden,
                         hipStream_t stream) {
  const int64_t n8 = rows * (hidden / 8);
  if (n8 > 0xFFFFFFFFll - 256 * kGatePer) return hipErrorInvalidValue;
  const int grid = (int)((n8 + 256 * kGatePer - 1) / (256 * kGatePer));
  const FastDiv per_row = make_fastdiv((uint32_t)(hidden / 8));
  if (dtype == 0)
    hipLaunchKernelGGL((swiglu_kernel<f16>), dim3(grid), dim3(256), 0, stream,
                       reinterpret_cast<const f16*>(h), reinterpret_cast<f16*>(out), (uint32_t)n8, per_row);
  else
    hipLaunchKernelGGL((swiglu_kernel<bf16>), dim3(grid), dim3(256), 0, stream,
                       reinterpret_cast<const bf16*>(h), reinterpret_cast<bf16*>(out), (uint32_t)n8, per_row);
  return hipGetLastError();
}

bool adaln_supported(int dtype, int64_t K, int64_t C) {
  return dtype != LCV_BSA_F32 && K > 0 && K % 8 == 0 && K <= 1024 && C > 0 && C % kAdaRows == 0;
}

hipError_t launch_adaln(const float* t, const void* w, const void* b, int dtype, int R, int K, int chunks, int C,
                        float* out, hipStream_t stream) {
  const AdaArgs p{t, w, b, out, R, K, chunks * C, C};
  const int waves = std::min(p.M / kAdaRows, kAdaWaves);
  const dim3 grid((unsigned)((waves + 3) / 4), (unsigned)((R + 7) / 8));
  if (dtype == LCV_BSA_F16) {
    if (K <= 512) hipLaunchKernelGGL((adaln_kernel<f16, 1>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((adaln_kernel<f16, 2>), grid, dim3(256), 0, stream, p);
  } else {
    if (K <= 512) hipLaunchKernelGGL((adaln_kernel<bf16, 1>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((adaln_kernel<bf16, 2>), grid, dim3(256), 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_head_norm(const void* x, const int64_t* xs, void* out, const int64_t* os,
                            const void* w, int dtype, int B, int N, int H, int D, float eps,
                            hipStream_t stream) {
  HeadNormArgs p{x, xs[0], xs[1], xs[2], out, os[0], os[1], os[2], w, B, N, H, B * N * H, eps, -0.0f};
  const int rpw = 64 / (D / 8);
  const int grid = (p.rows + 4 * rpw - 1) / (4 * rpw);
  if (dtype == 0) {
    if (D == 128) hipLaunchKernelGGL((head_norm_kernel<f16, 128>), dim3(grid), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((head_norm_kernel<f16, 64>), dim3(grid), dim3(256), 0, stream, p);
  } else {
    if (D == 128) hipLaunchKernelGGL((head_norm_kernel<bf16, 128>), dim3(grid), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((head_norm_kernel<bf16, 64>), dim3(grid), dim3(256), 0, stream, p);
  }
  return hipGetLastError();
}

}  // namespace lcv
