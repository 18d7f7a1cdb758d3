// Text cross-attention (fp16 / bf16, D = 64 or 128): every query row of batch
// item b attends to all len[b] keys of its slice of a packed text, with the
// query's RMSNorm_FP32 applied on the way in (attention.py:318-352 with
// blocks.py:55-72; the reference normalises q in full-tensor passes and
// attends under a block-diagonal mask).
//
// Reading q and writing out once is the bound at short texts, the MFMAs at
// long ones; text K / V come from L2.  One workgroup of four waves takes 128
// query rows of one (b, h), wave w rows 32w .. 32w + 31.  Four waves share each
// K / V half tile of 32 keys, so a tile is fetched once per 128 rows; the
// products and the operand layouts are those of attn_half_kernel
// (attn_fwd.hip): S^T = K Q^T and O^T = V^T P^T on 16 x 16 x 32 MFMAs with P in
// registers.  The half tiles go through a ring of four LDS slots in the order
// K(0), V(0), K(1), V(1), ..., each fetched three elements ahead.
//   * Any text length: rows of the last half tile past the end re-read the last
//     key (in bounds, and no maximum moves), their P and, in LDS, their V rows
//     become zero.  (A masked score would be -inf * 0 at a scale of zero.)
//   * Any query count: rows past the end repeat the last row and are not
//     stored.
//   * The softmax offset of a row is the maximum of its first half tile; where a
//     later P sum passes 2^15 or is NaN (no score above -inf so far), or a row's
//     whole sum is zero, the workgroup walks the text again from the rows' exact
//     maxima (rescaling O inside the walk spills 61 registers).  P is there
//     exp2((score - max) scale), as exact as the scores are at any size; the first
//     walk's fma(score, scale, -offset) is off by the rounding of the offset, which
//     a row shares until it overflows (|offset| of 2^28 and more).
// Work ids run batch item fastest: items of different text lengths share an
// XCD's time, and each XCD's heads keep their text K / V in its L2.
//
// Measured at 28,800 queries x 32 heads x 128, bf16, over the boxes seen: 256 text
// tokens 150 to 190 us (809 TFLOP/s at 150), 512 tokens 248 to 272 us (974 TFLOP/s at
// 248), 13 tokens 81 to 86 us (5.8 TB/s at 81); two items of 231 and 13 tokens 301 to 370
// us against 2,830 us for torch's norms, copies and flash attention.  Against variants,
// each on one box: 128-row workgroups against 64-row ones (twice the tile fetches) 301 /
// 422 us; plain against non-temporal query loads 301 / 316 us; work ids head by head
// against row tile by row tile with all heads together 316 / 320 us, and 265 / 332 us at
// 512 tokens.  168 registers at D = 128, one spilled in bf16.
#include "attn_common.h"
#include "norm_common.h"

namespace lcv {
namespace {

constexpr float kMaxLaneSum = 32768.0f;  // bound on a lane's P sum of one half tile: P stays a normal fp16 value

struct TextArgs {
  TextAttn t;
  int32_t tiles;
  float neg_zero;
};

template <int N>
struct Par {
  static constexpr int value = N;
};

template <typename T, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 128 ? 3 : 4, D == 128 ? 3 : 4)))
void text_attn_kernel(TextArgs p) {
  typedef MfmaCfg<T, D> C;
  typedef typename Mfma<T>::vec8 vec8;
  constexpr int kSlotBytes = 32 * 2 * D;         // 32 rows of K or V
  constexpr int kGroup = 16 * 2 * D;             // bytes of 16 rows
  constexpr int kLoads = kSlotBytes / 1024 / 4;  // 1 KB DMA loads per wave per half tile
  constexpr int kRows = 128;                     // query rows per workgroup
  __shared__ __attribute__((aligned(1024))) uint8_t ring[4 * kSlotBytes];
  __shared__ int wave_dirty[4];
  static_assert(4 * kSlotBytes == kRows * 2 * D, "the ring stages the output rows");

  const int wid = xcd_linear_work_id(blockIdx.x, gridDim.x);
  const int b = wid % p.t.B;
  const int ht = wid / p.t.B;
  const int h = ht / p.tiles;
  const int row0 = (ht - h * p.tiles) * kRows;
  const int tid = threadIdx.x;
  const int wave = uniform_i32(tid / 64);
  const int lane = tid % 64;
  const int G = lane / 16;
  const int gi = lane % 16;
  const int len = p.t.len[b];
  const int nh = (len + 31) / 32;
  const int tail = len % 32;

  const T* qbase = reinterpret_cast<const T*>(p.t.q.ptr) + (int64_t)b * p.t.q.sb + (int64_t)h * p.t.q.sh;
  const T* kbase = reinterpret_cast<const T*>(p.t.k.ptr) + (int64_t)h * p.t.k.sh + (int64_t)p.t.start[b] * p.t.k.ss;
  const T* vbase = reinterpret_cast<const T*>(p.t.v.ptr) + (int64_t)h * p.t.v.sh + (int64_t)p.t.start[b] * p.t.v.ss;
  T* obase = reinterpret_cast<T*>(const_cast<void*>(p.t.out.ptr)) + (int64_t)b * p.t.out.sb + (int64_t)h * p.t.out.sh;
  const uint32_t k_row_bytes = (uint32_t)p.t.k.ss * sizeof(T), v_row_bytes = (uint32_t)p.t.v.ss * sizeof(T);
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)kbase, (short)0, (int)((uint32_t)(len - 1) * k_row_bytes + 2 * D), kBufferFlags);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)vbase, (short)0, (int)((uint32_t)(len - 1) * v_row_bytes + 2 * D), kBufferFlags);

  // Q^T operand: qf[qt][ks] holds row 32 wave + 16 qt + gi, D 32 ks + 8 G .. + 7.
  vec8 qf[2][D / 32];
  u32x4 wr[D / 32];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const int r = row0 + 32 * wave + 16 * qt + gi;
    const T* qrow = qbase + (int64_t)(r < p.t.N ? r : p.t.N - 1) * p.t.q.ss + 8 * G;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks)
      qf[qt][ks] = __builtin_bit_cast(vec8, *reinterpret_cast<const u32x4*>(qrow + 32 * ks));
  }
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
    wr[ks] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const T*>(p.t.q_weight) + 32 * ks + 8 * G);

  // ---- DMA of K / V half tile `half` into `slot`: 32 rows, wave w's kLoads
  // loads of 1 KB starting at row 8w (D = 128: 2 loads of 4 rows; D = 64: 1 of 8).
  auto dma = [&](int half, int isv, int slot) {
    const __amdgpu_buffer_rsrc_t rs = isv ? vrs : krs;
    const uint32_t row_bytes = isv ? v_row_bytes : k_row_bytes;
    const uint32_t m0v = lds_addr(ring + slot * kSlotBytes + 1024 * (kLoads * wave));
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int row = (kLoads * wave + u) * C::kRowsPerDma + lane / C::DC;  // 0 .. 31
      const int key = 32 * half + row < len ? 32 * half + row : len - 1;
      const int chunk = (lane % C::DC) ^ (isv ? C::vswz(row) : C::kswz(row));
      dma16<0>(rs, (uint32_t)key * row_bytes + 16u * chunk, 0, m0v + 1024u * u);
    }
  };
  dma(0, 0, 0);
  dma(0, 1, 1);
  if (nh > 1) dma(1, 0, 2);

  // ---- RMSNorm_FP32 of the wave's query rows: a row's D values sit in the
  // four lanes gi, gi + 16, gi + 32, gi + 48.
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    float ss = 0.0f;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = to_f32(qf[qt][ks][e]);
        ss = __builtin_fmaf(x, x, ss);
      }
    const float rs = rsqrtf(sum_quarters(ss) * (1.0f / D) + p.t.eps);
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      float x[8], y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = to_f32(qf[qt][ks][e]);
      norm_scale<T>(x, rs, wr[ks], p.neg_zero, y);
#pragma unroll
      for (int e = 0; e < 8; ++e) qf[qt][ks][e] = from_f32<T>(y[e]);  // y holds values of T: exact
    }
  }

  // LDS operand addresses, as in attn_half_kernel.
  int kaddr[D / 32];
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) kaddr[ks] = gi * (2 * D) + 16 * ((4 * ks + G) ^ C::kswz(gi));
  const int vrow = 4 * G + gi / 4;
  const int vaddr0 = vrow * (2 * D) + 16 * (((4 * (gi % 4)) / 8) ^ C::vswz(vrow)) + 2 * ((4 * (gi % 4)) % 8);

  f32x4 oacc[D / 16][2];  // O^T tile (dt, qt)
  auto zero_o = [&] {
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) oacc[dt][qt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  zero_o();
  float m_run[2] = {0.0f, 0.0f}, l_run[2] = {0.0f, 0.0f};
  const float sl2 = p.t.scale_log2;
  vec8 pf[2];
  f32x4 sacc[2][2];

  auto qk = [&](const uint8_t* Ks) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) sacc[kt][qt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int kReads = 2 * (D / 32);  // read r: D step r / 2, key tile r % 2
    constexpr int kPf = 3;
    vec8 kf[kReads];
    auto read_k = [&](int r) {
      kf[r] = __builtin_bit_cast(vec8, *reinterpret_cast<const u32x4*>(Ks + kaddr[r / 2] + kGroup * (r % 2)));
    };
#pragma unroll
    for (int r = 0; r < kPf; ++r) read_k(r);
    __builtin_amdgcn_sched_group_barrier(0x100, kPf, 0);
#pragma unroll
    for (int r = 0; r < kReads; ++r) {
      if (r + kPf < kReads) read_k(r + kPf);
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) sacc[r % 2][qt] = Mfma<T>::mma(kf[r], qf[qt][r / 2], sacc[r % 2][qt]);
      if (r + kPf < kReads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
  };
  auto rowmax = [&](int qt) {
    float mx = fmax3(sacc[0][qt][0], sacc[0][qt][1], sacc[0][qt][2]);
    mx = fmax3(mx, sacc[0][qt][3], sacc[1][qt][0]);
    mx = fmax3(mx, sacc[1][qt][1], sacc[1][qt][2]);
    mx = __builtin_elementwise_maximum(mx, sacc[1][qt][3]);
    return max_quarters(mx);
  };
  bool dirty = false, exact = false;
  auto exps = [&](int qt) {
    if (exact) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sacc[kt][qt][i] = (sacc[kt][qt][i] - m_run[qt]) * sl2;
    } else {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sacc[kt][qt][i] = __builtin_fmaf(sacc[kt][qt][i], sl2, -m_run[qt]);
    }
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) pf[qt][4 * kt + i] = from_f32<T>(fast_exp2(sacc[kt][qt][i]));
    return Mfma<T>::sum8(pf[qt], 0.0f);
  };
  auto pv = [&](const uint8_t* Vs) {
    constexpr int kDt = D / 16;
    constexpr int kPf = 2;
    vec8 vf[kDt];
    auto read_v = [&](int dt) {
      const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(Vs + (vaddr0 ^ (32 * dt))));
      const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(Vs + (vaddr0 ^ (32 * dt)) + kGroup));
      vf[dt] = __builtin_bit_cast(vec8, (short __attribute__((ext_vector_type(8)))){
                                            lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    };
#pragma unroll
    for (int dt = 0; dt < kPf; ++dt) read_v(dt);
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kPf, 0);
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt) {
      if (dt + kPf < kDt) read_v(dt + kPf);
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) oacc[dt][qt] = Mfma<T>::mma(vf[dt], pf[qt], oacc[dt][qt]);
      if (dt + kPf < kDt) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
  };

  // Half tile s: elements 2s (K, slot 2s mod 4) and 2s + 1 (V).  At the
  // barrier that starts an element every wave has consumed the one before, so
  // the element three ahead goes into its slot; at most two are in flight.
  auto run_half = [&](int s, auto par) {
    constexpr int P = decltype(par)::value;  // s mod 2
    const bool more = s + 1 < nh;
    if (more) wait_vmcnt<2 * kLoads>();
    else wait_vmcnt<kLoads>();
    __syncthreads();
    if (more) dma(s + 1, 1, (2 * P + 3) % 4);
    qk(ring + 2 * P * kSlotBytes);
    if (s == 0 && !exact) {
      m_run[0] = rowmax(0) * sl2;
      m_run[1] = rowmax(1) * sl2;
    }
    float l0 = exps(0), l1 = exps(1);
    if (!more && tail) {
#pragma unroll
      for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (16 * (e / 4) + 4 * G + e % 4 >= tail) pf[qt][e] = from_f32<T>(0.0f);
      l0 = Mfma<T>::sum8(pf[0], 0.0f);
      l1 = Mfma<T>::sum8(pf[1], 0.0f);
    }
    if (__ballot(!(l0 + l1 <= kMaxLaneSum))) dirty = true;  // wave-uniform, rare
    l_run[0] += l0;
    l_run[1] += l1;

    if (more) wait_vmcnt<2 * kLoads>();
    else wait_vmcnt<0>();
    __syncthreads();
    if (s + 2 < nh) dma(s + 2, 0, (2 * P + 4) % 4);
    uint8_t* Vs = ring + (2 * P + 1) * kSlotBytes;
    if (!more && tail) {  // V rows past the end: zero times P = 0, whatever the last key's V holds
      for (int i = tid; i < (32 - tail) * C::DC; i += 256)
        *reinterpret_cast<u32x4*>(Vs + tail * (2 * D) + 16 * i) = u32x4{0u, 0u, 0u, 0u};
      __syncthreads();
    }
    pv(Vs);
  };
  for (;;) {
    for (int s = 0; s < nh; s += 2) {
      run_half(s, Par<0>{});
      if (s + 1 < nh) run_half(s + 1, Par<1>{});
    }
    if (__ballot(!(sum_quarters(l_run[0]) > 0.0f) || !(sum_quarters(l_run[1]) > 0.0f))) dirty = true;
    if (lane == 0) wave_dirty[wave] = dirty ? 1 : 0;
    __syncthreads();  // every ring read done (no DMA is outstanding here); flags visible
    if (exact || !(wave_dirty[0] | wave_dirty[1] | wave_dirty[2] | wave_dirty[3])) break;  // workgroup-uniform
    exact = true;
    float mx[2] = {-__builtin_inff(), -__builtin_inff()};
    for (int s = 0; s < nh; ++s) {  // the last key's repeats change no maximum
      dma(s, 0, 0);
      wait_vmcnt<0>();
      __syncthreads();
      qk(ring);
      mx[0] = __builtin_elementwise_maximum(mx[0], rowmax(0));
      mx[1] = __builtin_elementwise_maximum(mx[1], rowmax(1));
      __syncthreads();  // slot 0 read by every wave before it is loaded again
    }
    m_run[0] = mx[0], m_run[1] = mx[1];
    l_run[0] = l_run[1] = 0.0f;
    zero_o();
    int s0 = 0;
    asm("" : "+s"(s0));  // the first fetches' addresses computed again, not kept over the walk
    dma(s0, 0, 0);
    dma(s0, 1, 1);
    if (nh > 1) dma(s0 + 1, 0, 2);
  }

  // ---- Normalise, stage the rows in the ring, write whole rows.  A row whose
  // scores are all -inf has a NaN sum, as a softmax over it does.
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    const float inv = 1.0f / sum_quarters(l_run[qt]);
    const int row = 32 * wave + 16 * qt + gi;
    uint8_t* orow = ring + row * (2 * D);
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      u32x2 w;
      w[0] = bits16(from_f32<T>(oacc[dt][qt][0] * inv)) | (bits16(from_f32<T>(oacc[dt][qt][1] * inv)) << 16);
      w[1] = bits16(from_f32<T>(oacc[dt][qt][2] * inv)) | (bits16(from_f32<T>(oacc[dt][qt][3] * inv)) << 16);
      *reinterpret_cast<u32x2*>(orow + 16 * ((2 * dt + G / 2) ^ C::kswz(row)) + 8 * (G % 2)) = w;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kRows * C::DC / 256; ++u) {
    const int pidx = tid + 256 * u;
    const int row = pidx / C::DC;
    const int c = pidx % C::DC;
    if (row0 + row < p.t.N)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(ring + row * (2 * D) + 16 * (c ^ C::kswz(row))),
                                  reinterpret_cast<u32x4*>(obase + (int64_t)(row0 + row) * p.t.out.ss + 8 * c));
  }
}

template <typename T, int D>
hipError_t launch(const TextAttn& t, hipStream_t stream) {
  TextArgs p{t, (t.N + 127) / 128, -0.0f};
  hipLaunchKernelGGL((text_attn_kernel<T, D>), dim3(t.B * t.H * p.tiles), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_text_attn(const TextAttn& t, int dtype, int D, hipStream_t stream) {
  if (dtype == LCV_BSA_F16) return D == 64 ? launch<f16, 64>(t, stream) : launch<f16, 128>(t, stream);
  return D == 64 ? launch<bf16, 64>(t, stream) : launch<bf16, 128>(t, stream);
}

}  // namespace lcv
