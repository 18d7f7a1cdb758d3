// Sparse attention over selected 64-token KV blocks for fp32 inputs, on bf16
// matrix cores (D = 64 or 128).
//
// Same semantics as the kernels of attn_fwd.hip (softmax over the listed
// blocks only; longcat_video/models/block_sparse_attention.py:201-250).  An
// fp32 value x of 2^-103 and more in size, or zero, is split exactly into three
// bf16 pieces, x = p0 + p1 + p2, each the round-to-nearest of what the previous
// ones leave (|p1| <= 2^-8 |x|, |p2| <= 2^-16 |x|; smaller values are seen to
// below, at kMinExact), and a product x y is formed from the six piece products
// p_i q_j with i + j <= 2: each is exact in fp32 and the dropped ones are
// below 2^-23 |x y| together, less than one fp32 rounding.  Six
// 16 x 16 x 32 bf16 MFMAs cost 96 matrix cycles where the eight fp32 MFMAs of
// the same tile cost 256.  Q, K, V and the softmax weights P are all split this
// way; scores, row maxima, weights, row sums and O stay fp32.
//
// Measured against the vector-ALU kernel (attn_valu_kernel), which forms every
// product from LDS operands: 8 heads x 12,480 tokens x 128, 13 of 195 blocks
// kept (42.5 GFLOP), 1,763 -> 284 us (24 -> 150 TFLOP/s; torch's fp32 GEMM of
// 8192^3 reaches 153 on this card); 2 heads x 4,096 x 64, 4 of 64 kept: 66.5 -> 16.2
// us.  4 and 0.6 us of these are the check for small values and P's scaling, at D = 64
// with longer lists (8 x 195 blocks) 5.7 of 164 us for the whole call.  Error against
// 64 bits (2-norm) 6.9e-7 -> 4.7e-7 and 4.0e-7 -> 2.7e-7.  At the first size the MFMA
// pipe is busy 39 % of the cycles, the VALU (a third of it splitting K and V tiles)
// 32 %, LDS 29 %, with no bank conflicts (before the check): what bounds it is how
// little the two or three workgroups of a CU overlap these, and the last generation
// of workgroups.
#include <algorithm>

#include "attn_common.h"

namespace lcv {
namespace {

// A value of at least kMinExact (or zero) has three pieces that are normal bf16
// numbers or zero, so nothing is cut off it: 2^-103 less 23 bits is 2^-126.
//   V: a smaller value, anywhere in the tiles, sends the workgroup to the second
//      walk.
//   P lies in [2^-149, 1]; scaled by 2^32 (exact, and divided out with the row sum)
//      its normal values are above the line, and O stays finite for |V| < 2^77.
//   Q: as V, and so does |q scale| >= kMaxQ.  Below that, what is cut off K (below
//      2^-126 a value) moves no score by more than D 2^-126 kMaxQ <= 2^-29.
constexpr float kMinExact = 0x1p-103f, kPScale = 0x1p32f, kMaxQ = 0x1p90f;

// 2 |x| as an integer less one: of nonzero values the order of |x|, zero the largest.
__device__ __forceinline__ uint32_t size_key(float x) { return (__builtin_bit_cast(uint32_t, x) << 1) - 1u; }
constexpr uint32_t kMinExactKey = (__builtin_bit_cast(uint32_t, kMinExact) << 1) - 1u;

// Pieces of a pair of fp32 values: w[i] holds piece i of x0 (low half) and x1.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&w)[3]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  f32x2 r = {x0, x1};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    w[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    if (i < 2) {
      const float lo = r[0] - __builtin_bit_cast(float, w[i] << 16);
      const float hi = r[1] - __builtin_bit_cast(float, w[i] & 0xffff0000u);
      r = {lo, hi};
    }
  }
}

__device__ __forceinline__ void split8(const f32x4& lo, const f32x4& hi, bf16x8 (&pc)[3]) {
  uint32_t w[4][3];
  split2(lo[0], lo[1], w[0]);
  split2(lo[2], lo[3], w[1]);
  split2(hi[0], hi[1], w[2]);
  split2(hi[2], hi[3], w[3]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
    pc[i] = __builtin_bit_cast(bf16x8, (u32x4){w[0][i], w[1][i], w[2][i], w[3][i]});
}

// The rare second walk: the arithmetic of valu_walk<float, D> (64 rows x 4
// lanes, the same 32-key groups and order of operations), but straight from
// memory and with each score formed twice instead of kept, so that it fits in
// the registers of the main loop.
template <int D>
__device__ __forceinline__ void slow_walk(const AttnParams& p, int bh, int qb, const float* qbase, const float* kbase,
                                          const float* vbase, float* obase) {
  constexpr int DQ = D / 4;
  const int col = (threadIdx.x % 4) * DQ;
  const int32_t qtok = block_base_token(p.g, qb) + voxel_row_offset(p.g, threadIdx.x / 4);
  float qv[DQ], ov[DQ];
#pragma unroll
  for (int dd = 0; dd < DQ; ++dd) {
    qv[dd] = qbase[(int64_t)qtok * p.q_ss + col + dd];
    ov[dd] = 0.0f;
  }
  float m_run = -__builtin_inff(), l_run = 0.0f;
  const int32_t* list = p.idx + ((int64_t)bh * p.nb + qb) * p.top_k;
  auto score = [&](int32_t tok) {
    const float* kr = kbase + (int64_t)tok * p.k_ss + col;
    float part = 0.0f;
#pragma unroll
    for (int dd = 0; dd < DQ; ++dd) part = fmaf(qv[dd], kr[dd], part);
    part += __shfl_xor(part, 1);
    part += __shfl_xor(part, 2);
    return part * p.scale_log2;
  };
#pragma unroll 1
  for (int j = next_valid(list, 0, p.top_k, p.nk); j < p.top_k; j = next_valid(list, j + 1, p.top_k, p.nk)) {
    const int32_t tok0 = block_base_token(p.gk, uniform_i32(list[j]));
#pragma unroll 1
    for (int half = 0; half < 64; half += 32) {
      float mx = m_run;
#pragma unroll 1
      for (int kk = 0; kk < 32; ++kk) mx = fmaxf(mx, score(tok0 + voxel_row_offset(p.gk, half + kk)));
      const float corr = fast_exp2(m_run - mx);
      l_run *= corr;
#pragma unroll
      for (int dd = 0; dd < DQ; ++dd) ov[dd] *= corr;
#pragma unroll 1
      for (int kk = 0; kk < 32; ++kk) {
        const int32_t tok = tok0 + voxel_row_offset(p.gk, half + kk);
        const float pe = fast_exp2(score(tok) - mx);
        const float* vr = vbase + (int64_t)tok * p.v_ss + col;
        l_run += pe;
#pragma unroll
        for (int dd = 0; dd < DQ; ++dd) ov[dd] = fmaf(pe, vr[dd], ov[dd]);
      }
      m_run = mx;
    }
  }
  const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
  for (int dd = 0; dd < DQ; ++dd) obase[(int64_t)qtok * p.o_ss + col + dd] = ov[dd] * inv;
}

// Waves per SIMD.  D = 128 keeps 48 registers of Q pieces, 32 of O and up to 32
// of tile prefetch: 196 in all, two waves (317 us for the whole call at the first
// size above; held to the 168 registers of three it spills Q pieces, 322).  D = 64
// needs half of each: four.
template <int D>
struct F32Occupancy {
  static constexpr int kWaves = D == 128 ? 2 : 4;
};

// One workgroup of four waves per (b, h, q-block), wave w owning query rows
// 16 w .. 16 w + 15.  A listed block is processed as two 32-key halves.  A half
// of K and V is loaded into registers while the half before it is computed,
// split once for all four waves and stored as three bf16 tiles each (row-major,
// 16-byte chunks XOR-swizzled as in the half-precision kernel); the lane layouts
// of S^T = K Q^T and O^T = V^T P^T are that kernel's too.
//
// Values that the split cannot carry (inf, NaN, or so close to the fp32
// maximum that they round to a bf16 infinity) turn their row's O into a NaN;
// a workgroup that ends with a non-finite O or row sum, or met a value below
// kMinExact where that counts, walks again on the vector ALU, whose result stands.
template <int D>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(F32Occupancy<D>::kWaves, F32Occupancy<D>::kWaves)))
void attn_f32_kernel(AttnParams p) {
  typedef MfmaCfg<bf16, D> C;
  typedef Mfma<bf16> M;
  constexpr int kRow = 2 * D;           // bytes per row of a piece
  constexpr int kPiece = 32 * kRow;     // one piece of a 32-row half
  constexpr int kGroup = 16 * kRow;     // 16 rows: the second key tile / key group
  constexpr int kC4 = D / 4;            // float4s per row
  constexpr int kTasks = 32 * kC4 / 256;
  constexpr int kStep = 256 / kC4;      // rows between a thread's tasks
  __shared__ __attribute__((aligned(1024))) uint8_t lds[6 * kPiece];
  uint8_t* const Kp = lds;
  uint8_t* const Vp = lds + 3 * kPiece;

  const int wid = xcd_linear_work_id(blockIdx.x, gridDim.x);
  const int bh = wid / p.nb;
  const int qb = p.order ? uniform_i32(p.order[wid]) : wid - bh * p.nb;
  if ((uint32_t)qb >= (uint32_t)p.nb) return;  // a launch-order entry outside [0, nb): nothing to do
  const int b = bh / p.H;
  const int h = bh - b * p.H;
  const int tid = threadIdx.x;
  const int wave = uniform_i32(tid / 64);
  const int lane = tid % 64;
  const int G = lane / 16;   // lane group: keys 4G.. of each 16-key tile, D rows 4G.. of O
  const int gi = lane % 16;  // this lane's query of the wave's 16

  const float* qbase = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh;
  float* obase = reinterpret_cast<float*>(p.out) + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh;
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)kbase, (short)0, (int)p.k_head_bytes, kBufferFlags);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)vbase, (short)0, (int)p.v_head_bytes, kBufferFlags);

  TileList list(p.idx + ((int64_t)bh * p.nb + qb) * p.top_k, p.top_k, p.nk);

  // Q^T pieces: qf[i][ks] holds piece i of query 16 wave + gi, D 32 ks + 8 G .. + 7.
  const int32_t qtok = block_base_token(p.g, qb) + voxel_row_offset(p.g, 16 * wave + gi);
  bf16x8 qf[3][D / 32];
  uint32_t least = ~0u;  // least size_key of the Q and V values this thread split; 0: Q or scale too large
  {
    const float* qrow = qbase + (int64_t)qtok * p.q_ss + 8 * G;
    f32x4 raw[D / 32][2];
    float q_max = 1.0f;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      raw[ks][0] = *reinterpret_cast<const f32x4*>(qrow + 32 * ks);
      raw[ks][1] = *reinterpret_cast<const f32x4*>(qrow + 32 * ks + 4);
    }
    list.finish(p.gk);
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      bf16x8 pc[3];
      split8(raw[ks][0], raw[ks][1], pc);
#pragma unroll
      for (int i = 0; i < 3; ++i) qf[i][ks] = pc[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        least = std::min(least, size_key(raw[ks][i / 4][i % 4]));
        q_max = fmaxf(q_max, __builtin_fabsf(raw[ks][i / 4][i % 4]));
      }
    }
    if (!(q_max * __builtin_fabsf(p.scale_log2) < kMaxQ)) least = 0;
  }

  // Tile staging: task u of a thread is float4 c4 of row r0 + kStep u of the
  // half.  Voxel sides are powers of two, so the token offset of row a + b of a
  // block is that of a plus that of b when a and b share no bits: the thread
  // keeps r0's, and kStep u and the second half (row 32) go into the scalar.
  const int r0 = tid / kC4;
  const int c4 = tid % kC4;
  const uint32_t koff = ((uint32_t)voxel_row_offset(p.gk, r0) * (uint32_t)p.k_ss + 4u * c4) * 4u;
  const uint32_t voff = ((uint32_t)voxel_row_offset(p.gk, r0) * (uint32_t)p.v_ss + 4u * c4) * 4u;
  // LDS byte of that float4's pieces (8 bytes each).  kStep rows further the
  // swizzle is the same, but for K at D = 128, where it flips chunk bit 3.
  const int kw0 = r0 * kRow + 16 * ((c4 / 2) ^ C::kswz(r0)) + 8 * (c4 % 2);
  const int vw0 = r0 * kRow + 16 * ((c4 / 2) ^ C::vswz(r0)) + 8 * (c4 % 2);
  const uint32_t k_row_bytes = (uint32_t)p.k_ss * 4u, v_row_bytes = (uint32_t)p.v_ss * 4u;
  uint32_t step_tok[kTasks];
#pragma unroll
  for (int u = 0; u < kTasks; ++u) step_tok[u] = (uint32_t)voxel_row_offset(p.gk, kStep * u);
  const uint32_t hi_tok = (uint32_t)voxel_row_offset(p.gk, 32);
  f32x4 kst[kTasks], vst[kTasks];
  auto load_k = [&](int32_t tok, int half) {
    const uint32_t t = (uint32_t)tok + (half ? hi_tok : 0u);
#pragma unroll
    for (int u = 0; u < kTasks; ++u)
      kst[u] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, koff, (int)((t + step_tok[u]) * k_row_bytes), 0));
  };
  auto load_v = [&](int32_t tok, int half) {
    const uint32_t t = (uint32_t)tok + (half ? hi_tok : 0u);
#pragma unroll
    for (int u = 0; u < kTasks; ++u)
      vst[u] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(vrs, voff, (int)((t + step_tok[u]) * v_row_bytes), 0));
  };
  auto store_tile = [&](const f32x4 (&st)[kTasks], uint8_t* tile, int w0, int flip) {
#pragma unroll
    for (int u = 0; u < kTasks; ++u) {
      uint32_t a[3], c[3];
      split2(st[u][0], st[u][1], a);
      split2(st[u][2], st[u][3], c);
      uint8_t* dst = tile + ((w0 ^ (u % 2 ? flip : 0)) + kStep * kRow * u);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(dst + i * kPiece) = (u32x2){a[i], c[i]};
    }
  };

  // LDS operand addresses, as in attn_half_kernel.
  const int kaddr0 = gi * kRow + 16 * (G ^ C::kswz(gi));
  const int vrow = 4 * G + gi / 4;
  const int vaddr0 = vrow * kRow + 16 * (((4 * (gi % 4)) / 8) ^ C::vswz(vrow)) + 2 * ((4 * (gi % 4)) % 8);

  f32x4 o[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) o[dt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -__builtin_inff(), l_run = 0.0f;
  const float sl2 = p.scale_log2;

  int j = list.next(0, p.gk);
  int32_t tok = j < p.top_k ? list.token(j) : 0;
  int half = 0;
  if (j < p.top_k) load_k(tok, 0);
  // Two barriers a half: the first comes after its K tile is written (every
  // wave is then past the previous half's V reads), the second after its V
  // tile is written (every wave is then past this half's K reads).  V loads fly
  // during QK^T, the next half's K loads during the softmax and PV.
  while (j < p.top_k) {
    store_tile(kst, Kp, kw0, D == 128 ? 128 : 0);
    load_v(tok, half);
    // The next half: the block's second one, then the next listed block.
    int jn = j;
    int32_t tokn = tok;
    if (half) {
      jn = list.next(j + 1, p.gk);
      tokn = jn < p.top_k ? list.token(jn) : 0;
    }
    const int halfn = half ^ 1;
    __syncthreads();

    // S^T = K Q^T.  The five small products sum apart from p0 q0, so that they
    // are not rounded at its size, and give the MFMAs independent chains.
    f32x4 sh[2], sl[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) sh[kt] = sl[kt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        bf16x8 kf[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
          kf[i] = *reinterpret_cast<const bf16x8*>(Kp + i * kPiece + kt * kGroup + (kaddr0 ^ (64 * ks)));
        sl[kt] = M::mma(kf[2], qf[0][ks], sl[kt]);
        sh[kt] = M::mma(kf[0], qf[0][ks], sh[kt]);
        sl[kt] = M::mma(kf[1], qf[1][ks], sl[kt]);
        sl[kt] = M::mma(kf[0], qf[2][ks], sl[kt]);
        sl[kt] = M::mma(kf[1], qf[0][ks], sl[kt]);
        sl[kt] = M::mma(kf[0], qf[1][ks], sl[kt]);
      }
      __builtin_amdgcn_sched_barrier(0);  // at most one step's operands in flight: registers
    }
    float s[8];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[4 * kt + i] = (sh[kt][i] + sl[kt][i]) * sl2;

    // Online softmax: the row's keys sit in the four lane groups.
    float mx = fmax3(s[0], s[1], s[2]);
    mx = fmax3(mx, s[3], s[4]);
    mx = fmax3(mx, s[5], s[6]);
    mx = max_quarters(fmax3(mx, s[7], m_run));
    if (__ballot(!(mx == m_run))) {  // some row's maximum moved
      const float corr = fast_exp2(m_run - mx);
      l_run *= corr;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[dt][i] *= corr;
      m_run = mx;
    }
    f32x4 pe[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) pe[e / 4][e % 4] = fast_exp2(s[e] - m_run) * kPScale;
    l_run += ((pe[0][0] + pe[0][1]) + (pe[0][2] + pe[0][3])) + ((pe[1][0] + pe[1][1]) + (pe[1][2] + pe[1][3]));
    bf16x8 pf[3];
    split8(pe[0], pe[1], pf);
    store_tile(vst, Vp, vw0, 0);
#pragma unroll
    for (int u = 0; u < kTasks; ++u)
#pragma unroll
      for (int i = 0; i < 4; i += 2)
        least = std::min(std::min(least, size_key(vst[u][i])), size_key(vst[u][i + 1]));
    __syncthreads();
    if (jn < p.top_k) load_k(tokn, halfn);

    // O^T += V^T P^T, two D tiles at a time.
#pragma unroll
    for (int d2 = 0; d2 < D / 32; ++d2) {
      bf16x8 vf[2][3];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const uint8_t* a = Vp + i * kPiece + (vaddr0 ^ (32 * (2 * d2 + t)));
          const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)a);
          const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(a + kGroup));
          vf[t][i] = __builtin_bit_cast(bf16x8, (short __attribute__((ext_vector_type(8)))){
                                                    lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
        }
      constexpr int kV[6] = {2, 1, 0, 1, 0, 0}, kP[6] = {0, 1, 2, 0, 1, 0};  // small products first
#pragma unroll
      for (int e = 0; e < 6; ++e)
#pragma unroll
        for (int t = 0; t < 2; ++t) o[2 * d2 + t] = M::mma(vf[t][kV[e]], pf[kP[e]], o[2 * d2 + t]);
    }
    j = jn;
    tok = tokn;
    half = halfn;
  }

  const float l_tot = sum_quarters(l_run);
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  float probe = l_tot * 0.0f;  // NaN once any value is not finite
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) probe = fmaf(o[dt][i], 0.0f, probe);
  if (__syncthreads_or(least < kMinExactKey || !(probe == 0.0f))) {
    slow_walk<D>(p, bh, qb, qbase, kbase, vbase, obase);
    return;
  }
  float* orow = obase + (int64_t)qtok * p.o_ss + 4 * G;
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) {
    f32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = o[dt][i] * inv;
    __builtin_nontemporal_store(w, reinterpret_cast<f32x4*>(orow + 16 * dt));
  }
}

bool rows16(const void* ptr, int64_t sb, int64_t sh, int64_t ss) {
  return ((uintptr_t)ptr & 15u) == 0 && sb % 4 == 0 && sh % 4 == 0 && ss % 4 == 0;
}

}  // namespace

bool attn_f32_usable(const AttnParams& p, int D) {
  return (D == 64 || D == 128) && rows16(p.q, p.q_sb, p.q_sh, p.q_ss) && rows16(p.k, p.k_sb, p.k_sh, p.k_ss) &&
         rows16(p.v, p.v_sb, p.v_sh, p.v_ss) && rows16(p.out, p.o_sb, p.o_sh, p.o_ss) &&
         p.k_head_bytes != 0xFFFFFFFFu && p.v_head_bytes != 0xFFFFFFFFu;
}

hipError_t launch_attn_f32(const AttnParams& p, int D, hipStream_t stream) {
  const dim3 grid(p.B * p.H * p.nb);
  if (D == 64) hipLaunchKernelGGL(attn_f32_kernel<64>, grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(attn_f32_kernel<128>, grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace lcv
