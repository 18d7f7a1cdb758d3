// Device helpers shared by the attention kernels: lane exchanges, the routing
// list walk, tile loads into LDS, MFMA wrappers and the LDS tile layout.
#pragma once

#include "bsa_common.h"

namespace lcv {
namespace {

constexpr int kBufferFlags = 0x00020000;  // raw buffer, 32-bit dwords (gfx9 family)

typedef __attribute__((address_space(3))) void lds_void;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// NaN-propagating max of three (v_maximum3_f32).
__device__ __forceinline__ float fmax3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

// Lanes l and l ^ 32 exchange x through v_permlane32_swap (a VALU op; no
// LDS round trip); the two results hold x[l] and x[l ^ 32] in some order.
__device__ __forceinline__ void swap_halves(float x, float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x),
                                                  __builtin_bit_cast(uint32_t, x), false, false);
  a = __builtin_bit_cast(float, (uint32_t)r[0]);
  b = __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float max_halves(float x) {
  float a, b;
  swap_halves(x, a, b);
  return __builtin_elementwise_maximum(a, b);
}
__device__ __forceinline__ float sum_halves(float x) {
  float a, b;
  swap_halves(x, a, b);
  return a + b;
}

__device__ __forceinline__ int next_valid(const int32_t* list, int j, int top_k, int nb) {
  while (j < top_k) {
    const int n = uniform_i32(list[j]);
    if (n >= 0 && n < nb) break;
    ++j;
  }
  return j;
}

// A q-block's routing list, read 64 entries at a time into one register:
// lane l holds the first token of block list[base + l] (-1 if the entry is
// outside [0, nb)), computed once per chunk with vector ops, plus a wave mask
// of the valid entries.  The tile loop then needs one v_readlane per tile
// and issues no vector loads of its own between tile fetches.
struct TileList {
  const int32_t* list;
  int top_k, nb, base;
  int raw;         // per lane: list entry base + l (INT_MAX past top_k)
  int tok;         // per lane
  uint64_t valid;  // bit l: entry base + l is a block in [0, nb)
  // Issues the load of entries 0..63; finish() converts them once they are
  // needed, so other loads can be in flight meanwhile.
  __device__ TileList(const int32_t* l, int k, int n) : list(l), top_k(k), nb(n), base(0) {
    raw = fetch(0);
  }
  __device__ int fetch(int b) const {
    const int j = b + lane_id();
    return j < top_k ? list[j] : 0x7fffffff;
  }
  __device__ void finish(const Geom& g) {
    const bool ok = raw >= 0 && raw < nb;
    tok = ok ? block_base_token(g, raw) : -1;
    valid = __ballot(ok);
  }
  __device__ void load(int b, const Geom& g) {
    base = b;
    raw = fetch(b);
    finish(g);
  }
  // First j' >= j whose entry is valid, or top_k.  j uniform.
  __device__ int next(int j, const Geom& g) {
    while (j < top_k) {
      if (j < base || j - base >= 64) load(j & ~63, g);
      const uint64_t m = valid >> (j - base);
      if (m) return j + (int)__builtin_ctzll(m);
      j = base + 64;
    }
    return top_k;
  }
  // First token of entry j (valid, within the current chunk).
  __device__ int32_t token(int j) const { return __builtin_amdgcn_readlane(tok, j - base); }
  // Number of entries before the first one >= n0 in an ascending list (for
  // any list: the count of leading entries < n0, which is a valid start).
  // Called with the first chunk in place; a one-chunk list needs no load.
  __device__ int count_below(int n0, const Geom& g) {
    int cnt = __popcll(__ballot(raw < n0));
    if (cnt < 64 || top_k <= 64) return cnt;
    for (int b = 64; b < top_k; b += 64) {
      load(b, g);
      const int c = __popcll(__ballot(raw < n0));
      cnt += c;
      if (c < 64) break;
    }
    return cnt;
  }
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16 bytes per lane from a raw buffer straight into LDS: lane i writes
// lds_dst + 16 i (1 KB per wave).  Issued as inline asm so that the only
// waits on it are the explicit wait_vmcnt<> calls (the compiler otherwise
// waits for every outstanding LDS load before any LDS read).
// The immediate OFF is added to both the memory and the LDS address, so four
// loads 1 KB apart in LDS share one M0 value when each lane's voffset is
// pre-reduced by OFF (the memory offset of a load's rows is at least OFF).
template <int OFF>
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset, int32_t soffset,
                                      uint32_t m0v) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%3 lds"
               ::"v"(voffset), "s"(rsrc), "s"(soffset), "i"(OFF), "{m0}"(m0v)
               : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

template <typename T>
struct Mfma;

template <>
struct Mfma<f16> {
  typedef f16x8 vec8;
  typedef _Float16 vec2 __attribute__((ext_vector_type(2)));
  __device__ static f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  // Sum of the 8 elements of v added to acc.
  __device__ static float sum8(vec8 v, float acc) {
    const vec2 one = {(f16)1.0f, (f16)1.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const vec2 pr = {v[2 * i], v[2 * i + 1]};
      acc = __builtin_amdgcn_fdot2(pr, one, acc, false);
    }
    return acc;
  }
};

template <>
struct Mfma<bf16> {
  typedef bf16x8 vec8;
  typedef __bf16 vec2 __attribute__((ext_vector_type(2)));
  __device__ static f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static float sum8(vec8 v, float acc) {
    const vec2 one = {(bf16)1.0f, (bf16)1.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const vec2 pr = {v[2 * i], v[2 * i + 1]};
      acc = __builtin_amdgcn_fdot2_f32_bf16(pr, one, acc, false);
    }
    return acc;
  }
};

// Tile geometry.  K and V rows are row-major in LDS, 2*D bytes per row,
// DC = D/8 16-byte chunks per row.  Chunk c of row r is stored at chunk
// position c ^ swz(r):
//   K: swz = (r / RP) % DC          -- 16 rows read one chunk column: conflict free
//   V: swz = 2 * ((r / RP) % (DC/2)) -- 8 rows x 32 bytes per 32-lane tr-read: conflict free
// where RP = 256 / (2*D) rows share one 256-byte bank span.
template <typename T, int D>
struct MfmaCfg {
  static constexpr int kThreads = 128;
  static constexpr int DC = D / 8;
  static constexpr int RP = 256 / (2 * D);
  static constexpr int kRowsPerDma = 64 / DC;  // rows per 1 KB wave load
  static_assert(D == 64 || D == 128, "MFMA tiling covers D = 64, 128");
  __device__ static int kswz(int r) { return (r / RP) % DC; }
  __device__ static int vswz(int r) { return 2 * ((r / RP) % (DC / 2)); }
};

// Lanes l and l ^ 16 exchange x through v_permlane16_swap; the two results
// hold x[l] and x[l ^ 16] in some order.
__device__ __forceinline__ void swap_rows16(float x, float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x),
                                                  __builtin_bit_cast(uint32_t, x), false, false);
  a = __builtin_bit_cast(float, (uint32_t)r[0]);
  b = __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float max_quarters(float x) {
  float a, b;
  swap_rows16(x, a, b);
  return max_halves(__builtin_elementwise_maximum(a, b));
}
__device__ __forceinline__ float sum_quarters(float x) {
  float a, b;
  swap_rows16(x, a, b);
  return sum_halves(a + b);
}

}  // namespace
}  // namespace lcv
