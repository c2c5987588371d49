// Tile-level pieces shared by the kernels' sources: MFMA forms, bounded buffer
// descriptors, LDS reads, lane exchanges, and the work items of the general
// attention kernels.
#pragma once

#include "attn_common.h"

namespace dx {
namespace {

// 32 x 32 x 16 products, and packing to their 16-bit operands.
template <typename T> struct Mfma;
template <> struct Mfma<bf16_t> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 r = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
    return __builtin_bit_cast(uint32_t, r);
  }
  // acc + lo + hi of a packed pair (v_dot2c_f32_bf16 against (1, 1)).
  static __device__ __forceinline__ float sum2(uint32_t p, float acc) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p),
                                           __builtin_bit_cast(bf16x2, 0x3f803f80u), acc, false);
  }
};
template <> struct Mfma<f16_t> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    f16x2 r = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
    return __builtin_bit_cast(uint32_t, r);
  }
  // acc + lo + hi of a packed pair (v_dot2c_f32_f16 against (1, 1)).
  static __device__ __forceinline__ float sum2(uint32_t p, float acc) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p),
                                  __builtin_bit_cast(f16x2, 0x3c003c00u), acc, false);
  }
};

// 16 x 16 x 32 (16-bit) and 16 x 16 x 4 (fp32) products.
template <typename T> struct Mfma16;
template <> struct Mfma16<bf16_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<f16_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int kBufWord3 = 0x00020000;  // gfx9-family raw buffer descriptor word 3

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const uint16_t* base, int rows,
                                                           int row_bytes, int D) {
  const int bytes = rows > 0 ? (rows - 1) * row_bytes + D * 2 : 0;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), (short)0, bytes,
                                           kBufWord3);
}

// Transposing LDS read (gfx950 ds_read_b64_tr_b16). Within each group of 16
// lanes, lane i receives element i % 4 of the 8-byte chunks addressed by
// lanes 4e + i / 4, e = 0..3 of its group.
typedef short v4i16 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 lds_read_tr16(const uint16_t* p) {
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4i16*)((__attribute__((address_space(3))) uint16_t*)(p)));
  return __builtin_bit_cast(u32x2, r);
}

// LDS accesses by byte address (for the swizzled layout, whose addresses are
// built with XOR).
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return uint32_t(uintptr_t((__attribute__((address_space(3))) const void*)(p)));
}
__device__ __forceinline__ u32x4 lds_read_b128_at(uint32_t addr) {
  return *reinterpret_cast<const lds_u32x4*>(addr);
}
__device__ __forceinline__ u32x2 lds_read_tr16_at(uint32_t addr) {
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_v4i16*>(addr));
  return __builtin_bit_cast(u32x2, r);
}

// Combine lanes i and i ^ 32 (v_permlane32_swap: a VALU exchange of the two
// wave halves, with no trip through the LDS queue as ds_bpermute takes).
__device__ __forceinline__ float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Max and sum over the four lanes of a query of the 16 x 16 products (lanes c,
// c + 16, c + 32, c + 48): the row swaps, again VALU exchanges.
__device__ __forceinline__ float quad_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return xor32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float quad_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return xor32_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// Key of register r of half kt: row 32 kt + 8 (r / 4) + 4 g + r % 4 of the
// tile, visible iff that row is below lim_rel (rows past the tile's valid
// keys or past this query's visible end are not). ``lim`` is lim_rel - 4 g.
__device__ __forceinline__ bool key_hidden(int kt, int r, int lim) {
  return 32 * kt + 8 * (r / 4) + (r % 4) >= lim;
}

// Cached rows of sequence b (the device cursor clamped to the capacity the
// launch was planned for, or the per-sequence length of a ragged batch).
__device__ __forceinline__ int any_cache_len(const AttnArgs& a, int b) {
  if (a.cache_len_dev) return min(max(*a.cache_len_dev, 0), a.cache_len);
  return a.n_seg ? a.seg_cache[b] : a.cache_len;
}

// Work item i of the grid. Workgroup i runs on XCD i % 8 (each XCD has its own
// L2): with a multiple of 8 (batch, head) pairs, XCD x takes a contiguous run
// of them, so a head's K/V (and a K/V head's query heads) go through one L2.
// Late query tiles, which see the most keys under a causal or block mask, go
// first. Partials stay numbered by (b, h, query tile, split). Cold, us per
// call, before (split fastest, then query tiles in order) -> now: D 256 causal
// 4000, 16 over 4 heads 467 -> 315; D 32 causal 4096 155 -> 91; D 256, 40 heads
// x 1500 in blocks of 200 198 -> 153; 2048 unmasked 166 -> 159.
// Where one work item reads each key (one query tile, a K/V head per query
// head) and all run at once (at most one per CU), an L2 has nothing to share:
// there a.spread keeps the splits of a head on consecutive workgroups. D 256, 64
// queries, 24 heads over 500 cached 21.9 us without it, 19.9 with it, 40 heads
// over 300 21.8 and 19.1; past one item per CU 24 heads over 1245 26.9 and 27.7.
struct AnyItem {
  int b, h, qt, split;
  int64_t partial;
};
__device__ __forceinline__ AnyItem any_item(const AttnArgs& a, int i) {
  const uint32_t G = uint32_t(a.B) * uint32_t(a.H), S = uint32_t(a.n_splits);
  uint32_t grp, rank;  // (batch, head) pair; rank within it
  if (a.spread) {
    grp = uint32_t(i) / S;
    rank = uint32_t(i) - grp * S;
  } else if (G % 8 == 0) {
    const uint32_t g8 = G / 8, slot = uint32_t(i) / 8;
    rank = slot / g8;
    grp = uint32_t(i) % 8 * g8 + (slot - rank * g8);
  } else {
    rank = uint32_t(i) / G;
    grp = uint32_t(i) - rank * G;
  }
  AnyItem it;
  const uint32_t rq = rank / S;
  it.split = int(rank - rq * S);
  it.qt = a.n_qtiles - 1 - int(rq);
  it.b = int(grp / uint32_t(a.H));
  it.h = int(grp) - it.b * a.H;
  it.partial = (int64_t(grp) * a.n_qtiles + it.qt) * S + it.split;
  return it;
}

}  // namespace
}  // namespace dx
