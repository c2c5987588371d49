// Blockwise-causal attention at head dim 256 for 16-bit inputs, prefill-shaped
// calls, on gfx950 (the semantics of attn_fwd.hip; decode-shaped calls and the
// other head dims of the general path stay in attn_any.hip).
//
// attn_any16_kernel gives a wave 16 queries: every K and V byte it reads from
// LDS feeds 16 x 16 MFMAs, twice the LDS bytes per FLOP that the matrix cores
// can be fed at (128 B per clock and CU), and it ran at 500 TFLOP/s. Here a
// wave owns 32 queries (v_mfma_f32_32x32x16, the formulation of attn_fwd.hip:
// S^T = K Q^T, so a lane holds one query and 16 keys, and P^T is already the
// B operand of O^T += V^T P^T), which halves those bytes:
//
//  * A work item is 128 queries of one (batch, head). Two streams of four waves
//    take alternate 32-key tiles of its range, so each SIMD holds two waves
//    and one's softmax runs beside the other's MFMAs; Q (64 VGPRs) and the
//    accumulators (128) stay in registers.
//  * Tiles land by LDS DMA as whole 512-byte rows, two stages per stream (128
//    KB); 16-byte chunk c of row r sits at c ^ swz_k(r) (K) or c ^ 4 swz_v(r)
//    (V): the prefill kernel's swizzles, conflict-free for the same reads. Q
//    arrives in the two second stages, before their first tiles.
//  * The streams swap halves of head_dim through LDS at the end (136 KB over
//    the stages, the workgroup's LDS), combine them with their maxima, and
//    store whole rows.
//
// 242 VGPRs, no spills. 2,048 queries, 16 heads, bf16: 149 -> 92 us (746
// TFLOP/s), bound by the serial S - softmax - PV of each wave and its rescale.
#include "attn_tile.h"

#include <float.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace dx {
namespace {

constexpr int kD = 256, kKS = kD / 16, kDT = kD / 32, kRB = 2 * kD;
constexpr int kWideN = 32;                   // keys per tile
constexpr int kTileB = kWideN * kRB;         // bytes of a K or V tile
constexpr int kStageB = 2 * kTileB;
constexpr int kStreamB = 2 * kStageB;        // two stages
constexpr int kHalf = kDT / 2;               // 32-wide head_dim blocks a stream keeps
constexpr int kHandV = 1 + 4 * kHalf;        // 16-byte vectors a lane hands over
constexpr int kWideLds = 2 * kHandV * 256 * 16 > 2 * kStreamB ? 2 * kHandV * 256 * 16 : 2 * kStreamB;

__device__ __forceinline__ int swz_k(int r) { return (r & 15) ^ ((r >> 4) & 1); }
__device__ __forceinline__ int swz_v(int r) { return (r & 3) ^ ((r >> 2) & 1); }

template <typename T>
__global__ __launch_bounds__(kWideThreads, 1) void attn_wide_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  prefetch_args(a);
  const AnyItem it = any_item(a, int(blockIdx.x));
  const int b = it.b, h = it.h, hk = h / a.kv_group;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int stream = wid >> 2, wave = wid & 3, lane = int(threadIdx.x) & 63;
  const int g = lane >> 5, n = lane & 31;
  const int cache_len = any_cache_len(a, b);
  const int q0 = it.qt * kWideQ;
  const int qi = q0 + wave * 32 + n;
  const bool qvalid = qi < a.Lq;
  const bool active = q0 + wave * 32 < a.Lq;  // wave-uniform
  const uint32_t lds = lds_addr(smem);

  // A DMA piece is two whole rows; lane l fills physical chunk l % 32 of row
  // l / 32 of it. Wave w of a stream sends pieces w, w + 4, w + 8, w + 12 of a
  // tile: rows 2 w + 8 i + l / 32 (the swizzles are linear in the row bits).
  const int lr = 2 * wave + g;
  const uint32_t kcol = uint32_t(n ^ swz_k(lr)), vcol = uint32_t(n ^ (4 * swz_v(lr)));

  // Q: rows 0..63 into stream 0's second stage, 64..127 into stream 1's (64
  // pieces, eight per wave); rows past Lq read as zeros. The descriptor covers
  // this item's rows only (q_rows_fit): all of a long q need not fit one.
  {
    const __amdgpu_buffer_rsrc_t rq =
        make_rsrc(a.q + b * a.q_sb + int64_t(q0) * a.q_sl + h * a.q_sh,
                  min(a.Lq - q0, kWideQ), int(a.q_sl) * 2, kD);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 64 * stream + 8 * i + lr;
      const uint32_t o = uint32_t(r) * uint32_t(a.q_sl) * 2 +
                         16u * (kcol ^ uint32_t(swz_k((8 * i) & 31)));
      dma_piece_at(rq, lds + stream * kStreamB + kStageB + (wave + 4 * i) * 1024,
                   q0 + r < a.Lq ? o : 0x80000000u);
    }
  }
  const EndBounds eb = end_bounds(a, q0, min(q0 + kWideQ, a.Lq) - 1);
  const int kv_min = cache_len + eb.lo, kv_max = cache_len + eb.hi;
  const int n_ct = (cache_len + kWideN - 1) / kWideN;  // tiles never straddle cache and new keys
  const int n_tiles = n_ct + (eb.hi + kWideN - 1) / kWideN;
  const int nt = (n_tiles - stream + 1) / 2;           // this stream's tiles
  const int iters = (n_tiles + 1) / 2;                 // barrier rounds
  const int c_ss2 = int(a.c_ss) * 2, k_sl2 = int(a.k_sl) * 2, v_sl2 = int(a.v_sl) * 2;
  const int64_t coff = b * a.c_sb + hk * a.c_sh;
  const __amdgpu_buffer_rsrc_t kc = make_rsrc(a.ck ? a.ck + coff : a.q, cache_len, c_ss2, kD);
  const __amdgpu_buffer_rsrc_t vc = make_rsrc(a.cv ? a.cv + coff : a.q, cache_len, c_ss2, kD);
  const __amdgpu_buffer_rsrc_t kn =
      make_rsrc(a.k + b * a.k_sb + hk * a.k_sh, kv_max - cache_len, k_sl2, kD);
  const __amdgpu_buffer_rsrc_t vn =
      make_rsrc(a.v + b * a.v_sb + hk * a.v_sh, kv_max - cache_len, v_sl2, kD);
  const uint32_t base = lds + stream * kStreamB;
  auto send = [&](int i) __attribute__((always_inline)) {
    const int t = 2 * i + stream;
    const bool in_cache = t < n_ct;
    const __amdgpu_buffer_rsrc_t rk = in_cache ? kc : kn, rv = in_cache ? vc : vn;
    const uint32_t sk = uint32_t(in_cache ? c_ss2 : k_sl2), sv = uint32_t(in_cache ? c_ss2 : v_sl2);
    const uint32_t row = uint32_t(in_cache ? t : t - n_ct) * kWideN + uint32_t(lr);
    const uint32_t ko = row * sk, vo = row * sv;
    const uint32_t at = base + (i & 1) * kStageB + wave * 1024;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      dma_piece_at(rk, at + p * 4096, ko + 8u * p * sk + 16u * (kcol ^ uint32_t(swz_k(8 * p))));
      dma_piece_at(rv, at + kTileB + p * 4096, vo + 8u * p * sv + 16u * vcol);
    }
  };
  if (nt > 0) send(0);
  const int my_end = qvalid ? cache_len + visible_end(a, qi, cache_len) : 0;

  wait_vmcnt<0>();
  __syncthreads();
  u32x4 qr[kKS];
  const float cs = a.scale_log2;  // signed
  {
    const uint32_t flip = cs < 0.f ? 0x80008000u : 0u;  // exact sign flip of both halves
    const uint32_t qa = lds + (wave >> 1) * kStreamB + kStageB + ((wave & 1) * 32 + n) * kRB;
#pragma unroll
    for (int s = 0; s < kKS; ++s)
      qr[s] = lds_read_b128_at(qa + 16 * ((2 * s + g) ^ swz_k(n))) ^ flip;
  }
  __syncthreads();  // Q read before the second stages' first tiles
  // c > 0: masked scores are -inf and exp2(-inf c) has to be 0 (a zero scale
  // weighs every visible key alike: exp2(~0)).
  const float c = fmaxf(fabsf(cs), FLT_MIN);

  // Operand addresses in stage 0 (see PairAddr in attn_fwd.hip): K row n,
  // chunk (2 s + g) ^ swz_k(n) = ((g ^ swz_k(n)) ^ 2 s); V rows r0 + 8 e + 16
  // u, 64-byte column group d ^ swz_v(r0).
  const int j = lane & 15, r0 = 4 * g + (j >> 2);
  const uint32_t ka = base + n * kRB + 16 * (g ^ swz_k(n));
  const uint32_t va =
      base + kTileB + r0 * kRB + 32 * ((lane >> 4) & 1) + 8 * (j & 3) + 64 * swz_v(r0);

  f32x16 acc[kDT];
#pragma unroll
  for (int d = 0; d < kDT; ++d) acc[d] = f32x16{};
  float m = -INFINITY, l = 0.f;
  for (int i = 0; i < iters; ++i) {
    if (i > 0) {
      // This wave's pieces of tile i; past the barrier the tile is whole and
      // the other stage's reads (tile i - 1) have returned.
      wait_vmcnt<0>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (i + 1 < nt) send(i + 1);
    if (i >= nt || !active) continue;
    const uint32_t st = (i & 1) * kStageB;
    f32x16 s = f32x16{};
#pragma unroll
    for (int k = 0; k < kKS; ++k)
      s = Mfma<T>::run(lds_read_b128_at((ka + st) ^ (32u * k)), qr[k], s);
    const int t = 2 * i + stream;
    const bool in_cache = t < n_ct;
    const int j0 = in_cache ? t * kWideN : cache_len + (t - n_ct) * kWideN;
    if (in_cache ? j0 + kWideN > cache_len : j0 + kWideN > kv_min) {
      int lim = (in_cache ? cache_len - j0 : my_end - j0) - 4 * g;
      asm volatile("" : "+v"(lim));
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (key_hidden(0, r, lim)) s[r] = -INFINITY;
    }
    float tm[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int r = 0; r < 16; ++r) tm[r % 4] = fmaxf(tm[r % 4], s[r]);
    const float m_new = fmaxf(m, xor32_max(fmaxf(fmaxf(tm[0], tm[1]), fmaxf(tm[2], tm[3]))));
    // The reference follows the maximum exactly (softmax_max in attn_fwd.hip
    // lets it lag by up to 2^8): the largest probability is 1, which 16 bits
    // hold exactly. 2,048 keys: error against 64 bits 2.22e-3 (2.33e-3 lagging,
    // 2.25e-3 from attn_any16_kernel) for 10% of the call.
    if (__any(m_new > m)) {
      if (!__all(m == -INFINITY)) {
        const float corr = m == -INFINITY ? 0.f : fast_exp2((m - m_new) * c);
        l *= corr;
#pragma unroll
        for (int d = 0; d < kDT; ++d) acc[d] *= corr;
      }
      m = m_new;
    }
    const float mb = m == -INFINITY ? 0.f : m * c;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(__builtin_fmaf(s[r], c, -mb));
    u32x4 pk[2];
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t p = Mfma<T>::pack(s[8 * u + 2 * e], s[8 * u + 2 * e + 1]);
        pk[u][e] = p;
        part[e & 1] = Mfma<T>::sum2(p, part[e & 1]);
      }
    l += part[0] + part[1];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int d = 0; d < kDT; ++d) {
        const uint32_t vu = ((va + st) ^ (64u * d)) + 16 * u * kRB;
        const u32x2 lo = lds_read_tr16_at(vu);
        const u32x2 hi = lds_read_tr16_at(vu + 8 * kRB);
        acc[d] = Mfma<T>::run(u32x4{lo[0], lo[1], hi[0], hi[1]}, pk[u], acc[d]);
      }
  }

  // Stream s keeps head_dim blocks [4 s, 4 s + 4) and hands (m, l) and the
  // others to the same lane of the other stream ([vector][lane]); both then
  // combine with the same weights, stream 0's terms first. The stream enters
  // as a constant, so that every block index is static.
  const float mref = m == -INFINITY ? -INFINITY : m * c;
  f32x4* const x = reinterpret_cast<f32x4*>(smem);
  const int ltid = wave * 64 + lane;
  auto finish = [&](auto stream_c) __attribute__((always_inline)) {
    constexpr int S = decltype(stream_c)::value;
    __syncthreads();  // every tile read is done
    f32x4* const hand = x + S * kHandV * 256;
    const f32x4* const got = x + (1 - S) * kHandV * 256;
    hand[ltid] = f32x4{mref, l, 0.f, 0.f};
#pragma unroll
    for (int dd = 0; dd < kHalf; ++dd)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16& v = acc[(1 - S) * kHalf + dd];
        hand[(1 + 4 * dd + q) * 256 + ltid] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
    __syncthreads();
    const f32x4 o = got[ltid];
    const float m0 = S == 0 ? mref : o[0], m1 = S == 0 ? o[0] : mref;
    const float l0 = S == 0 ? l : o[1], l1 = S == 0 ? o[1] : l;
    const float mm = fmaxf(m0, m1), ref = mm == -INFINITY ? 0.f : mm;
    const float w0 = fast_exp2(m0 - ref), w1 = fast_exp2(m1 - ref);
    // No visible key: 0 * inf = NaN, as the reference's softmax.
    const float inv = 1.0f / xor32_sum(__builtin_fmaf(l0, w0, l1 * w1));
#pragma unroll
    for (int dd = 0; dd < kHalf; ++dd)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = got[(1 + 4 * dd + q) * 256 + ltid];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float own = acc[S * kHalf + dd][4 * q + e];
          const float a0 = S == 0 ? own : v[e], a1 = S == 0 ? v[e] : own;
          acc[S * kHalf + dd][4 * q + e] = __builtin_fmaf(a0, w0, a1 * w1) * inv;
        }
      }
    __syncthreads();  // the hand-over is read: its space takes the result rows
    const uint32_t row = lds + (wave * 32 + n) * kRB;
#pragma unroll
    for (int dd = 0; dd < kHalf; ++dd)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16& v = acc[S * kHalf + dd];
        typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
        *reinterpret_cast<lds_u32x2*>(row + 16 * ((4 * (S * kHalf + dd) + q) ^ swz_k(n)) + 8 * g) =
            u32x2{Mfma<T>::pack(v[4 * q], v[4 * q + 1]), Mfma<T>::pack(v[4 * q + 2], v[4 * q + 3])};
      }
  };
  if (stream == 0) finish(std::integral_constant<int, 0>{});
  else finish(std::integral_constant<int, 1>{});
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 16 * i + int(threadIdx.x) / 32, ch = int(threadIdx.x) % 32;
    if (q0 + r < a.Lq)
      *reinterpret_cast<u32x4*>(a.out + b * a.o_sb + int64_t(q0 + r) * a.o_sl + h * a.o_sh + 8 * ch) =
          lds_read_b128_at(lds + r * kRB + 16 * (ch ^ swz_k(r & 31)));
  }
}

template <typename T>
hipError_t launch_wide_t(const AttnArgs& a, hipStream_t st) {
  const void* fn = reinterpret_cast<const void*>(&attn_wide_kernel<T>);
  const hipError_t e = opt_in_lds(fn, kWideLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((attn_wide_kernel<T>), dim3(unsigned(int64_t(a.B) * a.H * a.n_qtiles)),
                     dim3(kWideThreads), kWideLds, st, a);
  return hipGetLastError();
}

}  // namespace

// Modelled times (us) of this kernel and of attn_any16_kernel, by 32-key tiles:
//  * here: rounds of one workgroup per CU, 9.5 each, and 0.89 a tile of a CU's
//    items in turn (rounds x the mean item, or the longest one), up to 1.4
//    where every CU has work throughout;
//  * there: 7.6 (16.3 when it splits the keys and merges), 6 ns per tile of
//    every 64-query item, and 12 ns per item for its queries and results.
// Measured over 1 to 128 sequences, 1 to 32,768 queries and 16 to 8,000 keys
// (cold, us per call, that kernel -> this one). Here: 16 heads x 2048 155 -> 91;
// 24 heads x 1000 81 -> 48, causal 59 -> 46; 16 heads x 400 31 -> 23; 64 heads
// x 8192 over 128 keys 226 -> 209; 8 x 16 heads, 200 over 2000 160 -> 101; 32 x
// 16 heads, 83 over 8000 1376 -> 699. There: 8 heads x 1000 causal 34 -> 41, 24
// heads x 300 over 2000 57 -> 84; 8 x 16 heads, 64 over 8000 209 -> 278; 17 x 16
// heads, 16 over 500 49 -> 63 and 64 over 8000 497 -> 591; 64 x 16 heads, 1 over
// 100 36 -> 53. Wrong by more than 3% at three of 165: 8 x 16 heads, 16 over 500
// (30 for 29), and 40 x 16 heads (4 K/V) over 4000, 1 query (398 for 353) and 32
// (402 for 378).
bool wide_fits(int64_t B, int64_t Lq, int64_t Lk, int64_t H, int64_t cache_len,
               const int64_t* cache_lens, int64_t n_blocks, bool causal, int splits, int cus) {
  auto tiles = [](int64_t keys) { return double((keys + kWideN - 1) / kWideN); };
  double seen = tiles(Lk);  // mean new-key tiles of an item
  if (causal) seen = (seen + 1) / 2;
  else if (n_blocks > 1) seen *= double(n_blocks + 1) / double(2 * n_blocks);
  double longest = 0, mean = 0;
  for (int64_t i = 0; i < (cache_lens ? B : 1); ++i) {
    const double c = tiles(cache_lens ? cache_lens[i] : cache_len);
    longest = std::max(longest, c);
    mean += (c + seen) / double(cache_lens ? B : 1);
  }
  longest += tiles(Lk);
  const double items = double(B * H * ((Lq + kWideQ - 1) / kWideQ));
  const double rounds = std::ceil(items / cus), serial = std::max(longest, rounds * mean);
  const double here = 9.5 * rounds + (0.89 + 0.51 * items * mean / (cus * serial)) * serial;
  const int64_t tiles64 = (Lq + 63) / 64;
  const double there = (splits > 1 ? 16.3 : 7.6) +
                       double(B * H) * (0.006 * double(tiles64) * mean + 0.012 * double(Lq) / 64);
  return here <= there;
}

hipError_t launch_wide(AttnArgs a, int dtype, hipStream_t st) {
  a.n_qtiles = (a.Lq + kWideQ - 1) / kWideQ;
  a.n_splits = 1;
  return dtype == DX_BF16 ? launch_wide_t<bf16_t>(a, st) : launch_wide_t<f16_t>(a, st);
}

}  // namespace dx
