// Blockwise-causal attention for fp32 inputs, key tiles dealt to a workgroup's
// waves (gfx950; the semantics of attn_fwd.hip, the arithmetic of
// attn_any_kernel: fp32 MFMA, fp32 softmax).
//
// attn_any_kernel deals 64-query items of four waves, one per SIMD, and splits
// the keys only as far as the call's workspace holds fp32 partials: 332 queries
// x 24 heads over 1,328 keys are 144 items on 256 CUs, each wave alone on its
// SIMD, 23% of the fp32 MFMA rate. Here a work item is 16 QT queries of one
// (batch, head) and each of its NW waves takes key tiles w, w + NW, ... of 16
// keys, with its own online softmax, its own LDS tile and its own waits (the
// form of attn_wave_kernel): four or two times the items, two waves per SIMD,
// and no partials in memory.
//
//  * Products: v_mfma_f32_16x16x4_f32, S^T = K Q^T (keys on M, queries on N),
//    so a lane holds one query and four keys, and the probabilities are already
//    the B operand of O^T += V^T P^T. MFMA step j of head_dim group u takes
//    element 16 u + 4 g + j from lane group g, so K and q are read as float4.
//  * Tiles land by LDS DMA as whole rows, 16-byte chunk c of row r at c ^ f(r),
//    conflict-free for the K reads (16 rows, one chunk each) and the V reads
//    (16 floats of four rows). A wave refills its K part once the scores are
//    computed and its V part after PV; the other wave of the SIMD computes
//    meanwhile.
//  * Merge: the waves scale their sums to the common maximum and 1 / sum and
//    add them in wave order through LDS.
//
// 332 queries over 996 + 332 keys in 83-token blocks, 24 heads x 128: 136 -> 62
// us (79 TFLOP/s of 157 in fp32 MFMA), and the error against 64 bits 7.4e-7 ->
// 3.7e-7 (shorter chains). Its 504 items run at once, two to a CU, one wave of
// each on a SIMD. Counters: the MFMA units are busy 46% of the launch; a wave
// waits 27% of its time for its tiles and 51% to issue, behind its own and the
// other wave's dependent chains; a SIMD holds 1.56 of its two waves on average
// (items see 69 to 84 tiles). Measured and left out, with cold K/V: tiles (V
// alone) by registers instead of DMA 81 (78) against 74 us, the query rows
// through LDS 74.
#include "attn_tile.h"

#include <algorithm>
#include <cmath>

namespace dx {
namespace {

constexpr int kKeys = 16;  // keys per tile

template <int D, int QT, int NW> struct F32Shape {
  static constexpr int RB = 4 * D, CR = D / 4;          // bytes, 16-byte chunks per row
  static constexpr int RPP = 64 / CR;                   // rows per DMA piece
  static constexpr int tile = kKeys * RB;
  static constexpr int NP = tile / 1024;                // pieces per K (or V) tile
  static constexpr int wave = 2 * tile;
  static constexpr int rows = 16 * QT;                  // queries per item
  static constexpr int part = rows * RB;                // one wave's result, over the tiles
  static constexpr int ml = NW * std::max(wave, part);  // [NW][rows] {m, l}
  static constexpr int bytes = ml + NW * rows * 8;
  static_assert(bytes <= 160 * 1024, "one workgroup's LDS");
  static __device__ __forceinline__ int swz(int r) { return CR >= 16 ? r & 15 : (r >> 1) & 7; }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rsrc(const float* base, int rows,
                                                          int row_bytes, int D) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0,
                                           rows > 0 ? (rows - 1) * row_bytes + D * 4 : 0,
                                           kBufWord3);
}

template <int D, int QT, int NW>
__global__ __launch_bounds__(64 * NW, 1) void attn_f32_kernel(AttnArgs a) {
  using S = F32Shape<D, QT, NW>;
  constexpr int RB = S::RB, NP = S::NP, DG = D / 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  prefetch_args(a);
  const AnyItem it = any_item(a, int(blockIdx.x));
  const int b = it.b, h = it.h, hk = h / a.kv_group;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int lane = int(threadIdx.x) & 63, g = lane >> 4, c = lane & 15;
  const int cache_len = any_cache_len(a, b);
  const int q0 = it.qt * S::rows;

  const EndBounds eb = end_bounds(a, q0, min(q0 + S::rows, a.Lq) - 1);
  const int kv_min = cache_len + eb.lo, kv_max = cache_len + eb.hi;
  const int n_ct = (cache_len + kKeys - 1) / kKeys;  // tiles never straddle cache and new keys
  const int n_tiles = n_ct + (eb.hi + kKeys - 1) / kKeys;
  const int nt = n_tiles > wid ? (n_tiles - wid + NW - 1) / NW : 0;  // this wave's tiles
  const int c_ss4 = int(a.c_ss) * 4, k_sl4 = int(a.k_sl) * 4, v_sl4 = int(a.v_sl) * 4;
  const float* const fq = reinterpret_cast<const float*>(a.q);
  const float* const ck = reinterpret_cast<const float*>(a.ck);
  const float* const cv = reinterpret_cast<const float*>(a.cv);
  const int64_t coff = b * a.c_sb + hk * a.c_sh;
  const __amdgpu_buffer_rsrc_t kc = f32_rsrc(ck ? ck + coff : fq, cache_len, c_ss4, D);
  const __amdgpu_buffer_rsrc_t vc = f32_rsrc(cv ? cv + coff : fq, cache_len, c_ss4, D);
  const __amdgpu_buffer_rsrc_t kn =
      f32_rsrc(reinterpret_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh,
               kv_max - cache_len, k_sl4, D);
  const __amdgpu_buffer_rsrc_t vn =
      f32_rsrc(reinterpret_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh,
               kv_max - cache_len, v_sl4, D);

  // A DMA piece is RPP whole rows; lane l fills physical chunk l % CR of row
  // l / CR of it (f is linear in the row bits, so a piece XORs a constant).
  const int lr = lane / S::CR;
  const uint32_t col = uint32_t((lane % S::CR) ^ S::swz(lr));
  const uint32_t base = lds_addr(smem) + wid * S::wave;
  auto send = [&](int i, bool is_k) __attribute__((always_inline)) {
    const int t = wid + NW * i;
    const bool in_cache = t < n_ct;
    const __amdgpu_buffer_rsrc_t r = is_k ? (in_cache ? kc : kn) : (in_cache ? vc : vn);
    const uint32_t stride = uint32_t(in_cache ? c_ss4 : (is_k ? k_sl4 : v_sl4));
    const uint32_t row = (uint32_t(in_cache ? t : t - n_ct) * kKeys + uint32_t(lr)) * stride;
    const uint32_t at = base + (is_k ? 0 : S::tile);
#pragma unroll
    for (int p = 0; p < NP; ++p)
      dma_piece_at(r, at + p * 1024,
                   row + uint32_t(p * S::RPP) * stride + 16u * (col ^ uint32_t(S::swz(p * S::RPP))));
  };

  // q, pre-scaled: q[t][u][j] = query 16 t + c, element 16 u + 4 g + j. Rows
  // past Lq read the last row and become zeros (no branch between the loads).
  f32x4 q[QT][DG];
  int end[QT];  // keys visible to the lane's queries
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int qi = q0 + 16 * t + c;
    const float* row = fq + b * a.q_sb + int64_t(min(qi, a.Lq - 1)) * a.q_sl + h * a.q_sh;
#pragma unroll
    for (int u = 0; u < DG; ++u) q[t][u] = *reinterpret_cast<const f32x4*>(row + 16 * u + 4 * g);
  }
  if (nt > 0) {
    send(0, true);
    send(0, false);
  }
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int qi = q0 + 16 * t + c;
    const float qs = qi < a.Lq ? a.scale_log2 : 0.f;
    end[t] = qi < a.Lq ? cache_len + visible_end(a, qi, cache_len) : 0;
#pragma unroll
    for (int u = 0; u < DG; ++u) q[t][u] *= qs;
  }
  const uint32_t ka = base + c * RB + 16 * (g ^ S::swz(c));  // chunk 4 u + g: XOR 64 u
  uint32_t va[4];                                            // row 4 g + j, floats 16 u + c
#pragma unroll
  for (int j = 0; j < 4; ++j)
    va[j] = base + S::tile + (4 * g + j) * RB + 16 * ((c >> 2) ^ S::swz(4 * g + j)) + 4 * (c & 3);
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
  typedef __attribute__((address_space(3))) float lds_f32;

  const float kNegInf = -__builtin_inff();
  f32x4 o[QT][DG];
  float m[QT], l[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m[t] = kNegInf;
    l[t] = 0.f;
#pragma unroll
    for (int u = 0; u < DG; ++u) o[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int i = 0; i < nt; ++i) {
    const int tile = wid + NW * i;
    wait_vmcnt<NP>();  // K landed; behind it this tile's V
    // Four chains, so that no MFMA waits for the one before it.
    constexpr int NC = 4 / QT;
    f32x4 sc[QT][NC];
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int x = 0; x < NC; ++x) sc[t][x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < DG; ++u) {
      const f32x4 kv = *reinterpret_cast<const lds_f32x4*>(ka ^ (64u * u));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < QT; ++t) sc[t][j % NC] = mfma4(kv[j], q[t][u][j], sc[t][j % NC]);
    }
    const bool more = i + 1 < nt;
    if (more) {
      // The K reads have returned (the MFMAs took them): refill.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      send(i + 1, true);
    }
    const bool in_cache = tile < n_ct;
    const int j0 = in_cache ? tile * kKeys : cache_len + (tile - n_ct) * kKeys;
    const bool masked = in_cache ? j0 + kKeys > cache_len : j0 + kKeys > kv_min;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      f32x4 s = sc[t][0] + sc[t][1];
      if constexpr (NC == 4) s += sc[t][2] + sc[t][3];
      if (masked) {
        const int lim = (in_cache ? cache_len : end[t]) - j0 - 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = r < lim ? s[r] : kNegInf;
      }
      const float mn = fmaxf(m[t], quad_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
      const float ref = mn == kNegInf ? 0.f : mn;  // nothing visible yet: every p is 0
      if (__any(mn > m[t])) {
        const float corr = fast_exp2(m[t] - ref);
        l[t] *= corr;
#pragma unroll
        for (int u = 0; u < DG; ++u) o[t][u] *= corr;
      }
      m[t] = mn;
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = fast_exp2(s[r] - ref);
      l[t] += (s[0] + s[1]) + (s[2] + s[3]);
      sc[t][0] = s;
    }
    if (more) wait_vmcnt<NP>();  // V landed; behind it the next K
    else wait_vmcnt<0>();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < DG; ++u) {
        const float v = *reinterpret_cast<const lds_f32*>(va[j] ^ (64u * u));
#pragma unroll
        for (int t = 0; t < QT; ++t) o[t][u] = mfma4(v, sc[t][0][j], o[t][u]);
      }
    if (more) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      send(i + 1, false);
    }
  }

  // Merge over the waves that had tiles (at least wave 0, whose empty result
  // makes a query with no visible key NaN: 0 * inf, as the reference).
  const int used = min(NW, max(n_tiles, 1));
  f32x2* const ml = reinterpret_cast<f32x2*>(smem + S::ml);
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    l[t] = quad_sum(l[t]);
    if (g == 0) ml[wid * S::rows + 16 * t + c] = f32x2{m[t], l[t]};
  }
  __syncthreads();  // every wave's tile reads and DMA pieces are done too
  if (wid < used) {
    f32x4* const mine = reinterpret_cast<f32x4*>(smem + wid * S::part);
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const int row = 16 * t + c;
      f32x2 w[NW];
      float mm = kNegInf;
#pragma unroll
      for (int x = 0; x < NW; ++x) {
        w[x] = x < used ? ml[x * S::rows + row] : f32x2{kNegInf, 0.f};
        mm = fmaxf(mm, w[x][0]);
      }
      const float ref = mm == kNegInf ? 0.f : mm;
      float sum = 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) sum += fast_exp2(w[x][0] - ref) * w[x][1];
      const float k = fast_exp2(m[t] - ref) * (1.0f / sum);
      // Row 4 u + g of float4s holds the queries, query q at slot q ^ (row % 16).
#pragma unroll
      for (int u = 0; u < DG; ++u) {
        const int d4 = 4 * u + g;
        mine[d4 * S::rows + (row ^ (d4 & 15))] = o[t][u] * k;
      }
    }
  }
  __syncthreads();
  const f32x4* const all = reinterpret_cast<const f32x4*>(smem);
  float* const out = reinterpret_cast<float*>(a.out) + b * a.o_sb + h * a.o_sh;
  for (int x = int(threadIdx.x); x < S::rows * S::CR; x += 64 * NW) {
    const int row = x / S::CR, d4 = x % S::CR;
    const int slot = d4 * S::rows + (row ^ (d4 & 15));
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < used; ++w) v += all[w * (S::part / 16) + slot];
    if (q0 + row < a.Lq)
      *reinterpret_cast<f32x4*>(out + int64_t(q0 + row) * a.o_sl + 4 * d4) = v;
  }
}

template <int D, int QT, int NW>
hipError_t launch_dq(const AttnArgs& a, hipStream_t st) {
  using S = F32Shape<D, QT, NW>;
  const hipError_t e =
      opt_in_lds(reinterpret_cast<const void*>(&attn_f32_kernel<D, QT, NW>), S::bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((attn_f32_kernel<D, QT, NW>), dim3(unsigned(int64_t(a.B) * a.H * a.n_qtiles)),
                     dim3(64 * NW), S::bytes, st, a);
  return hipGetLastError();
}

template <int D>
hipError_t launch_d(const AttnArgs& a, const F32Plan& p, hipStream_t st) {
  if constexpr (D < 256) {
    if (p.waves == 8) return launch_dq<D, 1, 8>(a, st);
    if (p.qt == 2) return launch_dq<D, 2, 4>(a, st);
  }
  return launch_dq<D, 1, 4>(a, st);
}

}  // namespace

// Form by the 16-query items I: eight waves up to one item per CU; four waves
// up to 2.75 per CU; two query tiles per item past that, where there are items
// enough and K/V traffic counts (24 heads x 664 queries, D 128: 61 us against 72
// with one tile), and the second tile is not empty (32 x 24 heads, 16 queries
// over 500 cached keys: 100 us with it, 94 without; 24 queries 103 against
// 168). D 256 has LDS for four waves and one tile.
//
// Whether the call goes here at all: modelled times (us, s = D / 128) of the
// form and of attn_any_kernel. A CU's n items take the longest of: one wave's
// own chain of tiles, the matrix units' time for the tiles of all n, and the
// call's K/V from HBM at 5.8 TB/s, once, or once per round of resident items
// where it exceeds the 256 MB cache (a head's query tiles run in different
// rounds); then a fixed time, and one per item:
//                      fixed     chain         all          item
//   eight waves        8.8       3.3 s         -            -
//   four               5.9       0.6 + 1.3 s   1.45 s       0.15 + 1.8 s
//   four, two tiles    5.0       0.4 + 2.1 s   0.05 + 2.1 s 1.6 + 3.3 s
//   attn_any_kernel    4.9 (+ 7.1 s if split)  0.5 + 2.6 s  2.65 s  3.2
// by 16-key tiles dealt to an item's waves, or (attn_any_kernel, 64 queries an
// item, 32-key tiles) to its key splits. K/V counts a head's per query head.
// Fitted to 950 calls (1 to 64 sequences, 1 to 8000 queries, 16 to 4500 keys, D
// 32 to 256): nine of them run more than 3% slower than on the general kernel,
// and 22 would be that much faster here. Cold, us, that kernel -> this one, D
// 128: 332 x 24 heads over 996 in blocks of 83 136 -> 67; 400 x 24 over 500 96
// -> 77; 83 x 24 over 512 keys 36 -> 21; 2500 x 12 heads 416 -> 360. Stays: one
// query, 24 heads over 1000 23.5 (30.5 here); 4 x 24 heads, 300 onto 64 keys
// 23.6 (28.5); 32 x 16 heads, 64 over 1000 197 (220); 24 heads, 2000 onto 128
// keys 47 (53); 64 heads, 4000 onto 16 83 (145); D 256, 32 x 16 heads, 40 over
// 1000 423 (561). D 16 is not measured and stays.
F32Plan plan_f32(int64_t B, int64_t Lq, int64_t Lk, int64_t H, int64_t D, int64_t cache_len,
                 const int64_t* cache_lens, int64_t n_blocks, bool causal, int splits, int cus,
                 int form) {
  F32Plan p{};
  if (D < 32) return p;
  auto cdiv = [](int64_t x, int64_t y) { return (x + y - 1) / y; };
  const int64_t items = B * H * cdiv(Lq, 16);
  p.waves = D < 256 && items <= cus ? 8 : 4;
  p.qt = D < 256 && 4 * items > 11 * int64_t(cus) && Lq > 16 ? 2 : 1;
  if (form) {
    p.waves = D < 256 && form == 8 ? 8 : 4;
    p.qt = D < 256 && form == 2 ? 2 : 1;
  }
  const int64_t blocks = B * H * cdiv(Lq, 16 * p.qt);
  if (!grid_fits(blocks, 64 * p.waves)) return p;
  p.fits = form != 0;
  if (form) return p;

  // 16- and 32-key tiles of the mean item and of the longest one.
  double mean[2], longest[2];
  for (int k = 0; k < 2; ++k) {
    const int64_t keys = 16 << k;
    double seen = double(cdiv(Lk, keys));
    longest[k] = mean[k] = 0;
    for (int64_t i = 0; i < (cache_lens ? B : 1); ++i) {
      const double c = double(cdiv(cache_lens ? cache_lens[i] : cache_len, keys));
      longest[k] = std::max(longest[k], c);
      mean[k] += c / double(cache_lens ? B : 1);
    }
    longest[k] += seen;
    if (causal) seen = (seen + 1) / 2;
    else if (n_blocks > 1) seen *= double(n_blocks + 1) / double(2 * n_blocks);
    mean[k] += seen;
  }
  const double s = double(D) / 128, kv_bytes = double(B * H) * mean[0] * 16 * double(D) * 8;
  // Resident workgroups per CU: by LDS, or the two-tile form's registers.
  const double by_lds = 256.0 / double(D), by_regs = 1 + 128.0 / double(D);
  auto time = [&](int k, double workgroups, double per_cu, int64_t q_tiles, double parts,
                  double fixed, double chain, double all, double item) {
    const double n = std::ceil(workgroups / cus), rounds = std::ceil(workgroups / (per_cu * cus));
    const double reads = kv_bytes > 256e6 ? std::min(double(q_tiles), rounds) : 1;
    const double tiles = std::max(std::ceil(longest[k] / parts) * chain,
                                  n * std::ceil(mean[k] / parts) * all);
    return fixed + std::max(tiles, reads * kv_bytes / 5.8e6) + n * item;
  };
  const int64_t q_tiles = cdiv(Lq, 16 * p.qt), q_tiles64 = cdiv(Lq, 64);
  const double here =
      p.waves == 8 ? time(0, double(blocks), by_lds, q_tiles, 8, 8.8, 3.3 * s, 0, 0)
      : p.qt == 1  ? time(0, double(blocks), by_lds, q_tiles, 4, 5.9, 0.6 + 1.3 * s, 1.45 * s,
                          0.15 + 1.8 * s)
                   : time(0, double(blocks), by_regs, q_tiles, 4, 5.0, 0.4 + 2.1 * s,
                          0.05 + 2.1 * s, 1.6 + 3.3 * s);
  const double there =
      time(1, double(B * H * q_tiles64 * splits), by_lds, q_tiles64, splits,
           4.9 + (splits > 1 ? 7.1 * s : 0), 0.5 + 2.6 * s, 2.65 * s, 3.2);
  p.fits = here <= there;
  return p;
}

hipError_t launch_f32(AttnArgs a, int D, const F32Plan& p, hipStream_t st) {
  a.n_qtiles = (a.Lq + 16 * p.qt - 1) / (16 * p.qt);
  a.n_splits = 1;
  switch (D) {
    case 32: return launch_d<32>(a, p, st);
    case 64: return launch_d<64>(a, p, st);
    case 128: return launch_d<128>(a, p, st);
    default: return launch_d<256>(a, p, st);
  }
}

}  // namespace dx
