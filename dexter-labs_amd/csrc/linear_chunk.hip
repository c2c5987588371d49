// Projection of a decode-sized chunk (M <= 128 tokens) on gfx950:
// y = x W^T + b, nn.Linear's, rounded once (the output projection of
// SelfAttention.forward, models/dreamzero/model.py:183, on gfx1151 hipBLASLt
// through ops/gfx1151/gemm).
//
// 83 tokens over a 3072 x 3072 weight are a weight stream (18.9 MB) whose
// activations (0.5 MB) every workgroup reads again from L2. A CU takes in
// about 60 GB/s of the two together, so the split minimises the rows a CU
// reads, weights and tokens alike, and leaves no partial product in memory:
//
//  * A workgroup owns NT tiles of 16 output features and NM of 16 tokens over
//    the whole reduction. Past 64 tokens there are two token groups: 32
//    features x 48 tokens at the Wan-5B chunk (192 workgroups of 80 rows; 16
//    features x 96 tokens, 112 rows: 12.9 against 11.8 us a call). The groups
//    of one feature set share an XCD, so its weights leave HBM once.
//  * Weights and activations land in LDS by DMA in chunks of 128 reduction
//    elements, 256 contiguous bytes per row, NS stages deep; one barrier per
//    chunk publishes a stage and frees the oldest. (Loaded straight into the
//    operand layout, 16 rows x 64 bytes per instruction, rows come in at a
//    quarter of the rate: 21.6 us a call.)
//  * Eight waves: wave w takes MFMA step w % 4 of every chunk (32 elements,
//    v_mfma_f32_16x16x32, features on M, tokens on N) and half w / 4 of the
//    token tiles (of the feature tiles where the token tiles are odd in
//    number). A chunk's operand reads run behind the previous chunk's MFMAs.
//  * The four steps' sums meet in LDS at the end, added in step order (the
//    same bits on every run), then the bias, then one rounding.
//
// Measured per call, cold weights, against hipBLASLt (graph of 20 calls):
// 3072 x 3072: 83 tokens 11.8 us (16.7), 128 13.1 (20.0), 32 9.8 (11.0);
// 1536 x 1536: 83 tokens 6.6 (7.4), 24 5.4 (7.2). At 5120 x 5120 the two are
// mixed (64 tokens 22.2 against 22.5, 83 24.6 against 22.6), so the model
// takes this kernel up to 4096 features.
#include "attn_tile.h"

#include <algorithm>

namespace dx {
namespace {

struct LinearArgs {
  const uint16_t* x; int64_t x_sb, x_sl;  // activation [B][L][C], element strides
  const uint16_t* w; int64_t w_row;       // weight [N][C], row stride in elements
  const uint16_t* bias;                   // [N], may be null
  uint16_t* y;                            // contiguous [B L][N]
  int M, L, C, N;                         // tokens, L, in and out features
  int groups;                             // token groups
};

constexpr int kWaves = 8;
constexpr int kSteps = 4;                  // MFMA steps (of 32) per chunk
constexpr int kChunkK = 32 * kSteps;       // reduction elements per chunk
constexpr int kRowB = 2 * kChunkK;         // bytes per staged row
constexpr int kPieceRows = 1024 / kRowB;   // rows per DMA piece

template <int NT, int NM> struct LinearLds {
  static constexpr int rows = 16 * (NT + NM);
  static constexpr int stage = rows * kRowB;
  static constexpr int NS = std::min(8, 160 * 1024 / stage);
  static constexpr int sums = kSteps * NT * NM * 1024;  // the waves' results, over the stages
  static constexpr int bytes = std::max(NS * stage, sums);
  static_assert(NS >= 3 && bytes <= 160 * 1024, "three stages at least");
};

template <typename T, int NT, int NM>
__global__ __launch_bounds__(64 * kWaves, 1) void linear_chunk_kernel(LinearArgs a) {
  using L = LinearLds<NT, NM>;
  constexpr int NS = L::NS;
  // Waves 4..7 take the second half of the token tiles, or of the feature
  // tiles where the token tiles are odd in number.
  constexpr bool kTok = NM % 2 == 0;
  constexpr int NF = kTok ? NT : NT / 2, NH = kTok ? NM / 2 : NM;
  static_assert(kTok || NT % 2 == 0, "one of the tile counts halves");
  constexpr int kWPieces = NT * 16 / kPieceRows;
  constexpr int kMaxSlots = (L::rows / kPieceRows + kWaves - 1) / kWaves;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds = lds_addr(smem);

  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int lane = int(threadIdx.x) & 63, n = lane & 15, g = lane >> 4;
  const int tiles = a.N / 16;
  // Token groups of one feature tile set run on one XCD (workgroup i runs on
  // XCD i % 8), where they share its weight rows through the L2.
  const int blk = int(blockIdx.x), set = 8 * a.groups;
  const int f0 = blk / set * 8 + blk % 8, grp = blk % set / 8;
  if (f0 * NT >= tiles) return;
  const int t0 = f0 * NT, m0 = grp * 16 * NM, rows = min(a.M - m0, 16 * NM);

  // DMA slots of this wave: pieces wid, wid + 8, ... of a stage (the weight
  // rows' pieces, then those of the token rows that exist; rows past the last
  // token in the last piece repeat it). Lane l fills physical 16-byte slot
  // l % 16 of row l / 16, so it fetches logical slot (l % 16) ^ (row % 16).
  const int pieces = kWPieces + (rows + kPieceRows - 1) / kPieceRows;
  const int slots = (pieces - wid + kWaves - 1) / kWaves;
  __amdgpu_buffer_rsrc_t rs[kMaxSlots];
  uint32_t off[kMaxSlots];
  const uint32_t x_bytes = uint32_t((int64_t((a.M - 1) / a.L) * a.x_sb +
                                     int64_t(min(a.L, a.M) - 1) * a.x_sl + a.C) * 2);
#pragma unroll
  for (int i = 0; i < kMaxSlots; ++i) {
    const int p = wid + kWaves * i;
    const int row = p * kPieceRows + g;  // of the stage
    const uint32_t col = uint32_t(16 * (n ^ (row & 15)));
    if (p < kWPieces) {
      const int t = min(t0 + p / 4, tiles - 1);
      rs[i] = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t*>(a.w + int64_t(t) * 16 * a.w_row), (short)0,
          int((15 * a.w_row + a.C) * 2), kBufWord3);
      off[i] = uint32_t(row & 15) * uint32_t(a.w_row) * 2 + col;
    } else {
      rs[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x), (short)0,
                                                int(x_bytes), kBufWord3);
      const uint32_t m = uint32_t(m0 + min(row - 16 * NT, rows - 1)), b = m / uint32_t(a.L);
      off[i] = uint32_t((int64_t(b) * a.x_sb + int64_t(m - b * uint32_t(a.L)) * a.x_sl) * 2) + col;
    }
  }
  const int chunks = a.C / kChunkK;
  auto send = [&](int c, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMaxSlots; ++i)
      if (i < slots)
        dma_piece_at(rs[i], lds + st * L::stage + (wid + kWaves * i) * 1024,
                     off[i] + uint32_t(c) * kRowB);
  };
  // This wave's pieces of every chunk but the last `later` sent have landed. The
  // wait's count is an immediate: one for each slot count a wave can have (with
  // fewer, waves of few slots drained the ring every chunk: five layers at 43
  // tokens x 3072 took 275 us instead of 243, 246 with hipBLASLt).
  auto landed = [&](int later) __attribute__((always_inline)) {
    const int left = later * slots;
    static_assert(kMaxSlots <= 4, "a rung per slot count");
    if (kMaxSlots >= 4 && left >= (NS - 2) * 4) wait_vmcnt<(NS - 2) * 4>();
    else if (kMaxSlots >= 3 && left >= (NS - 2) * 3) wait_vmcnt<(NS - 2) * 3>();
    else if (kMaxSlots >= 2 && left >= (NS - 2) * 2) wait_vmcnt<(NS - 2) * 2>();
    else if (left >= NS - 2) wait_vmcnt<NS - 2>();
    else wait_vmcnt<0>();
  };

  const int step = wid & 3, half = wid >> 2;
  // Operand addresses in stage 0: row n of a 16-row tile, logical slot 4 step + g.
  const uint32_t at = lds + uint32_t(n * kRowB + 16 * ((4 * step + g) ^ n));
  f32x4 acc[NF][NH];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < NH; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int c = 0; c < NS - 1; ++c)
    if (c < chunks) send(c, c);
  // Two operand sets: a chunk's operand reads run behind the previous chunk's
  // MFMAs.
  u32x4 w[2][NF], x[2][NH];
  const int jh = kTok ? 0 : half * NF, ih = kTok ? half * NH : 0;  // this half's first tiles
  int st = 0;
  // Chunk c from its stage into operand set r.
  auto fetch = [&](int c, int r) __attribute__((always_inline)) {
    landed(min(chunks - 1 - c, NS - 2));
    // Bare barrier: pieces of later chunks stay in flight. Past it, chunk c is
    // in LDS and every wave's reads of chunk c - 1 have returned.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + NS - 1 < chunks) send(c + NS - 1, st == 0 ? NS - 1 : st - 1);
    const uint32_t base = at + uint32_t(st) * L::stage;
#pragma unroll
    for (int j = 0; j < NF; ++j) w[r][j] = lds_read_b128_at(base + uint32_t(jh + j) * 16 * kRowB);
#pragma unroll
    for (int i = 0; i < NH; ++i)
      x[r][i] = lds_read_b128_at(base + uint32_t(NT + ih + i) * 16 * kRowB);
    st = st + 1 == NS ? 0 : st + 1;
  };
  auto multiply = [&](int r) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NH; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[j][i] = Mfma16<T>::run(w[r][j], x[r][i], acc[j][i]);
  };
  fetch(0, 0);  // chunks: a multiple of 4
  for (int c = 1; c < chunks - 1; c += 2) {
    fetch(c, 1);
    multiply(0);
    fetch(c + 1, 0);
    multiply(1);
  }
  fetch(chunks - 1, 1);
  multiply(0);
  multiply(1);
  __syncthreads();  // every read of the stages is done
  f32x4* const sums = reinterpret_cast<f32x4*>(smem);  // [step][tile j NM + token tile][lane]
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < NH; ++i)
      sums[((step * NT + jh + j) * NM + ih + i) * 64 + lane] = acc[j][i];
  __syncthreads();
  // A lane's vector: features 4 g .. 4 g + 3 of token n of the tile.
  for (int x = int(threadIdx.x); x < NT * NM * 64; x += 64 * kWaves) {
    const int j = x / (64 * NM), m = m0 + (x / 64 % NM) * 16 + n;  // x % 64 is this lane
    const int t = t0 + j;
    if (t >= tiles || m >= m0 + rows) continue;
    f32x4 v = sums[x];
#pragma unroll
    for (int w = 1; w < kSteps; ++w) v += sums[w * NT * NM * 64 + x];
    const int f = t * 16 + 4 * g;
    if (a.bias) {
      const u32x2 bb = *reinterpret_cast<const u32x2*>(a.bias + f);
      v[0] += to_f32(T{uint16_t(bb[0] & 0xffffu)});
      v[1] += to_f32(T{uint16_t(bb[0] >> 16)});
      v[2] += to_f32(T{uint16_t(bb[1] & 0xffffu)});
      v[3] += to_f32(T{uint16_t(bb[1] >> 16)});
    }
    *reinterpret_cast<u32x2*>(a.y + int64_t(m) * a.N + f) =
        u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
  }
}

// Opt a kernel into its dynamic LDS (past the default window), per device.
template <typename T, int NT, int NM>
hipError_t launch_nm(const LinearArgs& a, int blocks, hipStream_t st) {
  constexpr int lds = LinearLds<NT, NM>::bytes;
  const hipError_t e = opt_in_lds(
      reinterpret_cast<const void*>(&linear_chunk_kernel<T, NT, NM>), lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((linear_chunk_kernel<T, NT, NM>), dim3(unsigned(blocks)), dim3(64 * kWaves),
                     lds, st, a);
  return hipGetLastError();
}

template <typename T, int NT>
hipError_t launch_nt(const LinearArgs& a, int nm, int blocks, hipStream_t st) {
  if (nm == 2) return launch_nm<T, NT, 2>(a, blocks, st);
  if constexpr (NT % 2 == 0) {
    if (nm == 3) return launch_nm<T, NT, 3>(a, blocks, st);
  }
  return launch_nm<T, NT, 4>(a, blocks, st);
}

// Two token groups past 64 tokens; then the fewest feature tiles per workgroup
// (1, 2 or 4) that leave at most one workgroup per CU.
template <typename T>
hipError_t launch_t(LinearArgs a, hipStream_t st) {
  const int tiles = a.N / 16, cus = device_cus();
  a.groups = a.M > 64 ? 2 : 1;
  int nt = 1;
  while (nt < 4 && (tiles + nt - 1) / nt * a.groups > cus) nt *= 2;
  int nm = std::max(2, (a.M + 16 * a.groups - 1) / (16 * a.groups));
  if (nt == 1 && nm == 3) nm = 4;  // one of the two counts has to halve
  const int blocks = ((tiles + nt - 1) / nt + 7) / 8 * 8 * a.groups;
  switch (nt) {
    case 1: return launch_nt<T, 1>(a, nm, blocks, st);
    case 2: return launch_nt<T, 2>(a, nm, blocks, st);
    default: return launch_nt<T, 4>(a, nm, blocks, st);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace dx

using namespace dx;

extern "C" int dx_linear_chunk(const void* x, int64_t x_sb, int64_t x_sl, int io_dtype,
                               const void* w, int64_t w_row, const void* bias, void* y,
                               int64_t B, int64_t L, int64_t C, int64_t N, void* stream) {
  DX_CHECK_ARG(io_dtype == DX_BF16 || io_dtype == DX_F16,
               "linear_chunk: dtype must be bf16 or f16 (got code %d)", io_dtype);
  DX_CHECK_ARG(B >= 0 && L >= 0 && C > 0 && N > 0, "linear_chunk: bad shape");
  DX_CHECK_ARG(L <= 128 && B <= 128 && B * L <= 128,
               "linear_chunk: %lld x %lld tokens exceed 128", (long long)B, (long long)L);
  DX_CHECK_ARG(C % 512 == 0 && C <= (1 << 20),
               "linear_chunk: C = %lld must be a multiple of 512", (long long)C);
  DX_CHECK_ARG(N % 16 == 0 && N <= (1 << 20), "linear_chunk: N = %lld must be a multiple of 16",
               (long long)N);
  if (B * L == 0) return DX_OK;
  DX_CHECK_ARG(x && w && y, "linear_chunk: null pointer");
  DX_CHECK_ARG(aligned16(x) && aligned16(w) && aligned16(y) && (!bias || aligned16(bias)),
               "linear_chunk: pointers must be 16-byte aligned");
  DX_CHECK_ARG(x_sb >= 0 && x_sl >= 0 && x_sb % 8 == 0 && x_sl % 8 == 0 && w_row % 8 == 0 &&
                   w_row >= C && w_row < (int64_t(1) << 22),
               "linear_chunk: strides must be multiples of 8 elements (weight rows C .. 2^22)");
  // Rows are read through descriptors with 32-bit offsets.
  const int64_t x_bytes = 2 * ((B - 1) * x_sb + (L - 1) * x_sl + C);
  DX_CHECK_ARG(x_sb < (int64_t(1) << 31) && x_sl < (int64_t(1) << 31) &&
                   x_bytes < (int64_t(1) << 31),
               "linear_chunk: x spans %lld bytes (< 2^31)", (long long)x_bytes);
  LinearArgs a{};
  a.x = static_cast<const uint16_t*>(x); a.x_sb = x_sb; a.x_sl = x_sl;
  a.w = static_cast<const uint16_t*>(w); a.w_row = w_row;
  a.bias = static_cast<const uint16_t*>(bias);
  a.y = static_cast<uint16_t*>(y);
  a.M = int(B * L); a.L = int(L); a.C = int(C); a.N = int(N);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const hipError_t e = io_dtype == DX_BF16 ? launch_t<bf16_t>(a, st) : launch_t<f16_t>(a, st);
  if (e != hipSuccess) {
    set_error("linear_chunk: launch failed: %s", hipGetErrorString(e));
    return DX_ELAUNCH;
  }
  return DX_OK;
}
