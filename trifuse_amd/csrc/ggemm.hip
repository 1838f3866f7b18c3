// Prefill path: grouped GEMM over expert-contiguous routes.
//
// Two kernels: ggemm_wr_kernel (weights in registers; input widths a multiple
// of 128, described below at its definition) and ggemm_kernel, for odd
// multiples of 64, 8-bit codes with bf16 storage of many rows (lds_dequant) and
// scales or biases that start off a 4-byte boundary:
//
// Each workgroup computes a BM x BN tile of one expert's output with eight
// waves, two per SIMD, so that one wave's loads, dequantisation and LDS
// traffic overlap the other's MFMAs. Per K step of 64 (one quantisation
// group) it
//   * copies BM activation rows (x rows of the routed tokens, or rows of the
//     expert-sorted SwiGLU output) from global memory straight into LDS
//     (buffer loads with an LDS destination),
//   * loads BN packed weight rows (4-bit: 32 bytes, 8-bit: 64 bytes of each
//     row per step) into registers, dequantises them (s*q+b in fp32,
//     rounded to the storage dtype, bf16 or half) and writes them to LDS;
//     for inputs up to 2048 wide (and arrays on 16-byte boundaries) the scales
//     and biases of the tile's rows
//     are copied into LDS once per tile (coalesced) instead of being loaded
//     per step as 2-byte values from 64 rows at a time,
//   * runs v_mfma_f32_32x32x16_bf16 (or _f16) on the two LDS tiles, each wave owning a
//     WM x WN sub-tile (WM*WN/64 fp32 accumulators per lane); 32-row blocks
//     past the end of the expert's segment skip their fragment reads and MFMAs.
//
// Pipeline: two LDS stages for each operand. While the MFMAs of step k read
// stage k%2, the activations of step k+1 are copied into stage (k+1)%2, the
// packed weights of step k+1 (loaded during step k-1) are dequantised into
// stage (k+1)%2 and the packed weights of step k+2 are loaded; one barrier
// per step.
//
// LDS rows are 64 bf16 (8 chunks of 16 B); chunk c of row r is stored at
// c ^ ((r >> 1) & 7), so the 16 lanes of a ds_read_b128 pass (16 consecutive
// rows, one chunk) hit 16 distinct 16-byte bank groups.
//
// Rows outside the segment and weight rows past N get a buffer offset beyond
// the buffer and read as zero, so the loop has no divergent branches.
//
// Epilogue: each wave converts its accumulators (SwiGLU for gate/up) to bf16
// in a private LDS block, 32 rows at a time, and writes them out as 16-byte
// row chunks: h rows (gate/up), expert-output rows in sorted order (down) or
// rows scattered to their flat route (gather_qmm).
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "tfm_device.h"
#include "tfm_internal.h"

// Compiled once per storage dtype and code width, so that the instances build
// in parallel: as is for 4-bit codes with bf16 storage (which also holds the
// launch functions), and from ggemm_f16.hip, ggemm_i8.hip and
// ggemm_f16_i8.hip for the others.
#ifndef TFM_GG_F16
#define TFM_GG_F16 0
#endif
#ifndef TFM_GG_BITS
#define TFM_GG_BITS 4
#endif
#define TFM_GG_MAIN (TFM_GG_BITS == 4 && !TFM_GG_F16)

namespace tfm {

constexpr int BK = 64;
constexpr uint32_t kOob = 0x80000000u;  // buffer offset that reads as zero

enum GgemmMode { kGgGateUp = 0, kGgDown = 1, kGgPlain = 2 };

struct GgArgs {
  const uint16_t* x;     // activations (x rows, or sorted h rows for down)
  uint32_t x_bytes;      // size of x (buffer range)
  RowMap rm;
  Grouping g;
  tfm_affine wa, wb;     // gate/up (wb unused otherwise)
  int N;                 // output columns of one matrix
  int Kin;
  uint16_t* out;         // gate/up: h [n_routes, N]; down: y [n_routes, N]; plain: out [rows, N]
  int sb16;              // ggemm_wr_kernel: scale and bias rows start on 16-byte boundaries
};

// Row of accumulator element v of lane `lane` inside a 32x32 block of
// v_mfma_f32_32x32x16_bf16 (its column is lane % 32; operands: lane l
// supplies row/column l%32 and k = 8*(l/32) .. 8*(l/32)+7).
__device__ __forceinline__ int acc_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

__device__ __forceinline__ int swz(int row, int chunk) {
  return row * BK + ((chunk ^ ((row >> 1) & 7)) << 3);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gg_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// 4 bytes (one 32-bit word of an 8-bit weight row) -> 4 values s*q+b in the
// storage dtype (bf16, or half when F16).
template <bool F16>
__device__ __forceinline__ uint2 dequant_word_u8(uint32_t w, float s, float b) {
  float d[4];
  dequant4_u8(w, s, b, d);
  uint2 pk;
  pk.x = pack_st2<F16>(d[0], d[1]);
  pk.y = pack_st2<F16>(d[2], d[3]);
  return pk;
}

// 8 nibbles (one 32-bit word of a 4-bit weight row) -> 8 values s*q+b.
template <bool F16>
__device__ __forceinline__ uint4 dequant_word(uint32_t w, float s, float b) {
  float d[8];
  dequant8(w, s, b, d);
  uint4 pk;
  pk.x = pack_st2<F16>(d[0], d[1]);
  pk.y = pack_st2<F16>(d[2], d[3]);
  pk.z = pack_st2<F16>(d[4], d[5]);
  pk.w = pack_st2<F16>(d[6], d[7]);
  return pk;
}

// One 32x32x16 MFMA on bf16 or half operands (fp32 accumulators).
template <bool F16>
using op8_t = std::conditional_t<F16, f16x8_t, bf16x8_t>;
template <bool F16>
__device__ __forceinline__ f32x16_t mfma32(op8_t<F16> a, op8_t<F16> b, f32x16_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// silu(g) * u with the hardware exp and reciprocal (relative error ~1e-7,
// far below the bf16 rounding that follows).
__device__ __forceinline__ float swiglu(float g, float u) {
  const float e = __builtin_amdgcn_exp2f(-g * 1.44269504f);
  return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
}

// 16 bytes per lane from a buffer into LDS: lane l writes dst + 16*l (dst is
// wave-uniform). Out-of-range offsets deliver zeros.
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t r, uint16_t* dst, uint32_t voff, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
#else
  (void)r; (void)dst; (void)voff; (void)soff;
#endif
}

// The same with 4 bytes per lane: lane l's dword lands at dst + 4 l bytes.
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t r, uint16_t* dst, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, voff, 0, 0, 0);
#else
  (void)r; (void)dst; (void)voff;
#endif
}

// Calls f(std::integral_constant<int, I>) for I = B .. E-1 (compile-time
// iteration: every index into register arrays is a constant).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int MODE, int BITS_>
struct GgCfg {
  static constexpr int BM = BM_, BN = BN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, BITS = BITS_;
  static constexpr int CPR_B = BITS / 2;            // 16-byte packed chunks of a weight row per step
  static constexpr int WAVES = WAVES_M * WAVES_N;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int MB = WM / 32;                // 32-row MFMA blocks per wave
  static constexpr int NB = WN / 32;                // 32-column MFMA blocks per wave
  static constexpr int LA = BM / (8 * WAVES);       // 8-row LDS copies per wave per step
  static constexpr int LB = BN * CPR_B / THREADS;   // packed 16-byte chunks per thread per step
  static constexpr int OUT_COLS = MODE == kGgGateUp ? BN / 2 : BN;
  static constexpr int WCOLS = MODE == kGgGateUp ? WN / 2 : WN;   // output columns per wave
  static constexpr int SROW = WCOLS + 8;            // staging row stride (bf16), 16 B pad
  static_assert(LA >= 1 && LA * 8 * WAVES == BM, "A copies must tile the block rows");
  static_assert(BITS == 4 || BITS == 8, "4-bit or 8-bit weights");
  static_assert(LB >= 1 && LB * THREADS == BN * CPR_B, "B chunks must tile the block columns");
  static_assert(64 % CPR_B == 0 && (64 / CPR_B) <= BN / 2, "a wave's chunks stay in one half of the tile");
  static_assert(LB * 4 >= 3, "B words are spread over three sub-steps");
  static_assert(MODE != kGgGateUp || NB % 2 == 0, "gate/up wave tiles pair gate and up blocks");
  static_assert(WAVES % 4 == 0, "staging blocks are spread over the four LDS stages");
  static_assert(32 * SROW * (WAVES / 4) <= BM * BK, "epilogue staging must fit in an A stage");
};

// Packed weights of one K step for one thread.
template <int LB>
struct RawB {
  uint4 b[LB];
  uint32_t s[LB], bias[LB];
};

// Largest input width whose scales and biases a tile keeps in LDS (32 groups
// per weight row); wider inputs load them per step with the packed codes.
constexpr int kLdsScaleKin = 32 * BK;

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int MODE, int BITS, bool F16, bool SL>
__global__ __launch_bounds__(WAVES_M_ * WAVES_N_ * 64, 1) void ggemm_kernel(GgArgs args) {
  using C = GgCfg<BM_, BN_, WAVES_M_, WAVES_N_, MODE, BITS>;
  constexpr int CPR_B = C::CPR_B;
  constexpr int BM = C::BM, BN = C::BN, MB = C::MB, NB = C::NB, LA = C::LA, LB = C::LB;
  constexpr int T = C::THREADS;
  // Two stages each of A and B, as separate objects so that the compiler's
  // wait tracking tells LDS copies into one stage from reads of the other.
  __shared__ __attribute__((aligned(16))) uint16_t sA0[BM * BK];
  __shared__ __attribute__((aligned(16))) uint16_t sA1[BM * BK];
  __shared__ __attribute__((aligned(16))) uint16_t sB0[BN * BK];
  __shared__ __attribute__((aligned(16))) uint16_t sB1[BN * BK];
  // SL: scales and biases of the tile's weight rows for the whole input
  // width (up to 32 groups per row), copied once per tile.
  __shared__ __attribute__((aligned(16))) uint16_t sSc[SL ? BN * 32 : 8];
  __shared__ __attribute__((aligned(16))) uint16_t sBi[SL ? BN * 32 : 8];
  // The tile prefix and the expert index live in weight stage 1, which is
  // first written after the prologue's barrier.
  int* const s_tiles = reinterpret_cast<int*>(sB1);
  int& s_expert = s_tiles[65];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int E = args.g.E;

  // M-tile prefix over experts.
  if (tid < 64) {
    int t = 0;
    if (tid < E) {
      const int cnt = grp_offset(args.g, tid + 1) - grp_offset(args.g, tid);
      t = (cnt + BM - 1) / BM;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(t, d, 64);
      if (lane >= d) t += o;
    }
    s_tiles[tid + 1] = t;
    if (tid == 0) s_tiles[0] = 0;
  }
  __syncthreads();
  const int NT = (args.N + C::OUT_COLS - 1) / C::OUT_COLS;
  const int mtiles = s_tiles[E];
  const int64_t total = (int64_t)mtiles * NT;
  // XCD-aware remap: workgroups are dispatched round-robin over 8 XCDs, so
  // XCD x gets a contiguous range of tiles (m-tile major) for L2 reuse.
  const int xcd = blockIdx.x & 7;
  const int64_t local = blockIdx.x >> 3;
  const int64_t share = (total + 7) / 8;
  const int64_t ti = xcd * share + local;
  if (local >= share || ti >= total) return;
  const int mt = (int)(ti / NT), nt = (int)(ti % NT);
  if (tid < E && s_tiles[tid] <= mt && mt < s_tiles[tid + 1]) s_expert = tid;
  __syncthreads();
  const int e = s_expert;
  const int seg0 = grp_offset(args.g, e), seg1 = grp_offset(args.g, e + 1);
  const int m0 = seg0 + (mt - s_tiles[e]) * BM;
  const int rows_valid = min(BM, seg1 - m0);
  const int n0 = nt * C::OUT_COLS;
  const int KT = args.Kin / BK;

  // ---- A: global -> LDS copies ----
  // Wave w fills rows [w*BM/W, (w+1)*BM/W), 8 rows (1 KB) per instruction:
  // lane l of copy i writes LDS slot l%8 of row w*BM/W + i*8 + l/8, which
  // under the swizzle holds chunk (l%8) ^ ((row >> 1) & 7).
  const __amdgpu_buffer_rsrc_t ra = gg_rsrc(args.x, args.x_bytes);
  const __amdgpu_buffer_rsrc_t rnull = gg_rsrc(args.x, 0);
  uint32_t a_off[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = wave * (BM / C::WAVES) + i * 8 + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    if (r < rows_valid) {
      const int64_t src = MODE == kGgDown ? (int64_t)(m0 + r) : route_row(args.rm, m0 + r);
      a_off[i] = (uint32_t)((src * args.Kin + c * 8) * 2);
    } else {
      a_off[i] = kOob;
    }
  }
  // Step kt of A into LDS stage `dst`; steps past the last read zeros.
  auto a_copy = [&](uint16_t* dst, int kt) {
    const __amdgpu_buffer_rsrc_t r = kt < KT ? ra : rnull;
#pragma unroll
    for (int i = 0; i < LA; ++i) lds_dma16(r, dst + (wave * (BM / C::WAVES) + i * 8) * BK, a_off[i], kt * BK * 2);
  };

  // ---- B: packed weights ----
  // Chunk q = i*T + tid -> weight row q/CPR_B, part q%CPR_B (16 bytes: 32
  // nibbles or 16 bytes of codes). Gate/up tiles hold BN/2 gate rows then
  // BN/2 up rows.
  const uint32_t qrow = (uint32_t)args.Kin * BITS / 8, srow = (uint32_t)(args.Kin / BK) * 2;
  __amdgpu_buffer_rsrc_t rbq[LB], rbs[LB], rbb[LB];
  uint32_t b_qoff[LB], b_soff[LB];
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int qw = i * T + wave * 64;  // first chunk of this wave (uniform)
    const bool up = MODE == kGgGateUp && qw / CPR_B >= BN / 2;
    const tfm_affine& bm = up ? args.wb : args.wa;
    const int q = qw + lane;
    const int r = q / CPR_B;
    const int bn = MODE == kGgGateUp ? n0 + (r & (BN / 2 - 1)) : n0 + r;
    const size_t ebase = (size_t)e * args.N;
    rbq[i] = gg_rsrc(reinterpret_cast<const char*>(bm.q) + ebase * qrow, (uint32_t)args.N * qrow);
    rbs[i] = gg_rsrc(static_cast<const char*>(bm.scales) + ebase * srow, (uint32_t)args.N * srow);
    rbb[i] = gg_rsrc(static_cast<const char*>(bm.biases) + ebase * srow, (uint32_t)args.N * srow);
    const bool ok = bn < args.N;
    b_qoff[i] = ok ? (uint32_t)bn * qrow + (q % CPR_B) * 16 : kOob;
    b_soff[i] = ok ? (uint32_t)bn * srow : kOob;
  }

  // SL: the tile's weight rows fall into HALVES contiguous row ranges of the
  // scale and bias matrices (gate/up: BN/2 gate rows, then BN/2 up rows;
  // otherwise BN rows of one matrix). Each range is copied into LDS in 1 KB
  // pieces at a 1 KB-aligned offset (HS bytes apart), so the zeros or
  // neighbouring rows that a partial last piece brings in land in padding.
  // Rows past N read as zero. Per K step a thread then reads its row's scale
  // and bias from LDS instead of two 2-byte loads from 64 different rows.
  constexpr int HALVES = MODE == kGgGateUp ? 2 : 1;
  constexpr int HROWS = BN / HALVES;
  const int G = args.Kin / BK;
  const int hbytes = HROWS * G * 2;
  const int hs = (hbytes + 1023) & ~1023;
  int sidx[LB];
  if constexpr (SL) {
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const tfm_affine& bm = h ? args.wb : args.wa;
      const size_t ebase = (size_t)e * args.N;
      const auto rs = gg_rsrc(static_cast<const char*>(bm.scales) + ebase * srow, (uint32_t)args.N * srow);
      const auto rb = gg_rsrc(static_cast<const char*>(bm.biases) + ebase * srow, (uint32_t)args.N * srow);
      const uint32_t g0 = (uint32_t)n0 * srow;
      for (int c = wave; c * 1024 < hbytes; c += C::WAVES) {
        lds_dma16(rs, sSc + (h * hs + c * 1024) / 2, g0 + c * 1024 + lane * 16, 0);
        lds_dma16(rb, sBi + (h * hs + c * 1024) / 2, g0 + c * 1024 + lane * 16, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int r = (i * T + tid) / CPR_B;
      sidx[i] = (r / HROWS) * (hs / 2) + (r % HROWS) * G;
    }
  }
  // Packed codes of step kt (and, without SL, its scale and bias).
  auto bload_q = [&](RawB<LB>& st, int kt) {
    const bool live = kt < KT;
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      st.b[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(live ? rbq[i] : rnull, b_qoff[i], kt * (BK * BITS / 8), 0));
      if constexpr (!SL) {
        st.s[i] = __builtin_amdgcn_raw_buffer_load_b16(live ? rbs[i] : rnull, b_soff[i], kt * 2, 0);
        st.bias[i] = __builtin_amdgcn_raw_buffer_load_b16(live ? rbb[i] : rnull, b_soff[i], kt * 2, 0);
      }
    }
  };
  // SL: scale and bias of step kt from LDS (steps past the end reuse the
  // last group; their codes and activations are zero).
  auto bload_sb = [&](RawB<LB>& st, int kt) {
    if constexpr (SL) {
      const int g = kt < KT ? kt : KT - 1;
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        st.s[i] = sSc[sidx[i] + g];
        st.bias[i] = sBi[sidx[i] + g];
      }
    }
  };
  auto bload = [&](RawB<LB>& st, int kt) {
    bload_q(st, kt);
    bload_sb(st, kt);
  };
  // Word w (of LB*4) of the dequantised B step: 8 elements (one LDS chunk)
  // for 4-bit, 4 elements (half a chunk) for 8-bit.
  auto bstore_word = [&](const RawB<LB>& st, uint16_t* dst, int w) {
    const int i = w / 4, k = w % 4;
    const int q = i * T + tid;
    const float sc = st2f<F16>((uint16_t)st.s[i]), bi = st2f<F16>((uint16_t)st.bias[i]);
    if constexpr (BITS == 4) {
      const uint4 pk = dequant_word<F16>(word_of(st.b[i], k), sc, bi);
      *reinterpret_cast<uint4*>(&dst[swz(q >> 1, (q & 1) * 4 + k)]) = pk;
    } else {
      const uint2 pk = dequant_word_u8<F16>(word_of(st.b[i], k), sc, bi);
      *reinterpret_cast<uint2*>(&dst[swz(q >> 2, (q & 3) * 2 + (k >> 1)) + (k & 1) * 4]) = pk;
    }
  };

  // ---- wave tile ----
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  int brow[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (MODE == kGgGateUp)
      brow[j] = j < NB / 2 ? wn * (C::WN / 2) + j * 32 : BN / 2 + wn * (C::WN / 2) + (j - NB / 2) * 32;
    else
      brow[j] = wn * C::WN + j * 32;
  }

  f32x16_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // MFMAs of one LDS stage (fragments of K sub-step ks+1 are read during the
  // MFMAs of ks); the dequantised next B step is written during sub-steps
  // 1..3, so its loads have had more than a step to arrive.
  // MBL = the wave's 32-row blocks that hold rows of the segment (0..MB): the
  // wave reads A fragments and runs MFMAs for those blocks only. With MBL = 0
  // (every row of the wave past the segment) it skips fragment reads and
  // MFMAs altogether, which frees its SIMD's matrix pipe for the other wave
  // there, and only does its share of the loads and LDS writes.
  auto compute = [&](auto mbl_tag, const uint16_t* A, const uint16_t* Bs, const RawB<LB>& nxt,
                     uint16_t* nB) {
    constexpr int MBL = decltype(mbl_tag)::value;
    op8_t<F16> af[2][MB], bfr[2][NB];
    auto frag = [&](int ks, int slot) {
      const int kc = ks * 2 + (lane >> 5);
#pragma unroll
      for (int i = 0; i < MBL; ++i)
        af[slot][i] = *reinterpret_cast<const op8_t<F16>*>(&A[swz(wm * C::WM + i * 32 + (lane & 31), kc)]);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        bfr[slot][j] = *reinterpret_cast<const op8_t<F16>*>(&Bs[swz(brow[j] + (lane & 31), kc)]);
    };
    if constexpr (MBL > 0) frag(0, 0);
    static_for<0, 4>([&](auto kc_) {
      constexpr int ks = decltype(kc_)::value;
      if constexpr (MBL > 0) {
        if constexpr (ks < 3) frag(ks + 1, (ks + 1) & 1);
#pragma unroll
        for (int i = 0; i < MBL; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[i][j] = mfma32<F16>(af[ks & 1][i], bfr[ks & 1][j], acc[i][j]);
      }
      if constexpr (ks >= 1) {
#pragma unroll
        for (int w = (ks - 1) * LB * 4 / 3; w < ks * LB * 4 / 3; ++w) bstore_word(nxt, nB, w);
      }
    });
  };
  // End of a step: the barrier's release fence waits for this wave's LDS
  // writes (copies and dequantised B) and its outstanding weight loads; after
  // it every wave's writes are visible.
  auto step_end = [&]() { __syncthreads(); };

  // With an odd step count the loop runs one more step on zeros (A and B
  // both read from null buffers), which adds nothing.
  RawB<LB> st0, st1;
  a_copy(sA0, 0);
  bload_q(st0, 0);
  bload_q(st1, 1);
  // SL: every wave's scale copies are complete and visible after this barrier
  if constexpr (SL) __syncthreads();
  bload_sb(st0, 0);
  bload_sb(st1, 1);
#pragma unroll
  for (int w = 0; w < LB * 4; ++w) bstore_word(st0, sB0, w);
  step_end();
  auto main_loop = [&](auto mbl_tag) {
    for (int kt = 0; kt < KT; kt += 2) {
      a_copy(sA1, kt + 1);
      bload(st0, kt + 2);
      __builtin_amdgcn_sched_barrier(0);
      compute(mbl_tag, sA0, sB0, st1, sB1);
      step_end();
      a_copy(sA0, kt + 2);
      bload(st1, kt + 3);
      __builtin_amdgcn_sched_barrier(0);
      compute(mbl_tag, sA1, sB1, st0, sB0);
      step_end();
    }
  };
  // Live row blocks of this wave (wave-uniform), one compiled loop per count.
  static_assert(MB == 2 || MB == 4, "row blocks per wave");
  const int live_rows = rows_valid - wm * C::WM;
  const int mbl = live_rows <= 0 ? 0 : min(MB, (live_rows + 31) / 32);
  if (mbl == MB) {
    main_loop(std::integral_constant<int, MB>{});
  } else if constexpr (MB == 4) {
    if (mbl == 3)
      main_loop(std::integral_constant<int, 3>{});
    else if (mbl == 2)
      main_loop(std::integral_constant<int, 2>{});
    else if (mbl == 1)
      main_loop(std::integral_constant<int, 1>{});
    else
      main_loop(std::integral_constant<int, 0>{});
  } else {
    if (mbl == 1)
      main_loop(std::integral_constant<int, 1>{});
    else
      main_loop(std::integral_constant<int, 0>{});
  }

  // ---- epilogue ----
  // Private staging block of this wave: 32 rows x SROW bf16 inside one of the
  // four stages (every wave is past the last barrier, so LDS is free).
  uint16_t* stage = (wave & 3) == 0 ? sA0 : (wave & 3) == 1 ? sA1 : (wave & 3) == 2 ? sB0 : sB1;
  stage += (wave >> 2) * 32 * C::SROW;
  constexpr int CPR = C::WCOLS / 8;             // 16-byte chunks per staged row
  const int col_base = MODE == kGgGateUp ? n0 + wn * (C::WN / 2) : n0 + wn * C::WN;
  // Row blocks by compile-time index (a runtime loop with an early exit can
  // leave acc dynamically indexed, and then in scratch memory).
  static_for<0, MB>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const int r0 = wm * C::WM + i * 32;         // first tile row of this block
    if (r0 >= rows_valid) return;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int rr = acc_row(v, lane);
      if (MODE == kGgGateUp) {
#pragma unroll
        for (int jb = 0; jb < NB / 2; ++jb)
          stage[rr * C::SROW + jb * 32 + (lane & 31)] = f2st<F16>(swiglu(acc[i][jb][v], acc[i][jb + NB / 2][v]));
      } else {
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) stage[rr * C::SROW + jb * 32 + (lane & 31)] = f2st<F16>(acc[i][jb][v]);
      }
    }
    // Same-wave LDS accesses complete in order: the reads see the writes.
#pragma unroll
    for (int c0 = 0; c0 < 32 * CPR; c0 += 64) {
      const int c = c0 + lane;
      const int row = c / CPR, part = c % CPR;
      const int rr = r0 + row;
      const int n = col_base + part * 8;
      if (c < 32 * CPR && rr < rows_valid && n < args.N) {
        const uint4 v = *reinterpret_cast<const uint4*>(&stage[row * C::SROW + part * 8]);
        const int j = m0 + rr;
        const int64_t orow = MODE == kGgPlain ? (int64_t)route_flat(args.rm, j) : (int64_t)j;
        *reinterpret_cast<uint4*>(&args.out[orow * args.N + n]) = v;
      }
    }
  });
}

// ---------------------------------------------------------------------------
// 4- and 8-bit weights with inputs a multiple of 128 wide: the weights stay
// in registers.
//
// Tile: BM routed rows x 16 NJ WV weight rows, WV (4 or 8) waves. Wave w owns
// 16 NJ (32 or 64) weight rows for all BM rows (gate/up: gate rows 8 NJ w ..
// + 8 NJ - 1 and the same up rows; down and plain: rows 16 NJ w .. + 16 NJ - 1),
// as 16 x 16 blocks of v_mfma_f32_16x16x32_bf16 (or _f16): BM/16 row blocks x
// NJ column blocks, 4 fp32 accumulators each per lane. A gate block and its
// up block sit in the same lanes, so SwiGLU needs no exchange.
//
// Per super-step of 128 k (two quantisation groups):
//   * the BM activation rows are copied into LDS (one of two stages);
//   * lane l loads the 32 contiguous codes (16 or 32 bytes) k = 32 (l / 16)
//     .. + 31 of the super-step of each of its NJ weight rows; they share one
//     scale group. Codes 8 s .. 8 s + 7 of them are dequantised into the B
//     operand of sub-step s. The reduction order inside an MFMA is free, so
//     the A operand of sub-step s for lane l is the same k range: LDS chunk
//     4 (l / 16) + s of the row;
//   * one barrier, for the next stage's activations.
// Every packed weight is dequantised exactly once per tile and never goes
// through LDS. Per 128 k a wave runs 4 NJ x BM/16 MFMAs for one barrier: twice
// the work per barrier of the kernel above at the same tile.
//
// LDS: activation row r of a stage is 256 B (16 chunks of 16 B); chunk c is
// stored in slot c ^ (r & 15), so the 16 lanes of one read pass (16
// consecutive rows, one chunk) hit distinct bank groups. The scales and
// biases of the tile's rows are kept for four super-steps at a time (eight
// groups, 16 bytes a row) in a ring of two (few-row tiles of eight waves: four).
constexpr int BK2 = 128;

__device__ __forceinline__ f32x4_t mfma16(bf16x8_t a, bf16x8_t b, f32x4_t c, std::false_type) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma16(f16x8_t a, f16x8_t b, f32x4_t c, std::true_type) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Dequantisation of 8 codes (one lane's share of a sub-step) into four packed
// pairs, cut into eight slices 0..7 that the main loop spreads over its MFMAs.
// Scale and bias as loaded once per super-step: floats for bf16, (s, s) pairs
// for half.
//
// 4-bit: a byte 0..15 read as fp8 (e4m3, subnormal below 8) is code / 512, so
// one v_cvt_scalef32_pk with scale 512 turns two codes into two exact floats
// (v_cvt_f32_ubyte turns one, at the same cost: 5 cycles per wave
// instruction). bf16 then takes fp32 fused multiply-adds and one rounding.
// Half multiplies and adds in half: v_pk_fma_f16 rounds the exact s q + b once
// (codes and 11-bit scales are exact in half), where fp32 followed by a
// conversion rounds twice.
// 8-bit: bf16 converts byte by byte; half takes 1024 + q (the byte under an
// exponent byte) minus 1024, both exact, then the same fused multiply-add.
template <int BITS, bool F16>
struct Deq8 {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  using sb_t = std::conditional_t<F16, f16x2, float>;
  static constexpr int WORDS = BITS / 4;          // packed words of 8 codes

  uint32_t lo, hi;
  f32x2 pl, ph;
  f16x2 p16;
  float f;

  static __device__ __forceinline__ sb_t sb(uint16_t h) {
    if constexpr (F16) {
      const _Float16 v = __builtin_bit_cast(_Float16, h);
      return f16x2{v, v};
    } else {
      return bf2f(h);
    }
  }

  // out: the four packed pairs; w: the WORDS packed words.
  template <int EL>
  __device__ __forceinline__ void slice(const uint32_t* w, sb_t s, sb_t b, uint32_t* out) {
    constexpr int half = EL / 4, e4 = EL % 4;
    if constexpr (BITS == 4 && !F16) {
      if constexpr (EL == 0) {
        lo = w[0] & 0x0f0f0f0fu;                  // codes 0 2 4 6
        hi = (w[0] >> 4) & 0x0f0f0f0fu;           // codes 1 3 5 7
      }
      if constexpr (e4 == 0) pl = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo, 512.0f, half == 1);
      if constexpr (e4 == 1) ph = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi, 512.0f, half == 1);
      if constexpr (e4 == 2)
        out[2 * half] = pack_bf16x2(__builtin_fmaf(s, pl[0], b), __builtin_fmaf(s, ph[0], b));
      if constexpr (e4 == 3)
        out[2 * half + 1] = pack_bf16x2(__builtin_fmaf(s, pl[1], b), __builtin_fmaf(s, ph[1], b));
    } else if constexpr (BITS == 4) {
      if constexpr (EL == 0) {
        lo = w[0] & 0x0f0f0f0fu;
        hi = (w[0] >> 4) & 0x0f0f0f0fu;
      }
      if constexpr (EL == 1) {
        const uint32_t l = lo;
        lo = __builtin_amdgcn_perm(hi, l, 0x05010400u);  // codes 0 1 2 3
        hi = __builtin_amdgcn_perm(hi, l, 0x07030602u);  // codes 4 5 6 7
      }
      if constexpr (e4 >= 2) {
        const f16x2 q = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(half ? hi : lo, 512.0f, e4 == 3);
        out[EL - 2 - 2 * half] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(s, q, b));
      }
    } else if constexpr (!F16) {
      const float v = __builtin_fmaf(s, (float)((w[half] >> (8 * e4)) & 0xffu), b);
      if constexpr (EL % 2 == 0) f = v;
      else out[EL / 2] = pack_bf16x2(f, v);
    } else {
      constexpr int pair = EL / 2;
      if constexpr (EL % 2 == 0)
        p16 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, w[half], pair % 2 ? 0x04030402u : 0x04010400u)) -
              f16x2{(_Float16)1024.0f, (_Float16)1024.0f};
      else
        out[pair] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(s, p16, b));
    }
  }
};

// Tile of BM = 64, 96, 128 or 256 rows by BN = 16 NJ WV weight rows. Where the
// LDS and registers allow it, two or more workgroups share a compute unit, and
// one covers the other's load latency, barriers and epilogue: 64 x 8 waves two
// (48 KB, 64 with few rows, 128 registers), 64 x 4 four (40 KB), 96 x 4 (NJ = 4) and 128 x 4 two
// (64 and 72 KB, 256 registers), 128 x 8 and 256 x 8 one. WV = 4 with NJ = 2
// halves the weight rows of a tile (128: 64 gate and 64 up rows, or 128 down
// rows) for twice the tiles, where 8-wave tiles would leave compute units idle
// (a few experts or a few output columns: Granite decode batches, a dense
// matrix).
template <int BM>
constexpr int wr_waves_per_simd() { return BM == 64 ? 4 : 2; }

template <int BM, int MODE, int BITS, bool F16, int WV, bool FEW = false, int NJ = 2>
__global__ __launch_bounds__(WV * 64, (wr_waves_per_simd<BM>())) void ggemm_wr_kernel(GgArgs args) {
  constexpr int WAVES = WV, WN = 16 * NJ, BN = WN * WV;
  constexpr int NB = MODE == kGgGateUp ? NJ / 2 : NJ;  // column blocks of one matrix per wave
  constexpr int MB = BM / 16;                     // 16-row blocks per wave
  constexpr int OUT_COLS = MODE == kGgGateUp ? BN / 2 : BN;
  constexpr int LA = BM / (4 * WAVES);            // 4-row (1 KB) copies per wave per super-step
  static_assert(WV == 8 || (WV == 4 && BM <= 128), "8 waves, or 4 with tiles of up to 128 rows");
  static_assert(NJ == 2 || (NJ == 4 && WV == 4), "32 weight rows a wave, or 64 with 4 waves");
  static_assert(LA >= 1, "every wave copies activation rows");
  constexpr int SROW = 136;                       // epilogue staging row stride (128 columns + 16 B)
  constexpr int HALF_ROWS = BM / 2;               // staged rows per activation stage
  static_assert(BM == 64 || BM == 96 || BM == 128 || BM == 256, "tile rows");
  static_assert(HALF_ROWS * SROW <= BM * BK2, "epilogue staging fits a stage");
  // 128 rows of 64 weight rows a wave leave no registers for both super-steps'
  // raw weights: the next one's are requested halfway through sub-step 1, when
  // half of this one's are used up, and A fragments are read two pairs ahead.
  constexpr bool LATE = BM == 128 && NJ == 4;
  // A fragments read ahead of the MFMAs that use them, in row blocks. Two where
  // a third does not fit: 8-bit half down and plain tiles of 64 rows spilled 2 to
  // 12 of their 128 registers with three, and a reload from scratch memory waits
  // for every load in flight.
  constexpr int AHEAD = LATE || (BM == 64 && BITS == 8 && F16 && MODE != kGgGateUp) ? 2 : 3;
  using op_t = op8_t<F16>;
  using f16tag = std::integral_constant<bool, F16>;
  using D8 = Deq8<BITS, F16>;
  using sb_t = typename D8::sb_t;
  constexpr int RL = BITS / 4;                    // 16-byte raw loads per weight row and super-step
  constexpr int SBH = BN * 8;                     // scales (or biases) of the tile's rows, 8 groups

  __shared__ __attribute__((aligned(16))) uint16_t sA0[BM * BK2];
  __shared__ __attribute__((aligned(16))) uint16_t sA1[BM * BK2];
  // Scale and bias chunks kept: a ring of two, or with few rows and eight waves
  // (whose registers hold a compute unit to two workgroups, so the LDS has room)
  // four, the whole of a 2048-wide input, copied before the loop. In the few-row
  // loop nothing covers the memory latency of a copy: OLMoE 44 tokens 75.2 us a
  // layer with the ring of two, 72.1 with all four ahead.
  constexpr int SLOTS = FEW && WV == 8 ? 4 : 2;
  __shared__ __attribute__((aligned(16))) uint16_t sSb[SLOTS * 2 * SBH];  // [slot][scale, bias][row][8 groups]
  // Tile prefix, XCD bounds and expert index: in activation stage 1, first
  // written after the prologue's barrier.
  int* const s_tiles = reinterpret_cast<int*>(sA1);
  int* const s_bound = s_tiles + 66;
  int& s_expert = s_tiles[65];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int E = args.g.E;
  const int NT = (args.N + OUT_COLS - 1) / OUT_COLS;
  const int xcd = blockIdx.x & 7;
  const int local = blockIdx.x >> 3;

  // Tiles in m-major order (experts in order, their m-tiles, n-tiles
  // innermost). Workgroups are dispatched round-robin over the 8 XCDs; XCD
  // x takes a contiguous run of the order (its n-tiles and neighbouring
  // m-tiles share activations and weights in its L2) holding about 1/8 of
  // the estimated work. With 256-row tiles a tile costs about 13 + (live
  // 16-row blocks) units (measured: 23.6 + 1.85 x blocks microseconds at
  // 4096 tokens), so runs of short tiles are longer; 128-row tiles cost
  // about the same whatever their rows, and count one unit each.
  constexpr bool BAL = BM == 256;
  constexpr int CF = BAL ? 13 + MB : 1;
  if (tid < 64) {
    int cnt = 0;
    if (tid < E) cnt = grp_offset(args.g, tid + 1) - grp_offset(args.g, tid);
    const int full = cnt / BM, part = cnt % BM;
    const int cp = part > 0 ? (BAL ? 13 + min(MB, ((part + 63) / 64) * 4) : 1) : 0;
    const int mt_e = full + (part > 0 ? 1 : 0);
    const int cost_e = NT * (full * CF + cp);
    int mt_i = mt_e, cost_i = cost_e;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o1 = __shfl_up(mt_i, d, 64), o2 = __shfl_up(cost_i, d, 64);
      if (lane >= d) {
        mt_i += o1;
        cost_i += o2;
      }
    }
    s_tiles[tid + 1] = mt_i;
    if (tid == 0) s_tiles[0] = 0;
    const int W = __shfl(cost_i, 63, 64);
    // bound k: tiles whose start lies below target (xcd + k) W / 8
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int T = (int)(((int64_t)(xcd + k) * W) / 8);
      if (tid == 0) s_bound[k] = 0;
      const int pc = cost_i - cost_e;
      if (tid < E && pc < T && T <= cost_i) {
        const int rel = T - pc, fc = full * NT * CF;
        const int c = rel <= fc ? (rel + CF - 1) / CF : full * NT + (rel - fc + cp - 1) / cp;
        s_bound[k] = (mt_i - mt_e) * NT + c;
      }
    }
  }
  __syncthreads();
  const int ti = s_bound[0] + local;
  if (ti >= s_bound[1]) return;
  const int mt = ti / NT, nt = ti % NT;
  if (tid < E && s_tiles[tid] <= mt && mt < s_tiles[tid + 1]) s_expert = tid;
  __syncthreads();
  const int e = s_expert;
  const int seg0 = grp_offset(args.g, e), seg1 = grp_offset(args.g, e + 1);
  const int m0 = seg0 + (mt - s_tiles[e]) * BM;
  const int rows_valid = min(BM, seg1 - m0);
  const int n0 = nt * OUT_COLS;
  const int KT = args.Kin / BK2;
  const int G = args.Kin / BK;                    // quantisation groups per row

  // ---- activations: global -> LDS ----
  // Copy i of wave w: rows 4 (WAVES i + w) .. + 3 (copy i of all waves
  // together: rows 4 WAVES i .. + 4 WAVES - 1); lane l writes slot l % 16 of
  // row 4 (WAVES i + w) + l / 16, which holds chunk (l % 16) ^ (row & 15).
  const __amdgpu_buffer_rsrc_t ra = gg_rsrc(args.x, args.x_bytes);
  const __amdgpu_buffer_rsrc_t rnull = gg_rsrc(args.x, 0);
  uint32_t a_off[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = 4 * (WAVES * i + wave) + (lane >> 4);
    const int c = (lane & 15) ^ (r & 15);
    if (r < rows_valid) {
      const int64_t src = MODE == kGgDown ? (int64_t)(m0 + r) : route_row(args.rm, m0 + r);
      a_off[i] = (uint32_t)((src * args.Kin + c * 8) * 2);
    } else {
      a_off[i] = kOob;
    }
  }
  auto a_copy = [&](uint16_t* dst, int kt) {
    const __amdgpu_buffer_rsrc_t r = kt < KT ? ra : rnull;
#pragma unroll
    for (int i = 0; i < LA; ++i) lds_dma16(r, dst + 4 * (WAVES * i + wave) * BK2, a_off[i], kt * BK2 * 2);
  };
  // Copy i alone (the main loop spreads the copies over a super-step).
  auto a_copy1 = [&](uint16_t* dst, int kt, auto i_) {
    constexpr int i = decltype(i_)::value;
    const __amdgpu_buffer_rsrc_t r = kt < KT ? ra : rnull;
    lds_dma16(r, dst + 4 * (WAVES * i + wave) * BK2, a_off[i], kt * BK2 * 2);
  };

  // ---- weights ----
  const int g4 = lane >> 4;                       // k quarter of the super-step
  const uint32_t qrow = (uint32_t)args.Kin * BITS / 8, srow = (uint32_t)G * 2;
  __amdgpu_buffer_rsrc_t rbq[NJ];
  uint32_t b_qoff[NJ];
  int trow[NJ];                                   // weight row within the tile (0..255)
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const tfm_affine& bm = (MODE == kGgGateUp && j >= NB) ? args.wb : args.wa;
    const int col = 16 * (NB * wave + j % NB) + (lane & 15);
    trow[j] = MODE == kGgGateUp ? (j / NB) * (BN / 2) + col : col;
    const int bn = n0 + col;
    rbq[j] = gg_rsrc(reinterpret_cast<const char*>(bm.q) + (size_t)e * args.N * qrow, (uint32_t)args.N * qrow);
    b_qoff[j] = bn < args.N ? (uint32_t)bn * qrow + 4u * BITS * g4 : kOob;
  }
  auto bload = [&](uint4 (*raw)[RL], int kt) {
    const bool live = kt < KT;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < RL; ++r)
        raw[j][r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(live ? rbq[j] : rnull, b_qoff[j] + 16 * r, kt * 16 * BITS, 0));
  };

  // Scales and biases: chunk c holds groups 8c..8c+7 (super-steps 4c..4c+3) of
  // the tile's BN rows, 16 bytes a row, in ring slot c % SLOTS. The first half of
  // the waves copies scales, the second biases, 64 rows each: one 16-byte
  // LDS-DMA per wave and chunk. Rows that start on 4-byte boundaries only (G
  // not a multiple of 8, or arrays off a 16-byte boundary) take four 4-byte
  // copies. A row's last chunk may read
  // past its groups (the next row's, never used, or zeros past the matrix).
  // Loaded straight into registers instead, as 2-byte values of 64 rows at a
  // time, they cost as much as the packed codes; kept for the whole input
  // width (32 KB at 2048) they cost 128-row tiles a workgroup per compute unit.
  // Piece p of 2 BN / 64: scales (p < BN / 64) or biases of rows 64 sw .. + 63.
  constexpr int SBP = 2 * BN / (64 * WAVES);      // pieces per wave
  const bool sb16 = args.sb16 != 0;
  auto sb_copy = [&](int c) {
#pragma unroll
    for (int u = 0; u < SBP; ++u) {
      const int p = u * WAVES + wave;
      const int sw = p % (BN / 64);
      const bool sbias = p >= BN / 64, sup = MODE == kGgGateUp && 64 * sw >= BN / 2;
      const tfm_affine& sm = sup ? args.wb : args.wa;
      const auto rsb = gg_rsrc(static_cast<const char*>(sbias ? sm.biases : sm.scales) + (size_t)e * args.N * srow,
                               (uint32_t)args.N * srow);
      const int sn0 = n0 + 64 * sw - (sup ? BN / 2 : 0);  // matrix row of the first
      uint16_t* const dst = sSb + ((c & (SLOTS - 1)) * 2 + (sbias ? 1 : 0)) * SBH + 64 * 8 * sw;
      const bool live = 8 * c < G;
      if (sb16) {
        const int n = sn0 + lane;
        lds_dma16(rsb, dst, live && n < args.N ? (uint32_t)n * srow + 16u * c : kOob, 0);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {             // dword 64 i + lane: row 16 i + lane / 4, pair lane % 4
          const int n = sn0 + 16 * i + (lane >> 2);
          lds_dma4(rsb, dst + 128 * i, live && n < args.N ? (uint32_t)n * srow + 16u * c + 4u * (lane & 3) : kOob);
        }
      }
    }
  };
  // scale and bias of super-step kt for both rows (past the end: last group)
  auto sb_read = [&](sb_t* sc, sb_t* bi, int kt) {
    int g = 2 * kt + (g4 >> 1);
    g = g < G ? g : G - 1;
    const uint16_t* const p = sSb + ((g >> 3) & (SLOTS - 1)) * 2 * SBH + (g & 7);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      sc[j] = D8::sb(p[trow[j] * 8]);
      bi[j] = D8::sb(p[trow[j] * 8 + SBH]);
    }
  };
  auto deq = [&](op_t* b, uint4 (*raw)[RL], const sb_t* sc, const sb_t* bi) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      D8 d;
      uint32_t o[4];
      const uint32_t* w = reinterpret_cast<const uint32_t*>(&raw[j][0]);
      static_for<0, 8>([&](auto el_) { d.template slice<decltype(el_)::value>(w, sc[j], bi[j], o); });
      b[j] = __builtin_bit_cast(op_t, make_uint4(o[0], o[1], o[2], o[3]));
    }
  };

  f32x4_t acc[MB][NJ];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // One super-step on activation stage A: sub-step s runs the MFMAs of the
  // MBL live row blocks with B operand b (word s) and dequantises the B
  // operand of the next sub-step (word s + 1, or word 0 of the next
  // super-step's raw weights). The (sub-step, row block) pairs run as one
  // compile-time sequence with the A fragment of pair q + D read while pair
  // q computes (a ring of D + 1 fragments); the scheduler is asked for the
  // first D reads, then per pair the read D pairs ahead, NJ MFMAs and its share
  // of the dequantisation slices. The activation copies of the next super-step (into
  // stage An) are issued one every STEP pairs over the first half of the
  // sequence: issued together they would hold the wave at the address unit,
  // with no MFMAs issued, for most of a thousand cycles. Only the NC copies
  // of rows below 16 MBL are issued: the other rows are never read.
  // Fragment address of row block i, sub-step s: the lane's byte offset
  // (row lane % 16, slot (4 g4) ^ (lane % 16)) XOR 16 s, plus 4096 i. The
  // lane offset is made opaque per super-step so that the four per-sub-step
  // addresses are formed there instead of being held across the loop.
  const uint32_t a_lane = (uint32_t)((lane & 15) * BK2 * 2 + (((4 * g4) ^ (lane & 15)) << 4));
  auto compute = [&](auto mbl_tag, const uint16_t* A, op_t* b, uint4 (*rc)[RL], const sb_t* sc,
                     const sb_t* bic, uint4 (*rn)[RL], const sb_t* sn, const sb_t* bin, uint16_t* An,
                     int ktn, auto weight_load) __attribute__((always_inline)) {
    constexpr int MBL = decltype(mbl_tag)::value;
    constexpr int NQ = 4 * MBL, D = AHEAD, R = D + 1;
    constexpr int CR = 4 * WAVES;  // rows per copy round
    constexpr int NC = (16 * MBL + CR - 1) / CR < LA ? (16 * MBL + CR - 1) / CR : LA;
    constexpr int STEP = NQ / (2 * NC) > 0 ? NQ / (2 * NC) : 1;
    static_assert(STEP * (NC - 1) < NQ, "every copy is issued");
    op_t af[R];
    uint32_t nbw[NJ][4];                          // next B operand, packed pairs
    D8 dq[NJ];
    uint32_t al = a_lane;
    asm volatile("" : "+v"(al));
    const char* const Ab = reinterpret_cast<const char*>(A);
    auto rd = [&](auto q_) {
      constexpr int q = decltype(q_)::value, s = q / MBL, i = q % MBL;
      af[q % R] = *reinterpret_cast<const op_t*>(Ab + (al ^ (16u * s)) + 16 * BK2 * 2 * i);
    };
    static_for<0, D>([&](auto q_) { rd(q_); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NQ>([&](auto q_) {
      constexpr int q = decltype(q_)::value, s = q / MBL, i = q % MBL;
      if constexpr (q % STEP == 0 && q / STEP < NC) a_copy1(An, ktn, std::integral_constant<int, q / STEP>{});
      if constexpr (q == (LATE ? MBL + MBL / 2 : STEP * (NC - 1))) weight_load();
      if constexpr (q + D < NQ) rd(std::integral_constant<int, q + D>{});
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = mfma16(af[q % R], b[j], acc[i][j], f16tag{});
      // Slices of the next sub-step's B operand: slice c of 8 NJ is slice c % 8
      // of row c / 8 (word(s) s + 1, or the first of the next super-step's raw
      // weights).
      constexpr int c0 = 8 * NJ * i / MBL, c1 = 8 * NJ * (i + 1) / MBL;
      static_for<c0, c1>([&](auto c_) {
        constexpr int c = decltype(c_)::value, j = c / 8, el = c % 8;
        constexpr int w0 = s < 3 ? RL * (s + 1) : 0;
        const uint32_t* rw = (s < 3 ? reinterpret_cast<const uint32_t*>(&rc[j][0]) : reinterpret_cast<const uint32_t*>(&rn[j][0])) + w0;
        dq[j].template slice<el>(rw, s < 3 ? sc[j] : sn[j], s < 3 ? bic[j] : bin[j], nbw[j]);
      });
      if constexpr (i == MBL - 1) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          b[j] = __builtin_bit_cast(op_t, make_uint4(nbw[j][0], nbw[j][1], nbw[j][2], nbw[j][3]));
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // Live row blocks (uniform over the workgroup), so that empty rows cost no
  // MFMAs: in steps of four of 16 blocks, of two of 8; 2, 4, 5 or 6 with 96-row
  // tiles; 1, 2 or 4 with 64-row ones (16, 32 or 64 rows).
  auto by_live = [&](auto f) __attribute__((always_inline)) {
    if constexpr (MB == 16) {
      if (rows_valid > 192) f(std::integral_constant<int, 16>{});
      else if (rows_valid > 128) f(std::integral_constant<int, 12>{});
      else if (rows_valid > 64) f(std::integral_constant<int, 8>{});
      else f(std::integral_constant<int, 4>{});
    } else if constexpr (MB == 8) {
      if (rows_valid > 96) f(std::integral_constant<int, 8>{});
      else if (rows_valid > 64) f(std::integral_constant<int, 6>{});
      else if (rows_valid > 32) f(std::integral_constant<int, 4>{});
      else f(std::integral_constant<int, 2>{});
    } else if constexpr (MB == 6) {
      if (rows_valid > 80) f(std::integral_constant<int, 6>{});
      else if (rows_valid > 64) f(std::integral_constant<int, 5>{});
      else if (rows_valid > 32) f(std::integral_constant<int, 4>{});
      else f(std::integral_constant<int, 2>{});
    } else {
      if (rows_valid > 32) f(std::integral_constant<int, 4>{});
      else if (rows_valid > 16) f(std::integral_constant<int, 2>{});
      else f(std::integral_constant<int, 1>{});
    }
  };
  // ---- few rows (FEW instances): weights two super-steps ahead ----
  // In the main loop every super-step ends at a barrier that waits for all
  // of its loads, and the raw weights of super-step k+1 (whose first word
  // the last sub-step of super-step k dequantises) are requested at the start
  // of super-step k: one super-step of loads in flight. A tile of at most 16
  // rows (one row block) has too few MFMAs per super-step to cover a memory
  // latency that way. Here the raw weights of super-step k+2 are requested
  // right after the activation copy of super-step k+1, and the barrier waits
  // only for that copy (the vector memory counter retires in issue order), so
  // they stay in flight across it. The products and their order are those of
  // the main loop.
  if (FEW && rows_valid <= 16 && (KT & 3) == 0 && (SLOTS == 2 || KT <= 4 * SLOTS)) {
    if constexpr (FEW) {
      static_assert(BM == 64 && RL == 1 && NJ == 2, "few-row tiles: 64 rows, two weight loads a super-step");
      uint4 rw[4][NJ][RL];                         // raw weights of super-step k in slot k % 4
      sb_t fsc[2][NJ], fbi[2][NJ];                  // scales and biases of super-step k in set k % 2
      op_t fb[NJ];
#pragma unroll
      for (int c = 0; c < (SLOTS == 2 ? 1 : SLOTS); ++c) sb_copy(c);
      a_copy(sA0, 0);
      bload(rw[0], 0);
      bload(rw[1], 1);
      __syncthreads();  // scale copies and stage 0 complete and visible
      sb_read(fsc[0], fbi[0], 0);
      deq(fb, rw[0], fsc[0], fbi[0]);
      for (int kt0 = 0; kt0 < KT; kt0 += 4) {
        static_for<0, 4>([&](auto q_) {
          constexpr int q = decltype(q_)::value, c = q % 2, n = 1 - c;
          const int kt = kt0 + q;
          uint16_t* const A = c == 0 ? sA0 : sA1;
          uint16_t* const An = c == 0 ? sA1 : sA0;
          sb_read(fsc[n], fbi[n], kt + 1);
          if constexpr (q == 0 && SLOTS == 2) sb_copy(kt0 / 4 + 1);
          __builtin_amdgcn_sched_barrier(0);
          compute(std::integral_constant<int, 1>{}, A, fb, rw[q], fsc[c], fbi[c], rw[(q + 1) % 4], fsc[n],
                  fbi[n], An, kt + 1, [&] {
                    __builtin_amdgcn_sched_barrier(0);  // copies first: the wait below counts what follows them
                    bload(rw[(q + 2) % 4], kt + 2);
                  });
          // This wave's copies are done (only the NJ weight loads issued after
          // them may be outstanding), then every wave's.
          asm volatile("s_waitcnt vmcnt(2)\n\ts_barrier" ::: "memory");
        });
      }
    }
  } else {
  // ---- prologue ----
  uint4 r0[NJ][RL], r1[NJ][RL];
  sb_t sc0[NJ], bi0[NJ], sc1[NJ], bi1[NJ];
  op_t bop[NJ];
  sb_copy(0);
  a_copy(sA0, 0);
  bload(r0, 0);
  __syncthreads();  // scale copies and stage 0 complete and visible
  sb_read(sc0, bi0, 0);
  deq(bop, r0, sc0, bi0);

  // Super-step S: load the raw weights of S+1 and read its scales, compute
  // (copying S+1 into the other stage on the way), barrier. With an odd
  // count the loop runs one more super-step on zero activations. Scale chunk
  // c + 1 is requested in super-step 4c: the last read of its ring slot's
  // old chunk (c - 1 in a ring of two) was before the barrier that ended super-step 4c - 2, and
  // its first read comes in super-step 4c + 3.
  auto main_loop = [&](auto mbl_tag) {
    for (int kt = 0; kt < KT; kt += 2) {
      if constexpr (!LATE) bload(r1, kt + 1);
      sb_read(sc1, bi1, kt + 1);
      if ((kt & 3) == 0) sb_copy(kt / 4 + 1);
      __builtin_amdgcn_sched_barrier(0);
      compute(mbl_tag, sA0, bop, r0, sc0, bi0, r1, sc1, bi1, sA1, kt + 1, [&] { if constexpr (LATE) bload(r1, kt + 1); });
      __syncthreads();
      if constexpr (!LATE) bload(r0, kt + 2);
      sb_read(sc0, bi0, kt + 2);
      __builtin_amdgcn_sched_barrier(0);
      compute(mbl_tag, sA1, bop, r1, sc1, bi1, r0, sc0, bi0, sA0, kt + 2, [&] { if constexpr (LATE) bload(r0, kt + 2); });
      __syncthreads();
    }
  };
  by_live(main_loop);
  }

  // ---- epilogue ----
  // Rows staged row-major, CP columns per pass (the first BM/2 rows in
  // stage 0, the rest in stage 1), then written as 16-byte row pieces.
  // Gate/up: one pass of BN/2 columns (wave w holds columns 8 NJ w .. + 8 NJ - 1
  // after SwiGLU); down and plain: BN/128 passes of 128 columns, pass p staged
  // by the waves that hold columns 128p..128p+127 (four of 32, two of 64).
  constexpr int PASSES = MODE == kGgGateUp ? 1 : BN / 128;
  constexpr int CP = MODE == kGgGateUp ? BN / 2 : 128;
  constexpr int PARTS = CP / 8;                   // 16-byte pieces per staged row
  constexpr int RPI = WAVES * 64 / PARTS;         // rows written per iteration
  static_assert(CP + 8 <= SROW, "staged row fits its stride");
  static_for<0, PASSES>([&](auto p_) {
    constexpr int p = decltype(p_)::value;
    if (p > 0) __syncthreads();  // the previous pass's reads are done
    const bool mine = MODE == kGgGateUp || WN * wave / 128 == p;
    if (mine) {
      static_for<0, MB>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        if (16 * i >= rows_valid) return;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * i + 4 * g4 + v;
          uint16_t* st = (row < HALF_ROWS ? sA0 : sA1) + (row % HALF_ROWS) * SROW;
          if constexpr (MODE == kGgGateUp) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
              st[16 * (NB * wave + j) + (lane & 15)] = f2st<F16>(swiglu(acc[i][j][v], acc[i][j + NB][v]));
          } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) st[WN * wave % 128 + 16 * j + (lane & 15)] = f2st<F16>(acc[i][j][v]);
          }
        }
      });
    }
    __syncthreads();
    const int part = tid % PARTS;
    const int n = n0 + CP * p + part * 8;
#pragma unroll
    for (int r0i = 0; r0i < BM; r0i += RPI) {
      const int row = r0i + tid / PARTS;
      if (row < rows_valid && n < args.N) {
        const uint16_t* st = (row < HALF_ROWS ? sA0 : sA1) + (row % HALF_ROWS) * SROW;
        const uint4 v = *reinterpret_cast<const uint4*>(&st[part * 8]);
        const int j = m0 + row;
        const int64_t orow = MODE == kGgPlain ? (int64_t)route_flat(args.rm, j) : (int64_t)j;
        *reinterpret_cast<uint4*>(&args.out[orow * args.N + n]) = v;
      }
    }
  });
}

static int tile_rows_env(const char* name) {
  const char* s = std::getenv(name);
  const int n = s ? std::atoi(s) : 0;
  return n == 64 || n == 96 || n == 128 || n == 256 ? n : 0;
}

static int tile_override() {
  static const int v = tile_rows_env("TFM_GGEMM_TILE");
  return v;
}

static int down_tile_override() {
  static const int v = tile_rows_env("TFM_GGEMM_DOWN_TILE");
  return v;
}

static int waves_override() {
  static const int v = [] {
    const char* s = std::getenv("TFM_GGEMM_WAVES");
    const int n = s ? std::atoi(s) : 0;
    return n == 4 || n == 8 ? n : 0;
  }();
  return v;
}

// Tile rows of ggemm_kernel.
static bool use_tall(int64_t n_routes, int E) {
  const int o = tile_override();
  if (o == 256) return true;
  if (o == 128 || o == 64) return false;
  return n_routes >= (int64_t)E * 384;
}

static int gg_device_cus() {
  static int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      return 256;
    return n;
  }();
  return cus;
}

// Tile of the weights-in-registers kernel: rows BM, waves WV and 16-row weight
// blocks a wave NJ.
struct WrTile {
  int bm, wv, nj;
};

// Chosen from the average routes per expert a = n_routes / E and the number
// of 256-weight-row column tiles (gate/up: gate and up rows together; `wide`:
// at least one a compute unit over the experts, as OLMoE's and unlike
// Granite's gate/up). Kernel us at OLMoE (64 experts, 2048 -> 2 x 1024 -> 2048)
// and Granite (40 experts, 1536 -> 2 x 512 -> 1536) sizes, as rows x waves:
//  * A dense matrix (few experts and columns): the largest tile whose count
//    fills the compute units, else 64 x 4 (2048 x 2048 linear: 1024 rows 64x4
//    19.1, 128x4 23.7; 2048 rows 28.4 and 26.4).
//  * 96 x 4 (64 weight rows a wave: half the LDS reads and activation copies
//    per product), 4-bit codes, wide, where experts of about a routes fill one
//    such tile (44 < a <= 72, three deviations of evenly spread routes below
//    96) or two where 128 rows would take two as well (128 < a <= 155). us per
//    layer, gate/up and down, against the other tiles: OLMoE 400 tokens 106.8
//    and 114.4, 512 tokens 118.5 and 125.0, 1111 tokens 193.3 and 203.7; past
//    the fit it loses: 700 tokens 162.5 and 136.1, 900 tokens 183.9 and 170.2.
//    Not 8-bit codes, whose raw weights leave it too few registers. (The lines
//    are those of evenly spread routes; half storage, whose affine routers spread
//    them more, gains earlier: 360 tokens gate/up 55.0 on 64x8 and 48.2.)
//  * Down. 64 x 4 up to a = 44 (OLMoE 300 tokens, a = 38: 29.2 against 32.8 on
//    128x4; 400 tokens: 34.7 and 34.2), then 128 x 4 (512 tokens 38.2 against
//    42.0 on 64x4 and 40.0 on 128x8; Granite 1024 tokens 27.6, 28.3 on 256x8;
//    2800 tokens 62.1 and 68.2): two workgroups a compute unit overlap one's
//    epilogue with the other's main loop. 256 x 8 from a = 448 where the input
//    is at least 1024 wide, so that the main loop outweighs the epilogue
//    (OLMoE 2800 tokens, a = 350: 131.4 on 128x4, 132.6 on 256x8; 4000 tokens:
//    181.2 and 173.7; Granite, 512 wide, 4000 tokens: 85.5 and 91.6).
//  * Gate/up and gathered products. 64 rows up to a = 44 wide, 56 otherwise
//    (OLMoE 300 tokens 49.0 against 54.6 on 128x8, 400 tokens 66.0 and 56.7;
//    Granite 256 tokens, a = 51, 21.8 and 23.7; 8-bit codes 400 tokens 63.0
//    and 73.6, so to a = 56 there, but to 48 with half storage, whose affine
//    routers spread the loads more: 400 tokens 84.6 and 75.2), with 8 waves
//    while that gives two tiles a compute unit and, for 8-bit codes, most experts
//    have a route, else 4 (8-bit codes at 8 tokens 39.5 against 47.4, at 20
//    tokens 53.8 and 53.5; 4-bit codes at 14 tokens 36.8 against 35.5, half 34.8
//    and 32.7).
//    128 rows to a = 232 wide (1700 tokens, a = 212: 138.8 against 153.3 on
//    256x8; 2048 tokens, a = 256: 170.9 and 160.5), 480 otherwise (Granite
//    1500 tokens, a = 300: 54.0 and 62.0; 2800, a = 560: 93.7 and 84.9): the
//    256-row tile dequantises its weights once for twice the rows, but with
//    few tiles its last round leaves much of the chip idle. Eight waves while
//    an expert has one m-tile (512 tokens 61.7 against 64.4 on 128x4; half
//    58.0 and 62.6), four above (900 tokens 97.4 against 102.2; Granite 2048
//    71.8 and 78.3).
//  * Gate/up of 4-bit codes with bf16 storage: 128 x 4 with 64 weight rows a
//    wave, against the tile above: wide 700 tokens (a = 87) 66.9 and 71.6, 800
//    tokens 69.6 and 77.0, 860 tokens 84.5 and 87.7, 1000 tokens 104.0 and 106.5,
//    1300 tokens 120.6 and 131.6, 1750 tokens 130.2 and 144.0, 2400 tokens 178.3 and 187.7, 4000
//    tokens 277.0 and 271.6 (256x8). Not wide, where its rounds are full
//    enough: Granite 1024 tokens (a = 205, 336 tiles in a round of 512) 47.8
//    and 43.4, 1500 tokens (454) 51.2 and 54.5, 2048 tokens (592 in two) 10 us
//    a layer slower, 2500 tokens (704) 74.6 and 84.5, 4000 tokens (1080 in
//    three) 114.9 and 123.9. (The down GEMM is level or slower on it; half storage
//    has too few registers for it.)
// The lines were drawn at those two sizes. 840 calls at ten more (8 to 64
// experts, 256 to 8192 wide) take 0.79 of the time they took under the rule
// before it (geometric mean), the slowest 1.09.
// TFM_GGEMM_TILE=64/96/128/256 forces the rows, TFM_GGEMM_DOWN_TILE those of the
// down GEMM alone (TFM_GGEMM_TILE takes precedence), TFM_GGEMM_WAVES=4/8 the
// waves (of tiles of 64 or 128 rows that do not have that many already).
static WrTile wr_tile(int64_t n_routes, int E, int64_t cols, int kin, int mode, int bits, bool f16) {
  const int64_t cus = gg_device_cus();
  auto mtiles = [&](int bm) { return (n_routes + (int64_t)E * bm - 1) / ((int64_t)E * bm); };
  auto upto = [&](int a) { return n_routes <= (int64_t)E * a; };  // average routes at most a
  auto pick = [&]() -> WrTile {
    if (4 * E * cols < cus) {
      if (E * mtiles(256) * cols >= cus) return {256, 8, 2};
      if (E * mtiles(128) * cols * 2 >= cus) return {128, 4, 2};
      return {64, 4, 2};
    }
    const bool wide = E * cols >= cus;
    if (wide && bits == 4 && ((!upto(44) && upto(72)) || (!upto(128) && upto(155)))) return {96, 4, 4};
    if (mode == kGgDown) {
      if (upto(bits == 8 ? 56 : 44)) return {64, 4, 2};
      if (n_routes >= (int64_t)E * 448 && kin >= 1024) return {256, 8, 2};
      return {128, 4, 2};
    }
    if (upto(!wide ? 56 : bits == 4 ? 44 : f16 ? 48 : 56))
      return {64, (bits == 4 || n_routes > 2 * E) && E * mtiles(64) * cols >= 2 * cus ? 8 : 4, 2};
    if (mode == kGgGateUp && bits == 4 && !f16) {
      if (wide && upto(400)) return {128, 4, 4};
      // Tiles of E experts of a / 128 + 1/2 m-tiles, two a compute unit: the
      // rounds must be two thirds full.
      const int64_t tiles = (n_routes + (int64_t)E * 64) * cols / 128, round = 2 * cus;
      if (!wide && !upto(150) && 3 * tiles >= 2 * ((tiles + round - 1) / round) * round) return {128, 4, 4};
    }
    // 256-row tiles in one round of the compute units where 128-row ones need
    // more (Granite 700 tokens, a = 140: 35.1 against 38.8 on 128x4; 8-bit codes
    // 1000 tokens 45.5 and 49.6). With long and short tiles the live rows may
    // take at most 5/8 of their places: an XCD's run holds a tile or two more than an even share, and where
    // no tile is short that is a second round (64 experts 512 -> 2 x 256, a = 375: half
    // 34.1, bf16 45.8 for 8-bit codes, against 29.4 and 31.7 on 128x8; a = 275, whose
    // second tiles are nearly empty: 25.9 and 29.3 on 128x4).
    const int64_t live = (n_routes + (int64_t)E * 64 - 1) / ((int64_t)E * 64) * 64 * E * cols;
    if (!wide && E * mtiles(128) * cols > cus && E * mtiles(256) * cols <= cus &&
        (mtiles(256) == 1 || 8 * live <= 5 * 256 * cus))
      return {256, 8, 2};
    if (n_routes >= (int64_t)E * (wide ? 232 : 480)) return {256, 8, 2};
    // Eight waves also where their 128-row tiles take one well-filled round
    // (Granite 600 tokens: half 29.4 on 128x4 and 27.0, 8-bit codes 34.9 and 33.0).
    const int64_t round = E * mtiles(128) * cols;
    if (mode == kGgGateUp && !wide && 8 * round >= 5 * cus && round <= cus) return {128, 8, 2};
    return {128, upto(104) ? 8 : 4, 2};
  };
  const WrTile t = pick();
  int bm = tile_override();
  if (!bm) bm = mode == kGgDown ? down_tile_override() : 0;
  const int wv = waves_override();
  if ((!bm || bm == t.bm) && (!wv || wv == t.wv)) return t;
  if (!bm) bm = t.bm;
  if (bm == 96) return {96, 4, 4};
  if (bm == 256) return {256, 8, 2};
  return {bm, wv ? wv : bm == t.bm ? t.wv : bm == 64 ? 4 : 8, 2};
}

static unsigned grid_for(int64_t n_routes, int E, int BM, int NT) {
  const int64_t mt_max = (n_routes + BM - 1) / BM + (n_routes < E ? n_routes : E);
  int64_t total = mt_max * NT;
  // round up to a multiple of 8 so every XCD share is complete
  total = (total + 7) / 8 * 8;
  if (total < 8) total = 8;
  return (unsigned)total;
}

// Low address bits of the scale and bias arrays, which a caller may start at
// any element: copies into LDS need 4- or 16-byte boundaries.
static uintptr_t sb_address_bits(const GgArgs& a) {
  return reinterpret_cast<uintptr_t>(a.wa.scales) | reinterpret_cast<uintptr_t>(a.wa.biases) |
         reinterpret_cast<uintptr_t>(a.wb.scales) | reinterpret_cast<uintptr_t>(a.wb.biases);
}

template <int BM_, int BN_, int WAVES_M, int WAVES_N, int MODE, int BITS, bool F16>
static void launch_one(const GgArgs& a, int64_t n_routes, int E, hipStream_t s) {
  using C = GgCfg<BM_, BN_, WAVES_M, WAVES_N, MODE, BITS>;
  const int NT = (a.N + C::OUT_COLS - 1) / C::OUT_COLS;
  if (a.Kin <= kLdsScaleKin && (sb_address_bits(a) & 15) == 0)
    tfm_launch(ggemm_kernel<BM_, BN_, WAVES_M, WAVES_N, MODE, BITS, F16, true>, grid_for(n_routes, E, BM_, NT), C::THREADS, 0, s, a);
  else
    tfm_launch(ggemm_kernel<BM_, BN_, WAVES_M, WAVES_N, MODE, BITS, F16, false>, grid_for(n_routes, E, BM_, NT), C::THREADS, 0, s, a);
}

// The FEW instance of a 64-row launch (tiles of at most 16 rows keep their
// weights two super-steps ahead) runs where experts average at most
// kFewRowsAvg routes, so that most tiles hold at most 16 rows.
// TFM_GGEMM_FEW_ROWS=0 never uses it, =2 uses it for every 64-row launch.
constexpr int kFewRowsAvg = 12;
static bool use_few_rows(int64_t n_routes, int E) {
  static const int v = [] {
    const char* s = std::getenv("TFM_GGEMM_FEW_ROWS");
    return s && (s[0] == '0' || s[0] == '2') && s[1] == 0 ? s[0] - '0' : 1;
  }();
  return v == 2 || (v == 1 && n_routes <= (int64_t)E * kFewRowsAvg);
}

template <int BM, int MODE, int BITS, bool F16, int WV, int NJ = 2>
static void launch_wr(const GgArgs& a, int64_t n_routes, int E, hipStream_t s) {
  constexpr int OUT_COLS = (MODE == kGgGateUp ? 8 : 16) * NJ * WV;
  const int NT = (a.N + OUT_COLS - 1) / OUT_COLS;
  // With 256-row tiles an XCD's run of cheap tiles holds more tiles than an
  // even share: at most share x 29 / 17 + 2 (full tile 29 units, cheapest
  // 17); workgroups past their XCD's run exit at once.
  unsigned grid = grid_for(n_routes, E, BM, NT);
  if (BM == 256) grid = ((grid / 8 * 29 + 16) / 17 + 2) * 8;
  if constexpr (BM == 64 && BITS == 4) {
    if (use_few_rows(n_routes, E)) {
      tfm_launch(ggemm_wr_kernel<BM, MODE, BITS, F16, WV, true>, grid, WV * 64, 0, s, a);
      return;
    }
  }
  tfm_launch(ggemm_wr_kernel<BM, MODE, BITS, F16, WV, false, NJ>, grid, WV * 64, 0, s, a);
}

// 8-bit codes with bf16 storage, inputs up to 2048 wide: where the 256-row tiles
// of ggemm_kernel beat ggemm_wr_kernel. A code costs two to three vector
// instructions there either way, but a wave of 128 x 64 outputs reads a
// third less LDS than eight waves that each read the whole activation tile. us,
// ggemm_kernel against the tile wr_tile picks, a = routes per expert:
//  * Down and gathered products from a = 384, with more than half a round of the
//    compute units in full tiles: OLMoE 3072 tokens 139 and 154, 3600 158
//    and 174, Granite 2200 47 and 55, 6000 114 and 125; 16 experts 384 ->
//    768 at 4096 tokens 21 and 28. Fewer tiles leave too much idle
//    (16 experts 2048 -> 1024, 3072 tokens: 50 and 38; 2048 x 2048 linear, 4096
//    rows: 54 and 43). Not around a = 512, where
//    many experts start a third tile (Granite 2500 tokens 64 and 59).
//  * Gathered products from a = 57 to 150 with two rounds of 128-row tiles: 64
//    experts 1408 -> 2048, 4000 rows 70.1 and 72.6, 8000 rows 103.7 and 112.0;
//    12000 rows level, and 2048 -> 1408 133.7 and 126.4.
//  * Gate/up from 384 to 480 where two tiles an expert fill their rounds: OLMoE
//    3600 tokens 260 and 270, 32 experts 1024 -> 2 x 512 at 3500 tokens 39 and
//    49; Granite (320 tiles in two rounds) level. Beyond, level or up to 4%
//    slower (OLMoE 6000 tokens 421 and 406), except with few column tiles (16
//    experts 768 -> 2 x 384 at 4096 tokens 30 and 39).
static bool lds_dequant(int64_t n_routes, int E, int64_t cols, int kin, int mode) {
  if (kin > kLdsScaleKin || tile_override() || waves_override() || (mode == kGgDown && down_tile_override())) return false;
  const int64_t cus = gg_device_cus();
  auto avg = [&](int a) { return n_routes >= (int64_t)E * a; };
  const bool tall = avg(384) && 2 * n_routes * cols > 256 * cus;
  if (mode == kGgGateUp) {
    const int64_t tiles = 2 * E * cols;
    return tall && (4 * E * cols < cus || (!avg(480) && 4 * tiles >= 3 * ((tiles + cus - 1) / cus) * cus));
  }
  if (mode == kGgPlain && avg(57) && !avg(150) &&
      (n_routes + (int64_t)E * 128 - 1) / ((int64_t)E * 128) * E * cols >= 2 * cus)
    return true;
  return tall && !(avg(480) && !avg(528));
}

// Inputs a multiple of 128 wide: weights in registers (ggemm_wr_kernel);
// otherwise (odd multiples of 64, or scales or biases off a 4-byte boundary,
// which only 2-byte loads reach) ggemm_kernel.
template <int MODE, int BITS, bool F16>
static void launch_tile(const GgArgs& a_in, int64_t n_routes, int E, hipStream_t s) {
  GgArgs a = a_in;
  const uintptr_t sb = sb_address_bits(a);
  a.sb16 = (sb & 15) == 0 && a.Kin / BK % 8 == 0;
  const int64_t cols = ((MODE == kGgGateUp ? 2 : 1) * (int64_t)a.N + 255) / 256;
  const bool lds = BITS == 8 && !F16 && (sb & 15) == 0 && lds_dequant(n_routes, E, cols, a.Kin, MODE);
  if (a.Kin % BK2 == 0 && (sb & 3) == 0 && !lds) {
    const WrTile t = wr_tile(n_routes, E, cols, a.Kin, MODE, BITS, F16);
    if constexpr (BITS == 4) {
      if (t.bm == 96) {
        launch_wr<96, MODE, BITS, F16, 4, 4>(a, n_routes, E, s);
        return;
      }
    }
    if constexpr (BITS == 4 && !F16 && MODE == kGgGateUp) {
      if (t.bm == 128 && t.nj == 4) {
        launch_wr<128, MODE, BITS, F16, 4, 4>(a, n_routes, E, s);
        return;
      }
    }
    if (t.bm == 256) launch_wr<256, MODE, BITS, F16, 8>(a, n_routes, E, s);
    else if (t.bm == 128 && t.wv == 8) launch_wr<128, MODE, BITS, F16, 8>(a, n_routes, E, s);
    else if (t.bm == 128) launch_wr<128, MODE, BITS, F16, 4>(a, n_routes, E, s);
    else if (t.wv == 8) launch_wr<64, MODE, BITS, F16, 8>(a, n_routes, E, s);
    else launch_wr<64, MODE, BITS, F16, 4>(a, n_routes, E, s);
    return;
  }
  if (use_tall(n_routes, E))
    launch_one<256, 256, 2, 4, MODE, BITS, F16>(a, n_routes, E, s);
  else
    launch_one<128, 256, 2, 4, MODE, BITS, F16>(a, n_routes, E, s);
}

#define TFM_GG_RUN2(b, t) ggemm_run_##b##_##t
#define TFM_GG_RUN1(b, t) TFM_GG_RUN2(b, t)
#define TFM_GG_RUN TFM_GG_RUN1(TFM_GG_BITS, TFM_GG_F16)

void TFM_GG_RUN(int mode, const GgArgs& a, int64_t n_routes, int E, hipStream_t s) {
  constexpr int BITS = TFM_GG_BITS;
  constexpr bool F16 = TFM_GG_F16 != 0;
  switch (mode) {
    case kGgGateUp: launch_tile<kGgGateUp, BITS, F16>(a, n_routes, E, s); break;
    case kGgDown: launch_tile<kGgDown, BITS, F16>(a, n_routes, E, s); break;
    default: launch_tile<kGgPlain, BITS, F16>(a, n_routes, E, s); break;
  }
}

#if TFM_GG_MAIN
void ggemm_run_4_1(int mode, const GgArgs& a, int64_t n_routes, int E, hipStream_t s);
void ggemm_run_8_0(int mode, const GgArgs& a, int64_t n_routes, int E, hipStream_t s);
void ggemm_run_8_1(int mode, const GgArgs& a, int64_t n_routes, int E, hipStream_t s);

template <int MODE>
static void launch_mode(const GgArgs& a, int bits, bool f16, int64_t n_routes, int E, hipStream_t s) {
  if (bits == 8 && f16)
    ggemm_run_8_1(MODE, a, n_routes, E, s);
  else if (bits == 8)
    ggemm_run_8_0(MODE, a, n_routes, E, s);
  else if (f16)
    ggemm_run_4_1(MODE, a, n_routes, E, s);
  else
    ggemm_run_4_0(MODE, a, n_routes, E, s);
}

// TFM_GGEMM_SB_LAYOUT chose between layouts of whole-width scales in LDS. The
// four-super-step ring has one, so the variable is accepted and said to do nothing.
static void note_sb_layout() {
  static const bool noted = [] {
    const char* s = std::getenv("TFM_GGEMM_SB_LAYOUT");
    if (s) std::fprintf(stderr, "trifuse_moe: TFM_GGEMM_SB_LAYOUT=%s has no effect (scales and biases have one layout)\n", s);
    return s != nullptr;
  }();
  (void)noted;
}

static void check_shapes(int N, int Kin, int bits, int64_t x_rows) {
  note_sb_layout();
  if (bits != 4 && bits != 8) fail(TFM_E_UNSUPPORTED, "grouped GEMM: weights must be 4-bit or 8-bit");
  if (Kin % BK != 0) fail(TFM_E_UNSUPPORTED, "grouped GEMM: input width must be a multiple of 64");
  if (N % 64 != 0) fail(TFM_E_UNSUPPORTED, "grouped GEMM: output width must be a multiple of 64");
  // Buffer offsets are 32-bit: activations and one expert's packed weights
  // must stay below 2 GiB.
  if ((double)x_rows * Kin * 2 >= 2147483648.0 || (double)N * Kin * bits / 8 >= 2147483648.0)
    fail(TFM_E_UNSUPPORTED, "grouped GEMM: operand of 2 GiB or more");
}

void launch_ggemm_gateup(const uint16_t* x, RowMap rm, const Grouping& g, int64_t n_routes,
                         int E, const tfm_affine& gate, const tfm_affine& up, int N, int Kin,
                         int bits, bool f16, uint16_t* h, hipStream_t s) {
  if (n_routes <= 0) return;
  check_shapes(N, Kin, bits, rm.nx);
  GgArgs a{};
  a.x = x; a.x_bytes = (uint32_t)(rm.nx * Kin * 2); a.rm = rm; a.g = g; a.wa = gate; a.wb = up;
  a.N = N; a.Kin = Kin; a.out = h;
  launch_mode<kGgGateUp>(a, bits, f16, n_routes, E, s);
  check_hip(hipGetLastError(), "grouped GEMM gate/up launch");
}

void launch_ggemm_down(const uint16_t* hsorted, const Grouping& g, int64_t n_routes, int E,
                       const tfm_affine& w, int N, int Kin, int bits, bool f16, uint16_t* y_sorted,
                       hipStream_t s) {
  if (n_routes <= 0) return;
  check_shapes(N, Kin, bits, n_routes);
  GgArgs a{};
  a.x = hsorted; a.x_bytes = (uint32_t)(n_routes * Kin * 2);
  a.rm = RowMap{g.order, nullptr, 1, 0, nullptr}; a.g = g; a.wa = w; a.wb = w; a.N = N;
  a.Kin = Kin; a.out = y_sorted;
  launch_mode<kGgDown>(a, bits, f16, n_routes, E, s);
  check_hip(hipGetLastError(), "grouped GEMM down launch");
}

void launch_ggemm_plain(const uint16_t* x, RowMap rm, const Grouping& g, int64_t n_routes,
                        int E, const tfm_affine& w, int N, int Kin, int bits, bool f16, uint16_t* out,
                        hipStream_t s) {
  if (n_routes <= 0) return;
  check_shapes(N, Kin, bits, rm.nx);
  GgArgs a{};
  a.x = x; a.x_bytes = (uint32_t)(rm.nx * Kin * 2); a.rm = rm; a.g = g; a.wa = w; a.wb = w;
  a.N = N; a.Kin = Kin; a.out = out;
  launch_mode<kGgPlain>(a, bits, f16, n_routes, E, s);
  check_hip(hipGetLastError(), "grouped GEMM plain launch");
}

#endif  // TFM_GG_MAIN

}  // namespace tfm
