// Router linear, OLMoE/Granite routing and the OLMoE softmax.
//
// Bit-defined arithmetic (the routing must reproduce exactly):
//  * logits[t,e] = bf16(tree64(s_0..s_63) [+ bias[e]]), lane l summing
//    x*w over h in [l*c, l*c+c) (c = H/64) with sequential fmaf from 0, and
//    tree64 the natural pairwise tree over lanes (l^1 first, then l^2, ...).
//  * softmax: max by compare-select from -FLT_MAX (NaN skipped), e = exp(l-max)
//    with route_expf, normaliser = 1/(tree over four-value chunks, each chunk
//    summed in order), p = e * normaliser (MLXOLMoERouter.h:26-61).
//  * ranks as in MLXOLMoERouter.h:65-83 (OLMoE) and
//    MLXNativeGraniteMoEPrefill.h:92-109 (Granite).
#include "route_wave.h"
#include "tfm_device.h"
#include "tfm_internal.h"

#pragma clang fp contract(off)

namespace tfm {

// One wave per (token tile of TW tokens, expert tile of EPW experts).
template <int C, int TW, bool F16>
__global__ __launch_bounds__(256) void router_logits_kernel(const uint16_t* __restrict__ x,
                                                            const uint16_t* __restrict__ w,
                                                            const float* __restrict__ bias,
                                                            int T, int H, int E, int EPW,
                                                            uint16_t* __restrict__ logits) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n_tt = (T + TW - 1) / TW;
  const int n_et = (E + EPW - 1) / EPW;
  if (wave >= n_tt * n_et) return;
  const int tt = wave % n_tt, et = wave / n_tt;
  float xv[TW][C];
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    const int tok = tt * TW + t;
    if (tok < T) {
      const uint4* src = reinterpret_cast<const uint4*>(x + (int64_t)tok * H + lane * C);
#pragma unroll
      for (int i = 0; i < C / 8; ++i) {
        const uint4 v = src[i];
        xv[t][8 * i + 0] = lo_st<F16>(v.x); xv[t][8 * i + 1] = hi_st<F16>(v.x);
        xv[t][8 * i + 2] = lo_st<F16>(v.y); xv[t][8 * i + 3] = hi_st<F16>(v.y);
        xv[t][8 * i + 4] = lo_st<F16>(v.z); xv[t][8 * i + 5] = hi_st<F16>(v.z);
        xv[t][8 * i + 6] = lo_st<F16>(v.w); xv[t][8 * i + 7] = hi_st<F16>(v.w);
      }
    } else {
#pragma unroll
      for (int j = 0; j < C; ++j) xv[t][j] = 0.0f;
    }
  }
  const int e_end = min(E, (et + 1) * EPW);
  for (int e = et * EPW; e < e_end; ++e) {
    float wv[C];
    const uint4* src = reinterpret_cast<const uint4*>(w + (int64_t)e * H + lane * C);
#pragma unroll
    for (int i = 0; i < C / 8; ++i) {
      const uint4 v = src[i];
      wv[8 * i + 0] = lo_st<F16>(v.x); wv[8 * i + 1] = hi_st<F16>(v.x);
      wv[8 * i + 2] = lo_st<F16>(v.y); wv[8 * i + 3] = hi_st<F16>(v.y);
      wv[8 * i + 4] = lo_st<F16>(v.z); wv[8 * i + 5] = hi_st<F16>(v.z);
      wv[8 * i + 6] = lo_st<F16>(v.w); wv[8 * i + 7] = hi_st<F16>(v.w);
    }
    const float be = bias ? bias[e] : 0.0f;
    if constexpr (TW == 4) {
      float s[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        s[t] = 0.0f;
#pragma unroll
        for (int j = 0; j < C; ++j) s[t] = __builtin_fmaf(xv[t][j], wv[j], s[t]);
      }
      // Row t of the wave holds token t's logit.
      const float r = wave_tree_sum64x4(s[0], s[1], s[2], s[3]);
      const int tok = tt * 4 + (lane >> 4);
      if ((lane & 15) == 0 && tok < T) logits[(int64_t)tok * E + e] = f2st<F16>(bias ? r + be : r);
    } else {
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < C; ++j) s = __builtin_fmaf(xv[t][j], wv[j], s);
        s = wave_tree_sum64(s);
        const int tok = tt * TW + t;
        if (lane == 63 && tok < T) {
          const float v = bias ? s + be : s;
          logits[(int64_t)tok * E + e] = f2st<F16>(v);
        }
      }
    }
  }
}

// Prefill routing in one pass: router linear, top-k and the chunk histogram
// for the grouping, 4 or 16 tokens a workgroup of eight waves.
//
// The logits run on the matrix cores in their bit-defined order: an fp32 MFMA
// of k = 1 adds one product to each accumulator with a single rounding
// (subnormal results included), so a chain of C of them over the elements of
// lane segment l is the sequential fused multiply-add chain of that segment.
//  * 4 tokens: v_mfma_f32_4x4x1 (16 blocks: 16 segments of 4 tokens x 4
//    experts). Wave (m, half) holds segments 16m..16m+15 of half the experts;
//    lane 4b+i supplies x of token i and w of expert i in segment 16m+b, and
//    receives the 4 tokens' sums of expert i. The pairwise tree then runs over
//    the lanes' b (two DPP shifts, two lane-half exchanges that also move token
//    t to row t), and over m through LDS.
//  * 16 tokens: v_mfma_f32_16x16x1 (4 blocks: 4 segments of 16 tokens x 16
//    experts). Wave v holds segments 8v..8v+7 of every expert; lane 16b+i
//    supplies row i in segment 4q+b of its quad q. The tree's first three
//    levels are sums of a lane's registers, the last three go through LDS.
// Wave t then ranks tokens t, t + 8, .. from LDS as topk_kernel does.
//
// Operands come through LDS, because a lane's segment is C x 2 contiguous
// bytes: loaded straight into registers, every 16-byte load of a wave touches
// 64 separate 64-byte pieces, and the address unit takes about 64 cycles over
// it (256 such loads a workgroup: 4-token workgroups took 15.8 us however few
// there were, 11.4 through LDS). The copies read rows contiguously; the slot
// of a chunk is rotated by its row, so that the 16 lanes of a read pass hit 16
// bank groups. Router rows are private to a wave, two slots deep.
//
// Bound: 2 E H flop per token at 256 flop per clock and compute unit in the
// 16 x 16 form (the 4 x 4 form measured about a quarter of that), and the E H
// x 2 bytes of router rows per workgroup from L2. The 4-token form runs up to
// 1024 tokens, in one round of one workgroup a compute unit (75 workgroups at
// 300 tokens, 256 at 1024), where latency and not the few products is the bound;
// beyond, 16 tokens read the router a quarter as often.
__device__ __forceinline__ void route_dma16(__amdgpu_buffer_rsrc_t r, uint16_t* dst, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, 0, 0, 0);
#else
  (void)r; (void)dst; (void)voff;
#endif
}

// Ranks token t0 + t of the block from its E logits in LDS and counts its
// routes (whole wave).
template <int ROUTE, bool F16>
__device__ __forceinline__ void rank_token(const uint16_t* row, int64_t tok, int E, int K, int32_t* __restrict__ idx,
                                           float* __restrict__ gates_f32, int* h) {
  const int lane = threadIdx.x & 63;
  float g;
  int id;
  if (ROUTE == TFM_ROUTE_OLMOE) {
    uint16_t gb;
    id = olmoe_route_wave<F16>(row, E, K, &g, &gb);
  } else {
    id = granite_route_wave<F16>(row, E, K, &g);
  }
  if (lane < K) {
    idx[tok * K + lane] = id;
    gates_f32[tok * K + lane] = g;
    atomicAdd(&h[id], 1);
  }
}

template <int C, int ROUTE, bool F16, int NTW>
__global__ __launch_bounds__(512) void router_topk4_kernel(const uint16_t* __restrict__ x,
                                                           const uint16_t* __restrict__ w,
                                                           const float* __restrict__ bias, int T, int H, int E, int K,
                                                           int32_t* __restrict__ idx, float* __restrict__ gates_f32,
                                                           int32_t* __restrict__ hist) {
  constexpr int SEG = C / 8;                      // 16-byte chunks per lane segment
  constexpr int TS = 2;                           // expert tiles a step: two MFMA chains
  constexpr int STEPS = (NTW + TS - 1) / TS;
  constexpr int PE = 68;                          // padded row of 64 experts
  constexpr int ROW = 512;                        // a 1 KB row: 64 slots of 8 elements
  __shared__ __attribute__((aligned(16))) uint16_t s_x[4][4][ROW];
  __shared__ __attribute__((aligned(16))) uint16_t s_w0[8][4 * TS][ROW];
  __shared__ __attribute__((aligned(16))) uint16_t s_w1[8][4 * TS][ROW];
  __shared__ int h[65];
  // After the products the token rows are dead: partial sums, then logits.
  float (*const part)[4][PE] = reinterpret_cast<float (*)[4][PE]>(&s_x[0][0][0]);
  uint16_t (*const s_logit)[64] = reinterpret_cast<uint16_t (*)[64]>(&s_x[0][0][0] + 4 * 4 * PE * 2);
  static_assert(4 * 4 * PE * 4 + 4 * 64 * 2 <= (int)sizeof(s_x), "partial sums and logits fit the token rows");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid <= E) h[tid] = 0;
  const int t0 = blockIdx.x * 4;
  const int m = wave & 3, e0 = (wave >> 2) * 4 * NTW;
  const int b = lane >> 2, i4 = lane & 3;

  // Rows past T and past E are beyond their buffers and read as zero.
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x + (int64_t)t0 * H), (short)0, min(4, T - t0) * H * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(w), (short)0, E * H * 2, 0x00020000);
  // Chunk (b, s) of a row with index i mod 4 sits in slot (b SEG + s + rot(i))
  // mod 64; the byte offset within its row of the chunk that lane l copies to
  // slot l (slots past the segments' chunks get zeros).
  auto rot = [](int i) { return SEG == 4 ? i : SEG == 2 ? (i & 1) + 8 * (i >> 1) : 4 * i; };
  auto src = [&](int i, int mm) -> uint32_t {
    const int c = (lane - rot(i)) & 63;
    return c < 16 * SEG ? (uint32_t)(16 * mm * SEG + c) * 16u : 0x80000000u;
  };
  for (int q = wave; q < 16; q += 8) {
    const int t = q >> 2, mm = q & 3;
    route_dma16(rx, &s_x[mm][t][0], (uint32_t)t * H * 2 + src(t, mm));
  }
  uint32_t wsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wsrc[i] = src(i, m);
  auto copy_w = [&](uint16_t (*dst)[ROW], int step) {
#pragma unroll
    for (int r = 0; r < 4 * TS; ++r)
      route_dma16(rw, dst[r], (uint32_t)(e0 + 4 * TS * step + r) * H * 2 + wsrc[r & 3]);
  };
  copy_w(s_w0[wave], 0);
  __syncthreads();  // token rows and the first router rows are in LDS
  if constexpr (STEPS > 1) copy_w(s_w1[wave], 1);

  auto slot = [&](int s) { return ((b * SEG + s + rot(i4)) & 63) * 8; };
  f32x4_t acc[STEPS * TS];
#pragma unroll
  for (int n = 0; n < STEPS * TS; ++n) acc[n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int step = 0; step < STEPS; ++step) {
    uint16_t (*const ws)[ROW] = step % 2 == 0 ? s_w0[wave] : s_w1[wave];
    uint4 wr[TS][SEG], xr[SEG];
#pragma unroll
    for (int s = 0; s < SEG; ++s) {
      xr[s] = *reinterpret_cast<const uint4*>(&s_x[m][i4][slot(s)]);
#pragma unroll
      for (int n = 0; n < TS; ++n) wr[n][s] = *reinterpret_cast<const uint4*>(&ws[4 * n + i4][slot(s)]);
    }
    // The slot is read before it is copied over.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (step + 2 < STEPS) copy_w(ws, step + 2);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const uint32_t v = word_of(xr[j >> 3], (j >> 1) & 3);
      const float xv = j & 1 ? hi_st<F16>(v) : lo_st<F16>(v);
#pragma unroll
      for (int n = 0; n < TS; ++n) {
        const uint32_t u = word_of(wr[n][j >> 3], (j >> 1) & 3);
        acc[TS * step + n] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv, j & 1 ? hi_st<F16>(u) : lo_st<F16>(u), acc[TS * step + n], 0, 0, 0);
      }
    }
    // Next step's rows (a wave's own copies, in order) have arrived once only
    // those requested after them may be outstanding.
    if (step + 2 < STEPS)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * TS) : "memory");
    else if (step + 1 < STEPS)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __syncthreads();  // every wave is done with the token rows
#pragma unroll
  for (int n = 0; n < NTW; ++n) {
    float v[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      v[t] = acc[n][t];
      v[t] = dpp_plus<0x104, 0xf>(v[t]);          // row_shl:4  (segment ^ 1), kept by lanes 0-3 and 8-11 of a row
      v[t] = dpp_plus<0x108, 0xf>(v[t]);          // row_shl:8  (segment ^ 2), kept by lanes 0-3
    }
    const float r = row_roots4(v[0], v[1], v[2], v[3]);  // segments ^ 4 and ^ 8; row t: token t
    if ((lane & 15) < 4) part[m][lane >> 4][e0 + 4 * n + (lane & 15)] = r;
  }
  __syncthreads();
  if (tid < 256) {
    const int t = tid >> 6, e = tid & 63;
    if (e < E) {
      const float lg = (part[0][t][e] + part[1][t][e]) + (part[2][t][e] + part[3][t][e]);
      s_logit[t][e] = f2st<F16>(bias ? lg + bias[e] : lg);
    }
  }
  __syncthreads();  // every expert's logits of the block's tokens are in LDS
  if (wave < 4 && t0 + wave < T)  // wave-uniform
    rank_token<ROUTE, F16>(s_logit[wave], (int64_t)t0 + wave, E, K, idx, gates_f32, h);
  __syncthreads();
  if (tid <= E) hist[(int64_t)blockIdx.x * (E + 1) + tid] = h[tid];
}

template <int C, int ROUTE, bool F16, int NT>
__global__ __launch_bounds__(512) void router_topk16_kernel(const uint16_t* __restrict__ x,
                                                            const uint16_t* __restrict__ w,
                                                            const float* __restrict__ bias, int T, int H, int E, int K,
                                                            int32_t* __restrict__ idx, float* __restrict__ gates_f32,
                                                            int32_t* __restrict__ hist) {
  constexpr int SEG = C / 8;                      // 16-byte chunks per lane segment
  constexpr int ROW = 256;                        // a wave's 512 bytes of a row: 32 slots of 8 elements
  constexpr int PE = 68;
  __shared__ __attribute__((aligned(16))) uint16_t s_r0[8][16][ROW];
  __shared__ __attribute__((aligned(16))) uint16_t s_r1[8][16][ROW];
  __shared__ uint16_t s_logit[16][64];
  __shared__ int h[65];
  float (*const part)[16][PE] = reinterpret_cast<float (*)[16][PE]>(&s_r0[0][0][0]);  // after the products
  static_assert(8 * 16 * PE * 4 <= (int)sizeof(s_r0), "partial sums fit a ring slot");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid <= E) h[tid] = 0;
  const int t0 = blockIdx.x * 16;
  const int b = lane >> 4, i16 = lane & 15;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x + (int64_t)t0 * H), (short)0, min(16, T - t0) * H * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(w), (short)0, E * H * 2, 0x00020000);
  // 16 rows (tokens, or the experts of tile n) of this wave's 8 segments, two
  // rows a copy: chunk c of row r in slot (c + r) mod 32.
  auto copy16 = [&](__amdgpu_buffer_rsrc_t rs, uint16_t (*dst)[ROW], int first) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int r = 2 * k + (lane >> 5);
      const int c = ((lane & 31) - r) & 31;
      route_dma16(rs, dst[2 * k], c < 8 * SEG ? (uint32_t)(first + r) * H * 2 + (uint32_t)(8 * wave * SEG + c) * 16u : 0x80000000u);
    }
  };
  auto slot = [&](int q, int s) { return (((4 * q + b) * SEG + s + i16) & 31) * 8; };
  // Ring order: tokens, then expert tiles 0 .. NT-1. Rows are private to the
  // wave, so its own wait for its copies is enough. The counted wait takes the
  // token rows to be the older eight, so nothing may move across the line
  // between the two.
  copy16(rx, s_r0[wave], 0);
  __builtin_amdgcn_sched_barrier(0);
  copy16(rw, s_r1[wave], 0);
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  uint4 xr[2][SEG];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int s = 0; s < SEG; ++s) xr[q][s] = *reinterpret_cast<const uint4*>(&s_r0[wave][i16][slot(q, s)]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if constexpr (NT > 1) {
    copy16(rw, s_r0[wave], 16);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  float sum8[NT][4];                              // segments 8 wave .. + 7: token 4 b + r, expert 16 n + i16
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    uint16_t (*const ws)[ROW] = n % 2 == 0 ? s_r1[wave] : s_r0[wave];
    uint4 wr[2][SEG];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int s = 0; s < SEG; ++s) wr[q][s] = *reinterpret_cast<const uint4*>(&ws[i16][slot(q, s)]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read before it is copied over
    if (n + 2 < NT) copy16(rw, ws, 16 * (n + 2));
    f32x16_t acc[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[q][v] = 0.0f;
#pragma unroll
    for (int j = 0; j < C; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint32_t v = word_of(xr[q][j >> 3], (j >> 1) & 3), u = word_of(wr[q][j >> 3], (j >> 1) & 3);
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x1f32(j & 1 ? hi_st<F16>(v) : lo_st<F16>(v),
                                                      j & 1 ? hi_st<F16>(u) : lo_st<F16>(u), acc[q], 0, 0, 0);
      }
    // Block 4q + b's sums are registers 4 b .. 4 b + 3: three tree levels.
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float s0 = (acc[0][r] + acc[0][4 + r]) + (acc[0][8 + r] + acc[0][12 + r]);
      const float s1 = (acc[1][r] + acc[1][4 + r]) + (acc[1][8 + r] + acc[1][12 + r]);
      sum8[n][r] = s0 + s1;
    }
    if (n + 2 < NT)
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (n + 1 < NT)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __syncthreads();  // every wave is done with its rows
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][4 * b + r][16 * n + i16] = sum8[n][r];
  __syncthreads();
  for (int q = tid; q < 16 * 64; q += 512) {
    const int t = q >> 6, e = q & 63;
    if (e < E) {
      const float lg = ((part[0][t][e] + part[1][t][e]) + (part[2][t][e] + part[3][t][e])) +
                       ((part[4][t][e] + part[5][t][e]) + (part[6][t][e] + part[7][t][e]));
      s_logit[t][e] = f2st<F16>(bias ? lg + bias[e] : lg);
    }
  }
  __syncthreads();  // every expert's logits of the block's tokens are in LDS
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (t0 + wave + 8 * k < T)  // wave-uniform
      rank_token<ROUTE, F16>(s_logit[wave + 8 * k], (int64_t)t0 + wave + 8 * k, E, K, idx, gates_f32, h);
  __syncthreads();
  if (tid <= E) hist[(int64_t)blockIdx.x * (E + 1) + tid] = h[tid];
}

int router_topk_tokens(int T) { return T <= 1024 ? 4 : 16; }

template <int C, int ROUTE, bool F16>
static void launch_router_topk_c(const uint16_t* x, const uint16_t* w, const float* bias, int T, int H, int E, int K,
                                 int32_t* idx, float* gates_f32, int32_t* hist, hipStream_t s) {
  const unsigned tb = (unsigned)router_topk_tokens(T), blocks = ((unsigned)T + tb - 1) / tb;
#define TFM_RT(kernel) tfm_launch(kernel, blocks, 512, 0, s, x, w, bias, T, H, E, K, idx, gates_f32, hist)
  if (tb == 4 && E <= 40) TFM_RT((router_topk4_kernel<C, ROUTE, F16, 5>));
  else if (tb == 4) TFM_RT((router_topk4_kernel<C, ROUTE, F16, 8>));
  else if (E <= 48) TFM_RT((router_topk16_kernel<C, ROUTE, F16, 3>));
  else TFM_RT((router_topk16_kernel<C, ROUTE, F16, 4>));
#undef TFM_RT
}

template <int C, bool F16>
static void launch_router_topk_r(int route_kind, const uint16_t* x, const uint16_t* w, const float* bias, int T, int H,
                                 int E, int K, int32_t* idx, float* gates_f32, int32_t* hist, hipStream_t s) {
  if (route_kind == TFM_ROUTE_OLMOE)
    launch_router_topk_c<C, TFM_ROUTE_OLMOE, F16>(x, w, bias, T, H, E, K, idx, gates_f32, hist, s);
  else
    launch_router_topk_c<C, TFM_ROUTE_GRANITE, F16>(x, w, bias, T, H, E, K, idx, gates_f32, hist, s);
}

template <bool F16>
static bool router_topk_dt(int route_kind, const uint16_t* x, const uint16_t* w, const float* bias,
                           int T, int H, int E, int K, int32_t* idx, float* gates_f32, int32_t* hist, hipStream_t s) {
  switch (H) {
    case 512: launch_router_topk_r<8, F16>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s); break;
    case 1024: launch_router_topk_r<16, F16>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s); break;
    case 1536: launch_router_topk_r<24, F16>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s); break;
    case 2048: launch_router_topk_r<32, F16>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s); break;
    default: return false;
  }
  return true;
}

bool launch_router_topk(int route_kind, bool f16, const uint16_t* x, const uint16_t* w, const float* bias,
                        int T, int H, int E, int K, int32_t* idx, float* gates_f32, int32_t* hist, hipStream_t s) {
  if (T <= 0) return true;
  const bool ok = f16 ? router_topk_dt<true>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s)
                      : router_topk_dt<false>(route_kind, x, w, bias, T, H, E, K, idx, gates_f32, hist, s);
  if (ok) check_hip(hipGetLastError(), "router_topk launch");
  return ok;
}

// Any H % 64 == 0: the same arithmetic with scalar loads.
template <bool F16>
__global__ __launch_bounds__(256) void router_logits_generic(const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ w,
                                                             const float* __restrict__ bias,
                                                             int T, int H, int E,
                                                             uint16_t* __restrict__ logits) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wave >= T * E) return;
  const int tok = wave / E, e = wave % E;
  const int c = H / 64;
  float s = 0.0f;
  for (int j = 0; j < c; ++j)
    s = __builtin_fmaf(st2f<F16>(x[(int64_t)tok * H + lane * c + j]), st2f<F16>(w[(int64_t)e * H + lane * c + j]), s);
  s = wave_tree_sum64(s);
  if (lane == 63) logits[(int64_t)tok * E + e] = f2st<F16>(bias ? s + bias[e] : s);
}

template <int C, bool F16>
static void launch_router_c(const uint16_t* x, const uint16_t* w, const float* bias, int T,
                            int H, int E, uint16_t* logits, hipStream_t s) {
  if (T <= 64) {
    // Few tokens: one wave per (token, expert), so the router rows stream in
    // parallel across the chip.
    const int waves = T * E;
    tfm_launch(router_logits_kernel<C, 1, F16>, (waves + 3) / 4, 256, 0, s, x, w, bias, T, H, E, 1, logits);
  } else {
    // Many tokens: a wave keeps 4 token rows in registers and walks EPW
    // experts, reading router rows from L2: as few experts per wave as keep
    // about 2048 waves (EPW 1 to 16, a power of two).
    constexpr int TW = 4;
    const int64_t tiles = (T + TW - 1) / TW;
    int EPW = 1;
    while (EPW < 16 && tiles * ((E + 2 * EPW - 1) / (2 * EPW)) >= 2048) EPW *= 2;
    const int waves = (int)(tiles * ((E + EPW - 1) / EPW));
    tfm_launch(router_logits_kernel<C, TW, F16>, (waves + 3) / 4, 256, 0, s, x, w, bias, T, H, E, EPW, logits);
  }
}

template <bool F16>
static void router_logits_dt(const uint16_t* x, const uint16_t* w, const float* bias, int T,
                             int H, int E, uint16_t* logits, hipStream_t s) {
  switch (H) {
    case 512: launch_router_c<8, F16>(x, w, bias, T, H, E, logits, s); break;
    case 1024: launch_router_c<16, F16>(x, w, bias, T, H, E, logits, s); break;
    case 1536: launch_router_c<24, F16>(x, w, bias, T, H, E, logits, s); break;
    case 2048: launch_router_c<32, F16>(x, w, bias, T, H, E, logits, s); break;
    default: {
      const int64_t waves = (int64_t)T * E;
      router_logits_generic<F16><<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(x, w, bias, T, H, E, logits);
    }
  }
}

void launch_router_logits(bool f16, const uint16_t* x, const uint16_t* w, const float* bias, int T,
                          int H, int E, uint16_t* logits, hipStream_t s) {
  if (T <= 0) return;
  if (f16)
    router_logits_dt<true>(x, w, bias, T, H, E, logits, s);
  else
    router_logits_dt<false>(x, w, bias, T, H, E, logits, s);
  check_hip(hipGetLastError(), "router_logits launch");
}

// Affine-quantised router (native_affine_qmm of the router weight,
// export_native_olmoe_target.py:194-200) dequantised once per call into a
// dense [E, H] matrix in the storage dtype: w[e,h] = st(fmaf(s, q, b)), the
// value native_affine_ops.py:29-36 rounds to the scales' dtype. The dense
// router kernels then compute the logits in their bit-defined order. One
// thread per packed word (8 or 4 codes); group size 64.
template <bool F16, int BITS>
__global__ __launch_bounds__(256) void dequant_router_kernel(const uint32_t* __restrict__ q,
                                                             const uint16_t* __restrict__ sc,
                                                             const uint16_t* __restrict__ bi,
                                                             int64_t words, uint16_t* __restrict__ w) {
  constexpr int PER = 32 / BITS;
  constexpr uint32_t MASK = (1u << BITS) - 1u;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= words) return;
  const int64_t k0 = i * PER;               // first element: row k0 / H, column k0 % H
  const int64_t g = k0 / 64;                // rows are whole groups (H % 64 == 0)
  const float s = st2f<F16>(sc[g]), b = st2f<F16>(bi[g]);
  const uint32_t word = q[i];
  uint16_t out[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j)
    out[j] = f2st<F16>(__builtin_fmaf(s, (float)((word >> (BITS * j)) & MASK), b));
  if constexpr (PER == 8) {
    uint4 v;
    v.x = out[0] | ((uint32_t)out[1] << 16);
    v.y = out[2] | ((uint32_t)out[3] << 16);
    v.z = out[4] | ((uint32_t)out[5] << 16);
    v.w = out[6] | ((uint32_t)out[7] << 16);
    *reinterpret_cast<uint4*>(w + k0) = v;
  } else {
    uint2 v;
    v.x = out[0] | ((uint32_t)out[1] << 16);
    v.y = out[2] | ((uint32_t)out[3] << 16);
    *reinterpret_cast<uint2*>(w + k0) = v;
  }
}

void launch_dequant_router(bool f16, int bits, const tfm_affine& r, int E, int H, uint16_t* w,
                           hipStream_t s) {
  const int64_t words = (int64_t)E * H * bits / 32;
  if (words <= 0) return;
  const unsigned blocks = (unsigned)((words + 255) / 256);
  const uint32_t* q = static_cast<const uint32_t*>(r.q);
  const uint16_t* sc = static_cast<const uint16_t*>(r.scales);
  const uint16_t* bi = static_cast<const uint16_t*>(r.biases);
  if (f16 && bits == 8)
    dequant_router_kernel<true, 8><<<blocks, 256, 0, s>>>(q, sc, bi, words, w);
  else if (f16)
    dequant_router_kernel<true, 4><<<blocks, 256, 0, s>>>(q, sc, bi, words, w);
  else if (bits == 8)
    dequant_router_kernel<false, 8><<<blocks, 256, 0, s>>>(q, sc, bi, words, w);
  else
    dequant_router_kernel<false, 4><<<blocks, 256, 0, s>>>(q, sc, bi, words, w);
  check_hip(hipGetLastError(), "router dequant launch");
}

__device__ __forceinline__ float readlane_f(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// One wave per token. gates_native: bf16 probabilities (OLMoE) or fp32
// (Granite); gates_f32: fp32 copy. Either may be null.
template <int ROUTE, bool F16>
__global__ __launch_bounds__(256) void topk_kernel(const uint16_t* __restrict__ logits, int T,
                                                   int E, int K, int32_t* __restrict__ idx,
                                                   void* __restrict__ gates_native,
                                                   float* __restrict__ gates_f32) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;  // whole wave exits together
  const uint16_t* row = logits + (int64_t)t * E;
  float g;
  int id;
  if (ROUTE == TFM_ROUTE_OLMOE) {
    uint16_t gb;
    id = olmoe_route_wave<F16>(row, E, K, &g, &gb);
    if (lane < K && gates_native) static_cast<uint16_t*>(gates_native)[(int64_t)t * K + lane] = gb;
  } else {
    id = granite_route_wave<F16>(row, E, K, &g);
    if (lane < K && gates_native) static_cast<float*>(gates_native)[(int64_t)t * K + lane] = g;
  }
  if (lane < K) {
    idx[(int64_t)t * K + lane] = id;
    if (gates_f32) gates_f32[(int64_t)t * K + lane] = g;
  }
}

// Top-k of kTopkTokensPerBlock tokens per workgroup (one wave per token at a
// time), plus the histogram of the workgroup's routes over the E experts for
// the grouping pass (its chunk is kTopkTokensPerBlock * K flat routes).
template <int ROUTE, bool F16>
__global__ __launch_bounds__(256) void topk_hist_kernel(const uint16_t* __restrict__ logits, int T,
                                                        int E, int K, int32_t* __restrict__ idx,
                                                        float* __restrict__ gates_f32,
                                                        int32_t* __restrict__ hist) {
  __shared__ int h[65];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (tid <= E) h[tid] = 0;
  __syncthreads();
  constexpr int kPerWave = kTopkTokensPerBlock / 4;
  for (int i = 0; i < kPerWave; ++i) {
    const int t = blockIdx.x * kTopkTokensPerBlock + wave * kPerWave + i;
    if (t >= T) break;  // wave-uniform
    const uint16_t* row = logits + (int64_t)t * E;
    float g;
    int id;
    if (ROUTE == TFM_ROUTE_OLMOE) {
      uint16_t gb;
      id = olmoe_route_wave<F16>(row, E, K, &g, &gb);
    } else {
      id = granite_route_wave<F16>(row, E, K, &g);
    }
    if (lane < K) {
      idx[(int64_t)t * K + lane] = id;
      gates_f32[(int64_t)t * K + lane] = g;
      atomicAdd(&h[id], 1);
    }
  }
  __syncthreads();
  if (tid <= E) hist[(int64_t)blockIdx.x * (E + 1) + tid] = h[tid];
}

template <bool F16>
static void topk_hist_dt(int route_kind, const uint16_t* logits, int T, int E, int K, int32_t* idx,
                         float* gates_f32, int32_t* hist, hipStream_t s) {
  const unsigned blocks = (unsigned)((T + kTopkTokensPerBlock - 1) / kTopkTokensPerBlock);
  if (route_kind == TFM_ROUTE_OLMOE)
    tfm_launch(topk_hist_kernel<TFM_ROUTE_OLMOE, F16>, blocks, 256, 0, s, logits, T, E, K, idx, gates_f32, hist);
  else
    tfm_launch(topk_hist_kernel<TFM_ROUTE_GRANITE, F16>, blocks, 256, 0, s, logits, T, E, K, idx, gates_f32, hist);
}

void launch_topk_hist(int route_kind, bool f16, const uint16_t* logits, int T, int E, int K, int32_t* idx,
                      float* gates_f32, int32_t* hist, hipStream_t s) {
  if (T <= 0) return;
  if (f16)
    topk_hist_dt<true>(route_kind, logits, T, E, K, idx, gates_f32, hist, s);
  else
    topk_hist_dt<false>(route_kind, logits, T, E, K, idx, gates_f32, hist, s);
  check_hip(hipGetLastError(), "topk_hist launch");
}

template <bool F16>
static void topk_dt(int route_kind, const uint16_t* logits, int T, int E, int K, int32_t* idx,
                    void* gates_native, float* gates_f32, hipStream_t s) {
  const unsigned blocks = (unsigned)((T + 3) / 4);
  if (route_kind == TFM_ROUTE_OLMOE)
    topk_kernel<TFM_ROUTE_OLMOE, F16><<<blocks, 256, 0, s>>>(logits, T, E, K, idx, gates_native, gates_f32);
  else
    topk_kernel<TFM_ROUTE_GRANITE, F16><<<blocks, 256, 0, s>>>(logits, T, E, K, idx, gates_native, gates_f32);
}

void launch_topk(int route_kind, bool f16, const uint16_t* logits, int T, int E, int K, int32_t* idx,
                 void* gates_native, float* gates_f32, hipStream_t s) {
  if (T <= 0) return;
  if (f16)
    topk_dt<true>(route_kind, logits, T, E, K, idx, gates_native, gates_f32, s);
  else
    topk_dt<false>(route_kind, logits, T, E, K, idx, gates_native, gates_f32, s);
  check_hip(hipGetLastError(), "topk launch");
}

// Ranking only (values given): one wave per row.
template <int RULE, bool F16>
__global__ __launch_bounds__(256) void rank_topk_kernel(const uint16_t* __restrict__ values, int T,
                                                        int n, int K, int32_t* __restrict__ idx) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;  // whole wave exits together
  const bool valid = lane < n;
  const float v = valid ? st2f<F16>(values[(int64_t)t * n + lane]) : 0.0f;
  const bool vn = v != v;
  int rank = 0;
  for (int j = 0; j < n; ++j) {
    const float o = readlane_f(v, j);
    const bool on = o != o;
    const bool equal = (on && vn) || (!on && !vn && o == v);
    const bool ahead = RULE == TFM_ROUTE_OLMOE ? (!on && (vn || o > v)) : (!on && (vn || o < v));
    rank += (ahead || (equal && j < lane)) ? 1 : 0;
  }
  if (!valid) return;
  if (RULE == TFM_ROUTE_OLMOE) {
    if (rank < K) idx[(int64_t)t * K + rank] = lane;
  } else {
    if (rank >= n - K) idx[(int64_t)t * K + rank - (n - K)] = lane;
  }
}

void launch_rank_topk(int rule, bool f16, const uint16_t* values, int T, int n, int K, int32_t* idx,
                      hipStream_t s) {
  if (T <= 0) return;
  const unsigned blocks = (unsigned)((T + 3) / 4);
  if (rule == TFM_ROUTE_OLMOE && f16)
    rank_topk_kernel<TFM_ROUTE_OLMOE, true><<<blocks, 256, 0, s>>>(values, T, n, K, idx);
  else if (rule == TFM_ROUTE_OLMOE)
    rank_topk_kernel<TFM_ROUTE_OLMOE, false><<<blocks, 256, 0, s>>>(values, T, n, K, idx);
  else if (f16)
    rank_topk_kernel<TFM_ROUTE_GRANITE, true><<<blocks, 256, 0, s>>>(values, T, n, K, idx);
  else
    rank_topk_kernel<TFM_ROUTE_GRANITE, false><<<blocks, 256, 0, s>>>(values, T, n, K, idx);
  check_hip(hipGetLastError(), "rank_topk launch");
}

template <bool F16>
__global__ __launch_bounds__(256) void olmoe_softmax_kernel(const uint16_t* __restrict__ logits,
                                                            int T, int E,
                                                            uint16_t* __restrict__ probs) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;  // whole wave exits together
  const bool valid = lane < E;
  const float ld = valid ? st2f<F16>(logits[(int64_t)t * E + lane]) : -__builtin_inff();
  float norm;
  const float ex = wave_softmax_exp(ld, &norm);
  if (valid) probs[(int64_t)t * E + lane] = f2st<F16>(softmax_prob(ex, norm));
}

void launch_olmoe_softmax(bool f16, const uint16_t* logits, int T, int E, uint16_t* probs, hipStream_t s) {
  if (T <= 0) return;
  if (f16)
    olmoe_softmax_kernel<true><<<(unsigned)((T + 3) / 4), 256, 0, s>>>(logits, T, E, probs);
  else
    olmoe_softmax_kernel<false><<<(unsigned)((T + 3) / 4), 256, 0, s>>>(logits, T, E, probs);
  check_hip(hipGetLastError(), "olmoe_softmax launch");
}

}  // namespace tfm
