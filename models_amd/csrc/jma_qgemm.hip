// Matrix-core products of GGUF block-quantized weights with prefill-sized activation batches
// (the projections around attention, llama/LlamaForwardPass.java:1043-1067, 1131-1138), gfx950.
//
// The arithmetic is the matrix-vector kernels' (jma_quant.hip): integer block dots, then per output
// the in-order float chain over the row's blocks, so every output has the same bits. The integer
// dots run on the f16 matrix ops: weight quants and int8 activations are exact in f16, and every
// partial sum is an integer below 2^24, exact in the f32 accumulators whatever the order.
#include <hip/hip_runtime.h>
#include <type_traits>

#include "jma_kernels.h"

namespace jma {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

#define JMA_INL __attribute__((always_inline))

// A value at any alignment (blocks are 2-byte aligned): one load, the hardware splits it.
template <typename T>
__device__ __forceinline__ T load_any(const void* p) {
  T v;
  __builtin_memcpy(&v, p, sizeof(T));
  return v;
}

// 16 bytes per lane from global memory straight into LDS (lane i's at lds + 16 i).
__device__ __forceinline__ void dma16(const void* base, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7FFFFFF0, 0x00020000),
      (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

// Bytes 0 and 2 (or 1 and 3) of x, unsigned, as two halves less `bias`: 0x6400 | u is 1024 + u.
template <int kBias>
__device__ __forceinline__ uint32_t bytes_to_half2(uint32_t x, uint32_t sel) {
  const half2_t off = {(_Float16)(-1024.0f - kBias), (_Float16)(-1024.0f - kBias)};
  const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, x, sel)) + off;
  return __builtin_bit_cast(uint32_t, v);
}
template <int kBias>
__device__ __forceinline__ half8_t bytes_to_half8(uint32_t x0, uint32_t x1) {
  u32x4_t r;
  r[0] = bytes_to_half2<kBias>(x0, 0x04020400u);
  r[1] = bytes_to_half2<kBias>(x0, 0x04030401u);
  r[2] = bytes_to_half2<kBias>(x1, 0x04020400u);
  r[3] = bytes_to_half2<kBias>(x1, 0x04030401u);
  return __builtin_bit_cast(half8_t, r);
}

// Bits 4 kHigh .. + 3 of bytes 0 and 2 of x as two halves less kBias (as (1024 + 16 n) / 16 for the
// high nibbles; every step exact).
template <int kHigh, int kBias>
__device__ __forceinline__ half2_t nibbles(uint32_t x) {
  if constexpr (kHigh) {
    const half2_t v = __builtin_bit_cast(half2_t, (x & 0x00F000F0u) | 0x64006400u);
    return v * half2_t{(_Float16)0.0625f, (_Float16)0.0625f} + half2_t{(_Float16)(-64 - kBias), (_Float16)(-64 - kBias)};
  } else {
    const half2_t v = __builtin_bit_cast(half2_t, (x & 0x000F000Fu) | 0x64006400u);
    return v + half2_t{(_Float16)(-1024 - kBias), (_Float16)(-1024 - kBias)};
  }
}
template <int kHigh>
__device__ __forceinline__ half8_t nibbles8(uint32_t x0, uint32_t x1) {
  half2_t r[4] = {nibbles<kHigh, 8>(x0), nibbles<kHigh, 8>(x0 >> 8), nibbles<kHigh, 8>(x1), nibbles<kHigh, 8>(x1 >> 8)};
  return __builtin_bit_cast(half8_t, r);
}

// Bits 0..3 of x moved to bit 4 of bytes 0..3.
__device__ __forceinline__ uint32_t fifth_bits(uint32_t x) { return ((x * 0x00204081u) & 0x01010101u) << 4; }

// Half h of a weight block as loaded (Q4_0, Q5_0, Q8_0: a 16-bit scale, then fifth bits, nibbles or
// bytes), and its two runs of 8 quants as halves: run(c) holds elements 16 c + 8 h ...
template <int FMT>
struct HalfBlock {
  uint2 q[FMT == 1 ? 2 : 1];
  uint32_t qh;
  uint16_t scale;
  __device__ __forceinline__ void load(const uint8_t* p, uint32_t h) {
    scale = load_any<uint16_t>(p);
    if constexpr (FMT == 5) qh = load_any<uint32_t>(p + 2) >> (8u * h);
    q[0] = load_any<uint2>(p + (FMT == 5 ? 6 : 2) + 8u * h);
    if constexpr (FMT == 1) q[1] = load_any<uint2>(p + 18 + 8u * h);
  }
  __device__ __forceinline__ half8_t run(int c) const {
    if constexpr (FMT == 0) {
      return c ? nibbles8<1>(q[0].x, q[0].y) : nibbles8<0>(q[0].x, q[0].y);
    } else if constexpr (FMT == 1) {  // int8: the sign bit flipped makes v + 128
      return bytes_to_half8<128>(q[c].x ^ 0x80808080u, q[c].y ^ 0x80808080u);
    } else {
      uint32_t x0 = (q[0].x >> (4 * c)) & 0x0F0F0F0Fu;
      uint32_t x1 = (q[0].y >> (4 * c)) & 0x0F0F0F0Fu;
      x0 |= fifth_bits((qh >> (16 * c)) & 15u);
      x1 |= fifth_bits((qh >> (16 * c + 4)) & 15u);
      return bytes_to_half8<16>(x0, x1);
    }
  }
};

// One lane's outputs of a 32 x 32 tile, rows b + 8 (e / 4) + e % 4 of the batch: the optional bias or
// residual (one float add, after the chain), then the store. A residual's loads go out together.
__device__ __forceinline__ void store_tile(const float16_t& acc, uint32_t b, uint32_t batch, uint32_t r,
                                           uint32_t rows, float* out, const float* addend, uint32_t mode) {
  auto at = [&](int e) JMA_INL { return (uint64_t)(b + 8u * (e / 4) + e % 4) * rows + r; };
  auto ok = [&](int e) JMA_INL { return b + 8u * (e / 4) + e % 4 < batch; };
  float add[16];
  if (mode == 2) {
#pragma unroll
    for (int e = 0; e < 16; ++e) add[e] = addend[ok(e) ? at(e) : 0];
  } else if (mode == 1) {
    const float bias = addend[r];
#pragma unroll
    for (int e = 0; e < 16; ++e) add[e] = bias;
  }
#pragma unroll
  for (int e = 0; e < 16; ++e)
    if (ok(e)) out[at(e)] = mode != 0 ? acc[e] + add[e] : acc[e];
}

// Barrier once at most N of this wave's loads are in flight and its LDS writes are done. N is counted
// from the source, so it holds only while the compiler emits at least that many loads a step:
// tests/test_product_waits_cpu.py plays the emitted loads and waits of every instance.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  static_assert(N >= 0 && N < 64, "the load counter has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int N, typename F, int I = 0>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, F, I + 1>(static_cast<F&&>(f));
  }
}

}  // namespace

// Products of Q4_0 (FMT 0), Q8_0 (1) and Q5_0 (5): out[b][r] = the chain over the 32-element
// blocks of fma(weightScale * activationScale, dot, sum).
//
// A step is one 32-element block of every row of the tile. Three steps ahead, the activations go
// straight to LDS (four buffers) and each thread's half weight block to registers; one step ahead
// the half block is unpacked to LDS (two buffers). One barrier a step. The loads of a step are
// counted (kLoads): the barrier waits for the ones issued before the last two steps' only.
//
// What bounds it: per 32 x 32 tile and step 96 cycles of matrix ops (two for the dot, one for the
// scale products, which on the vector unit would take 64 cycles more) and 64 of fma, plus the
// unpacking, on one SIMD; the two overlap only partly (counters: matrix unit busy 38% of the compute
// units' busy time, vector issue 50%, LDS 28%; waves wait for loads or barriers a quarter of their
// time). 5120 weight rows of 3072 inputs, 2048 activation rows, kernel trace: Q4_0 552 us with integer
// dots on the vector unit, 150 us with this kernel (429 TOPS); Q8_0 554 -> 157; Q5_0 171.
template <int FMT, int BT, int WT, int NB, int NW>
__global__ __launch_bounds__(64 * NB * NW, 2) void qgemm_kernel(const QMatArgs a, const _Float16* act,
                                                                 const uint16_t* act_scale,
                                                                 uint32_t tiles_w, uint32_t tiles_w_recip,
                                                                 uint32_t total) {
  constexpr QGemmShape kS{BT, WT, NB, NW};
  constexpr uint32_t kB = qgemm_rows_b(kS), kW = qgemm_rows_w(kS), kThreads = qgemm_threads(kS);
  constexpr uint32_t kBlockBytes = FMT == 0 ? 18u : FMT == 1 ? 34u : 22u;
  constexpr uint32_t kUnits = kW * 2;              // staged half blocks of a step
  constexpr uint32_t kWaves = NB * NW, kPieces = kB / 32 * 2;  // 1 KB pieces of activations
  constexpr uint32_t kPPW = (kPieces + kWaves - 1) / kWaves;   // ... a wave loads (some twice)
  static_assert(kUnits <= kThreads, "at most one staged half block per thread");
  constexpr int kLoads = (FMT == 0 ? 2 : 3) + BT + kPPW;  // a wave's loads per step
  __shared__ __attribute__((aligned(16))) _Float16 w0[kW * 32], w1[kW * 32];
  __shared__ __attribute__((aligned(16))) _Float16 a0[kB * 32], a1[kB * 32], a2[kB * 32], a3[kB * 32];
  __shared__ uint16_t c0[kW], c1[kW];

  const uint32_t K = a.blocks;
  uint32_t tx, ty;
  qgemm_tile(blockIdx.x, tiles_w, tiles_w_recip, total, tx, ty);
  uint32_t mi = 0;
  for (uint32_t i = 1; i < a.count; ++i) mi = tx >= a.m[i].tile0 ? i : mi;
  const uint32_t rows = a.m[mi].rows;
  const uint32_t r0 = (tx - a.m[mi].tile0) * kW, b0 = ty * kB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, j = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wb = wave / NW, ww = wave % NW;

  // This thread's staged half block: half su_h of a block of weight row su_row of the tile.
  const uint32_t su_row = tid % kUnits / 2u, su_h = tid & 1u;
  const uint8_t* const w_row = a.m[mi].w + (uint64_t)min(r0 + su_row, rows - 1u) * K * kBlockBytes;
  const uint32_t w_slot = (su_row / 32u) * 1024u + su_h * 256u + (su_row % 32u) * 8u;
  // Activation tiles of the workgroup (a ragged last one repeats a valid tile).
  const uint32_t btiles = qact_tiles(a.batch);
  const char* piece[kPPW];
#pragma unroll
  for (uint32_t i = 0; i < kPPW; ++i) {
    const uint32_t p = (wave + kWaves * i) % kPieces;
    piece[i] = (const char*)act + (uint64_t)min(b0 / 32u + p / 2u, btiles - 1u) * 64u * a.cols + p % 2u * 1024u;
  }
  const uint16_t* scale_at[BT];
#pragma unroll
  for (int i = 0; i < BT; ++i)
    scale_at[i] = act_scale + (uint64_t)min(b0 / 32u + wb * BT + i, btiles - 1u) * 32u * K + j;

  HalfBlock<FMT> wreg[4];
  uint32_t asc[4][BT];
  // Step k's loads (past the last block: that block again), into slot P = k mod 4.
  auto load = [&](uint32_t k, auto slot, _Float16* as) JMA_INL {
    constexpr int P = decltype(slot)::value;
    k = min(k, K - 1u);
    wreg[P].load(w_row + (uint64_t)k * kBlockBytes, su_h);
#pragma unroll
    for (int i = 0; i < BT; ++i) asc[P][i] = scale_at[i][k * 32u];
#pragma unroll
    for (uint32_t i = 0; i < kPPW; ++i)
      dma16(piece[i], as + (wave + kWaves * i) % kPieces * 512u, lane * 16u, k * 2048u);
  };
  auto put = [&](auto slot, _Float16* ws, uint16_t* cs) JMA_INL {
    constexpr int P = decltype(slot)::value;
    // (No branch: both threads of a row write its scale, and threads past the last half block
    // write one again. A branch here would end the block, and the compiler would sink the float
    // chains past it, holding every tile's matrix results in registers.)
#pragma unroll
    for (int c = 0; c < 2; ++c) *(half8_t*)(ws + w_slot + c * 512) = wreg[P].run(c);
    cs[su_row] = wreg[P].scale;
  };

  float16_t acc[BT][WT];
#pragma unroll
  for (int i = 0; i < BT; ++i)
#pragma unroll
    for (int t = 0; t < WT; ++t) acc[i][t] = float16_t{};
  const float16_t zero{};

  auto step = [&](uint32_t k, auto slot) JMA_INL {
    constexpr int P = decltype(slot)::value;
    _Float16* const ring[4] = {a0, a1, a2, a3};
    const _Float16* const as = ring[P];
    const _Float16* const ws = P % 2 ? w1 : w0;
    const uint16_t* const cs = P % 2 ? c1 : c0;
    load(k + 3, std::integral_constant<int, (P + 3) % 4>{}, ring[(P + 3) % 4]);
    half8_t av[BT][2], wv[WT][2], sav[BT], swv[WT];
    const bool scaled = h == 0 && k < K;  // a step past the last block adds 0 * dot
    // Scale operands: input 0 of the lanes h = 0 holds the scale, the rest are zeros, so the
    // matrix op forms the exact products weightScale * activationScale.
#pragma unroll
    for (int i = 0; i < BT; ++i) {
#pragma unroll
      for (int c = 0; c < 2; ++c) av[i][c] = *(const half8_t*)(as + (wb * BT + i) * 1024 + c * 512 + lane * 8);
      sav[i] = __builtin_bit_cast(half8_t, u32x4_t{scaled ? asc[P][i] : 0u, 0u, 0u, 0u});
    }
#pragma unroll
    for (int t = 0; t < WT; ++t) {
#pragma unroll
      for (int c = 0; c < 2; ++c) wv[t][c] = *(const half8_t*)(ws + (ww * WT + t) * 1024 + c * 512 + lane * 8);
      const uint32_t sc = cs[(ww * WT + t) * 32 + j];
      swv[t] = __builtin_bit_cast(half8_t, u32x4_t{scaled ? sc : 0u, 0u, 0u, 0u});
    }
    // Tile n's matrix ops, with the float chain of tile n - 1 between them.
    float16_t d[2], sc[2];
    static_for<BT * WT + 1>([&](auto idx) JMA_INL {
      constexpr int n = decltype(idx)::value;
      if constexpr (n < BT * WT) {
        constexpr int i = n / WT, t = n % WT;
        d[n % 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][0], wv[t][0], zero, 0, 0, 0);
        sc[n % 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sav[i], swv[t], zero, 0, 0, 0);
        d[n % 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][1], wv[t][1], d[n % 2], 0, 0, 0);
      }
      if constexpr (n > 0) {
        constexpr int m = n - 1;
        float16_t& c = acc[m / WT][m % WT];
#pragma unroll
        for (int e = 0; e < 16; ++e) c[e] = __builtin_fmaf(sc[m % 2][e], d[m % 2][e], c[e]);
      }
    });
    put(std::integral_constant<int, (P + 1) % 4>{}, P % 2 ? w0 : w1, P % 2 ? c0 : c1);
    // Order: the operand reads, the first tile's matrix ops, then a share of the vector work after
    // every further matrix op.
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * BT + 3 * WT, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
    static_for<3 * (BT * WT - 1)>([&](auto) JMA_INL {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
    });
    wait_barrier<2 * kLoads>();  // step k + 1's activations have arrived
    __builtin_amdgcn_sched_barrier(0);
  };

  load(0, std::integral_constant<int, 0>{}, a0);
  load(1, std::integral_constant<int, 1>{}, a1);
  load(2, std::integral_constant<int, 2>{}, a2);
  put(std::integral_constant<int, 0>{}, w0, c0);
  wait_barrier<2 * kLoads>();
  for (uint32_t k = 0; k < K; k += 4)
    static_for<4>([&](auto p) JMA_INL { step(k + decltype(p)::value, p); });
  // No load into this workgroup's LDS may outlive it.
  __builtin_amdgcn_s_waitcnt((0 & 15) | (7 << 4) | (15 << 8));

  float* const out = a.m[mi].out;
  const float* const addend = a.m[mi].addend;
#pragma unroll
  for (int t = 0; t < WT; ++t) {
    const uint32_t r = r0 + (ww * WT + t) * 32u + j;
    if (r >= rows) continue;
#pragma unroll
    for (int i = 0; i < BT; ++i)
      store_tile(acc[i][t], b0 + (wb * BT + i) * 32u + 4u * h, a.batch, r, rows, out, addend, a.addend_mode);
  }
}

// ---------------------------------------------------------------- K-quants

// One lane per activation row group of 64: 4 bytes each from global memory straight into LDS.
__device__ __forceinline__ void dma4(const void* base, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7FFFFFF0, 0x00020000),
      (__attribute__((address_space(3))) void*)lds, 4, voff, soff, 0, 0);
}

// Products of Q4_K (FMT 2) and Q5_K (4) weights on Q8_K activations, in the float order of
// dot_q4_k_q8_k_row_scalar / dot_q5_k_q8_k_row_scalar (backend-native/src/main/rust/model-kernels/
// src/lib.rs:3410-3518): per 256-element block qsum = sum over the eight 32-element groups of
// scale_g * dot_g and msum = sum of min_g * (the group's two 16-element activation sums), then
// sum = fma(d * as, qsum, sum) and sum = fma(-(dmin * as), msum, sum).
//
// A weight is staged as the half scale_g * (quant - C), C = 8 or 16, so the matrix ops accumulate
// qsum - C * ssum, with ssum = sum of scale_g * (the group's sums): an integer of at most
// 256 * 63 * 8 * 127 < 2^24 (Q5_K: per 128 elements), exact in f32; ssum and msum are one matrix
// op each (16 inputs: the block's sums). qsum = fma(C, ssum, .) then rounds once, as the integer's
// conversion does; Q5_K adds its two parts as integers.
//
// Measured (5120 weight rows of 3072 inputs, 2048 activation rows, kernel trace): Q4_K 508 us with
// integer dots on the vector unit, 118 us (547 TOPS) here; Q5_K 166 us. Per step of a 128 x 128 tile 256
// cycles of matrix ops on each SIMD beside 256 of operand reads from LDS; by counters neither fills the
// time (Q4_K: matrix unit busy 36% of the compute units' busy time, vector issue 48%, LDS 38%, a
// quarter of that bank conflicts; Q5_K, with 1.6 times the LDS accesses and 2.3 times the vector work per
// matrix op in its smaller tile: 21, 63 and 38%).
//
// Steps, buffers and loads as qgemm_kernel's, a step one 32-element group; the 4-bit quants of a
// pair of groups are loaded once, the block's header one block ahead.
template <int FMT, int BT, int WT, int NB, int NW>
__global__ __launch_bounds__(64 * NB * NW, 2) void qkgemm_kernel(
    const QMatArgs a, const _Float16* act, const _Float16* sums, const float* scales, uint32_t tiles_w,
    uint32_t tiles_w_recip, uint32_t total) {
  constexpr QGemmShape kS{BT, WT, NB, NW};
  constexpr uint32_t kB = qgemm_rows_b(kS), kW = qgemm_rows_w(kS), kThreads = qgemm_threads(kS);
  constexpr uint32_t kBlockBytes = FMT == 2 ? 144u : 176u;
  constexpr int kBias = FMT == 2 ? 8 : 16;
  constexpr uint32_t kUnits = kW * 2, kWaves = NB * NW, kPieces = kB / 32 * 2;
  constexpr uint32_t kPPW = (kPieces + kWaves - 1) / kWaves;
  constexpr uint32_t kScales = (kB + 63) / 64;  // 64-row pieces of activation scales
  static_assert(kUnits <= kThreads, "at most one staged half block per thread");
  // A wave's loads in step g of a block. The barrier that closes a step leaves that step's and the one
  // before's in flight, so what a step loads is there three steps later: step 4's scales in step 7.
  constexpr int kScaleStep = 4;
  static_assert(kScaleStep + 3 <= 7, "the last step reads the block's activation scales");
  constexpr auto loads = [](int g) {
    return (int)kPPW + (g % 2 == 0 ? 2 : 0) + (g == 3 ? (FMT == 4 ? 3 : 1) : 0) + (g == 4 ? BT : 0) +
           (g == kScaleStep ? (int)kScales : 0);
  };
  __shared__ __attribute__((aligned(16))) _Float16 w0[kW * 32], w1[kW * 32];
  __shared__ __attribute__((aligned(16))) _Float16 a0[kB * 32], a1[kB * 32], a2[kB * 32], a3[kB * 32];
  __shared__ __attribute__((aligned(16))) _Float16 s_sc[kW * 16], s_mn[kW * 16];
  __shared__ __attribute__((aligned(16))) float s_as[kScales * 64];
  __shared__ float s_d[kW], s_dm[kW];

  const uint32_t KB = a.blocks;
  uint32_t tx, ty;
  qgemm_tile(blockIdx.x, tiles_w, tiles_w_recip, total, tx, ty);
  uint32_t mi = 0;
  for (uint32_t i = 1; i < a.count; ++i) mi = tx >= a.m[i].tile0 ? i : mi;
  const uint32_t rows = a.m[mi].rows;
  const uint32_t r0 = (tx - a.m[mi].tile0) * kW, b0 = ty * kB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, j = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wb = wave / NW, ww = wave % NW;

  const uint32_t su_row = tid % kUnits / 2u, su_h = tid & 1u;
  const uint8_t* const w_row = a.m[mi].w + (uint64_t)min(r0 + su_row, rows - 1u) * KB * kBlockBytes;
  const uint32_t w_slot = (su_row / 32u) * 1024u + su_h * 256u + (su_row % 32u) * 8u;
  const uint32_t s_slot = (su_row / 32u) * 512u + su_h * 256u + (su_row % 32u) * 8u;
  const uint32_t btiles = qact_tiles(a.batch);
  const char* piece[kPPW];
#pragma unroll
  for (uint32_t i = 0; i < kPPW; ++i) {
    const uint32_t p = (wave + kWaves * i) % kPieces;
    piece[i] = (const char*)act + (uint64_t)min(b0 / 32u + p / 2u, btiles - 1u) * 64u * a.cols + p % 2u * 1024u;
  }
  const _Float16* sums_at[BT];
#pragma unroll
  for (int i = 0; i < BT; ++i)
    sums_at[i] = sums + (uint64_t)min(b0 / 32u + wb * BT + i, btiles - 1u) * 512u * KB + lane * 8u;
  uint32_t scale_off[kScales];
#pragma unroll
  for (uint32_t i = 0; i < kScales; ++i)
    scale_off[i] = (min(b0 / 32u + 2u * i + h, btiles - 1u) * KB * 32u + j) * 4u;

  uint2 wq[4][2];   // quant bytes 8 h .. and 16 + 8 h .. of pairs of groups, by pair mod 4
  u32x4_t hdr;      // the next block's d, dmin and packed scales and mins
  uint2 qhn[2];     // its fifth bits (bytes as wq)
  uint32_t sc_w[2], mn_w[2], dd;  // the staged block's scales and mins as bytes, d and dmin
  uint32_t qh[4];
  auto block_at = [&](uint32_t kb) JMA_INL { return w_row + (uint64_t)min(kb, KB - 1u) * kBlockBytes; };
  auto load_pair = [&](uint32_t kb, auto pair) JMA_INL {
    constexpr int p = decltype(pair)::value;
    const uint8_t* q = block_at(kb) + (FMT == 4 ? 48 : 16) + 32 * p + 8u * su_h;
    wq[p][0] = load_any<uint2>(q);
    wq[p][1] = load_any<uint2>(q + 16);
  };
  auto load_header = [&](uint32_t kb) JMA_INL {
    const uint8_t* q = block_at(kb);
    hdr = load_any<u32x4_t>(q);
    if constexpr (FMT == 4) {
      qhn[0] = load_any<uint2>(q + 16 + 8u * su_h);
      qhn[1] = load_any<uint2>(q + 32 + 8u * su_h);
    }
  };
  auto take_header = [&]() JMA_INL {
    dd = hdr[0];
    sc_w[0] = hdr[1] & 0x3F3F3F3Fu;
    mn_w[0] = hdr[2] & 0x3F3F3F3Fu;
    sc_w[1] = (hdr[3] & 0x0F0F0F0Fu) | ((hdr[1] >> 2) & 0x30303030u);
    mn_w[1] = ((hdr[3] >> 4) & 0x0F0F0F0Fu) | ((hdr[2] >> 2) & 0x30303030u);
    if constexpr (FMT == 4) qh[0] = qhn[0].x, qh[1] = qhn[0].y, qh[2] = qhn[1].x, qh[3] = qhn[1].y;
  };
  // Step (kb, g)'s activations (past the last block: that block's again).
  auto load_a = [&](uint32_t kb, int g, _Float16* as) JMA_INL {
#pragma unroll
    for (uint32_t i = 0; i < kPPW; ++i)
      dma16(piece[i], as + (wave + kWaves * i) % kPieces * 512u, lane * 16u,
            (min(kb, KB - 1u) * 8u + (uint32_t)g) * 2048u);
  };
  // Group g of the staged block as scale * (quant - kBias).
  auto put = [&](auto group, _Float16* ws) JMA_INL {
    constexpr int g = decltype(group)::value, p = g / 2;
    const half2_t s = __builtin_bit_cast(half2_t, bytes_to_half2<0>(sc_w[g / 4], 0x04000400u + 0x00010001u * (g % 4)));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      half2_t r[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // halves (0, 2), (1, 3) of word e / 2
        const uint32_t x = (e / 2 ? wq[p][c].y : wq[p][c].x) >> (8 * (e % 2));
        if constexpr (FMT == 2) {
          r[e] = nibbles<g % 2, 8>(x) * s;
        } else {
          const uint32_t five = (qh[2 * c + e / 2] >> (8 * (e % 2) + g)) & 0x00010001u;
          const uint32_t n = g % 2 ? (x >> 4) & 0x000F000Fu : x & 0x000F000Fu;
          const half2_t v = __builtin_bit_cast(half2_t, n | (five << 4) | 0x64006400u);
          r[e] = (v + half2_t{(_Float16)-1040.0f, (_Float16)-1040.0f}) * s;
        }
      }
      *(half8_t*)(ws + w_slot + c * 512) = __builtin_bit_cast(half8_t, r);
    }
  };
  // The block's scale and min operands (inputs 2 g and 2 g + 1: group g) and its d and dmin.
  auto put_block = [&]() JMA_INL {
    auto operand = [&](uint32_t x) JMA_INL {
      u32x4_t r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = bytes_to_half2<0>(x, 0x04000400u + 0x00010001u * i);
      return __builtin_bit_cast(half8_t, r);
    };
    *(half8_t*)(s_sc + s_slot) = operand(su_h ? sc_w[1] : sc_w[0]);
    *(half8_t*)(s_mn + s_slot) = operand(su_h ? mn_w[1] : mn_w[0]);
    const half2_t d = __builtin_bit_cast(half2_t, dd);
    s_d[su_row] = (float)d[0];
    s_dm[su_row] = (float)d[1];
  };

  float16_t acc[BT][WT], dot[BT][WT];
  int32_t part[FMT == 4 ? BT : 1][FMT == 4 ? WT : 1][16];
  half8_t sum_op[BT];
#pragma unroll
  for (int i = 0; i < BT; ++i)
#pragma unroll
    for (int t = 0; t < WT; ++t) acc[i][t] = float16_t{};
  const float16_t zero{};

  auto step = [&](uint32_t kb, auto group) JMA_INL {
    constexpr int g = decltype(group)::value;
    _Float16* const ring[4] = {a0, a1, a2, a3};
    const _Float16* const as = ring[g % 4];
    const _Float16* const ws = g % 2 ? w1 : w0;
    load_a(g < 5 ? kb : kb + 1, (g + 3) % 8, ring[(g + 3) % 4]);
    if constexpr (g % 2 == 0) load_pair(g < 4 ? kb : kb + 1, std::integral_constant<int, (g / 2 + 2) % 4>{});
    if constexpr (g == 3) load_header(kb + 1);
    if constexpr (g == 4) {
#pragma unroll
      for (int i = 0; i < BT; ++i) sum_op[i] = *(const half8_t*)(sums_at[i] + (uint64_t)kb * 512u);
    }
    if constexpr (g == kScaleStep) {
#pragma unroll
      for (uint32_t i = 0; i < kScales; ++i) dma4(scales, s_as + 64 * i, scale_off[i], kb * 128u);
    }
    half8_t av[BT][2], wv[WT][2];
#pragma unroll
    for (int i = 0; i < BT; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c) av[i][c] = *(const half8_t*)(as + (wb * BT + i) * 1024 + c * 512 + lane * 8);
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c) wv[t][c] = *(const half8_t*)(ws + (ww * WT + t) * 1024 + c * 512 + lane * 8);
    constexpr bool first = g == 0 || (FMT == 4 && g == 4);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < BT; ++i)
#pragma unroll
        for (int t = 0; t < WT; ++t)
          dot[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][c], wv[t][c], first && c == 0 ? zero : dot[i][t], 0, 0, 0);
    if constexpr (g == 7) take_header();
    put(std::integral_constant<int, (g + 1) % 8>{}, g % 2 ? w0 : w1);
    if constexpr (g == 0) put_block();
    if constexpr (FMT == 4 && g == 3) {
#pragma unroll
      for (int i = 0; i < BT; ++i)
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) part[i][t][e] = (int32_t)dot[i][t][e];
    }
    if constexpr (g == 7) {
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        const uint32_t wt = ww * WT + t;
        const half8_t sc_op = *(const half8_t*)(s_sc + wt * 512 + lane * 8);
        const half8_t mn_op = *(const half8_t*)(s_mn + wt * 512 + lane * 8);
        const float wd = s_d[wt * 32 + j], wdm = s_dm[wt * 32 + j];
#pragma unroll
        for (int i = 0; i < BT; ++i) {
          const float16_t ss = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_op[i], sc_op, zero, 0, 0, 0);
          const float16_t ms = __builtin_amdgcn_mfma_f32_32x32x16_f16(sum_op[i], mn_op, zero, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float as_b = s_as[(wb * BT + i) * 32 + 8 * (e / 4) + 4 * h + e % 4];
            float qsum;
            if constexpr (FMT == 2) qsum = __builtin_fmaf((float)kBias, ss[e], dot[i][t][e]);
            else qsum = (float)((int32_t)dot[i][t][e] + part[i][t][e] + kBias * (int32_t)ss[e]);
            float d, dm;
            {
#pragma clang fp contract(off)
              d = wd * as_b;
              dm = wdm * as_b;
            }
            acc[i][t][e] = __builtin_fmaf(-dm, ms[e], __builtin_fmaf(d, qsum, acc[i][t][e]));
          }
        }
      }
    }
    wait_barrier<loads(g) + loads((g + 7) % 8)>();  // the next step's activations have arrived
    __builtin_amdgcn_sched_barrier(0);
  };

  load_header(0);
  load_pair(0, std::integral_constant<int, 0>{});
  load_pair(0, std::integral_constant<int, 1>{});
  load_a(0, 0, a0);
  load_a(0, 1, a1);
  load_a(0, 2, a2);
  take_header();
  put(std::integral_constant<int, 0>{}, w0);
  wait_barrier<0>();
  for (uint32_t kb = 0; kb < KB; ++kb) static_for<8>([&](auto g) JMA_INL { step(kb, g); });
  // No load into this workgroup's LDS may outlive it.
  __builtin_amdgcn_s_waitcnt((0 & 15) | (7 << 4) | (15 << 8));

  float* const out = a.m[mi].out;
  const float* const addend = a.m[mi].addend;
#pragma unroll
  for (int t = 0; t < WT; ++t) {
    const uint32_t r = r0 + (ww * WT + t) * 32u + j;
    if (r >= rows) continue;
#pragma unroll
    for (int i = 0; i < BT; ++i)
      store_tile(acc[i][t], b0 + (wb * BT + i) * 32u + 4u * h, a.batch, r, rows, out, addend, a.addend_mode);
  }
}

// Products of Q6_K weights on Q8_K activations, in the float order of dot_q6_k_q8_k_row_scalar
// (RS:3519-3577): per 256-element block eight integer class sums (class l: the elements whose index
// within their 32-element run is l + 8 m), then lane_l = fma(d * as, isum_l, lane_l); after the
// last block the eight lanes are added in order to 0.
//
// scale * quant takes 13 bits, so a weight is two halves, scale * (quant & ~1) (even, at most 4096)
// and scale * (quant & 1), both exact, each with matrix ops of its own into one accumulator: an
// integer of at most 32 * 4096 * 127 < 2^24. A step is one class of a block (32 elements of every
// row); the activations come in class order (qact_class_index). Eight waves of one 32 x 32 tile,
// each output with its eight chains; otherwise the steps, buffers and loads of qgemm_kernel. The
// call of qkgemm_kernel's note with Q6_K weights: 917 us on the vector unit, 234 us here: splitting the
// weights and 16 fma per tile and class beside 4 matrix ops a class, with waits between (counters:
// matrix unit 25% of the busy time, vector issue 38%, LDS 45%, two fifths of that bank conflicts).
__global__ __launch_bounds__(64 * kQ6KShape.nb * kQ6KShape.nw, 2) void q6gemm_kernel(
    const QMatArgs a, const _Float16* act, const float* scales, uint32_t tiles_w, uint32_t tiles_w_recip,
    uint32_t total) {
  constexpr QGemmShape kS = kQ6KShape;
  constexpr uint32_t NW = kS.nw;
  constexpr uint32_t kB = qgemm_rows_b(kS), kW = qgemm_rows_w(kS), kThreads = qgemm_threads(kS);
  constexpr uint32_t kBlockBytes = 210u, kWaves = kS.nb * kS.nw, kScales = kB / 64;
  static_assert(kThreads == kW * 8 && kB / 32 * 2 == kWaves, "a staged part per thread, an activation piece per wave");
  constexpr auto loads = [](int l) { return 1 + (l == 1 ? 4 : 0) + (l == 5 ? (int)kScales : 0); };
  __shared__ __attribute__((aligned(16))) _Float16 w0[kW * 64], w1[kW * 64];
  __shared__ __attribute__((aligned(16))) _Float16 a0[kB * 32], a1[kB * 32], a2[kB * 32], a3[kB * 32];
  __shared__ __attribute__((aligned(16))) float s_as[kB];
  __shared__ float s_d[kW];

  const uint32_t KB = a.blocks;
  uint32_t tx, ty;
  qgemm_tile(blockIdx.x, tiles_w, tiles_w_recip, total, tx, ty);
  uint32_t mi = 0;
  for (uint32_t i = 1; i < a.count; ++i) mi = tx >= a.m[i].tile0 ? i : mi;
  const uint32_t rows = a.m[mi].rows;
  const uint32_t r0 = (tx - a.m[mi].tile0) * kW, b0 = ty * kB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, j = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wb = wave / NW, ww = wave % NW;

  // This thread's staged part: the 16 elements s of runs rr and rr + 2 of 128-element half hf.
  const uint32_t su_row = tid / 8u, hf = tid >> 2 & 1u, rr = tid >> 1 & 1u, s = tid & 1u;
  const uint8_t* const w_row = a.m[mi].w + (uint64_t)min(r0 + su_row, rows - 1u) * KB * kBlockBytes;
  const uint32_t w_slot = (su_row / 32u) * 2048u + hf * 512u + rr * 256u + (su_row % 32u) * 8u + s * 4u;
  const uint32_t btiles = qact_tiles(a.batch);
  const char* const piece = (const char*)act + (uint64_t)min(b0 / 32u + wave / 2u, btiles - 1u) * 64u * a.cols +
                            wave % 2u * 1024u;
  uint32_t scale_off[kScales];
#pragma unroll
  for (uint32_t i = 0; i < kScales; ++i)
    scale_off[i] = (min(b0 / 32u + 2u * i + h, btiles - 1u) * KB * 32u + j) * 4u;

  u32x4_t ql, qh, qln, qhn;  // the staged block's low nibbles and (shifted to bit 0) high bits; the next's
  uint2 scn;
  uint16_t dn;
  half2_t sc[2];  // scales of runs rr and rr + 2
  uint16_t d16;
  auto load_w = [&](uint32_t kb) JMA_INL {
    const uint8_t* q = w_row + (uint64_t)min(kb, KB - 1u) * kBlockBytes;
    qln = load_any<u32x4_t>(q + 64u * hf + 32u * rr + 16u * s);
    qhn = load_any<u32x4_t>(q + 128u + 32u * hf + 16u * s);
    scn = load_any<uint2>(q + 192u + 8u * hf);
    dn = load_any<uint16_t>(q + 208u);
  };
  auto take_w = [&]() JMA_INL {
    ql = qln;
    qh = qhn >> (2u * rr);
    const uint32_t shift = 8u * (2u * rr + s);
    const _Float16 s0 = (_Float16)(short)(int8_t)(scn.x >> shift), s1 = (_Float16)(short)(int8_t)(scn.y >> shift);
    sc[0] = half2_t{s0, s0};
    sc[1] = half2_t{s1, s1};
    d16 = dn;
  };
  auto load_a = [&](uint32_t kb, int l, _Float16* as) JMA_INL {
    dma16(piece, as + wave * 512u, lane * 16u, (min(kb, KB - 1u) * 8u + (uint32_t)l) * 2048u);
  };
  // Class l of the staged block: elements l and l + 8 of this part, runs rr and rr + 2.
  auto put = [&](auto cls, _Float16* ws) JMA_INL {
    constexpr int l = decltype(cls)::value, y = l / 4, b = l % 4;
    constexpr uint32_t sel = 0x0C000C04u + 0x00010001u * b;  // bytes b of both words, zero-extended
    const uint32_t lo = __builtin_amdgcn_perm(ql[y], ql[y + 2], sel), hi = __builtin_amdgcn_perm(qh[y], qh[y + 2], sel);
    const uint32_t v[2] = {(lo & 0x000F000Fu) | ((hi & 0x00030003u) << 4), ((lo >> 4) & 0x000F000Fu) | (hi & 0x00300030u)};
    uint2 even, odd;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const half2_t e = __builtin_bit_cast(half2_t, (v[i] & 0x003E003Eu) | 0x64006400u);
      (i ? even.y : even.x) = __builtin_bit_cast(uint32_t, (e + half2_t{(_Float16)-1056.0f, (_Float16)-1056.0f}) * sc[i]);
      typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
      const u16x2_t o = __builtin_bit_cast(u16x2_t, v[i] & 0x00010001u) * __builtin_bit_cast(u16x2_t, sc[i]);
      (i ? odd.y : odd.x) = __builtin_bit_cast(uint32_t, o);  // the scale's bits or 0
    }
    *(uint2*)(ws + w_slot) = even;
    *(uint2*)(ws + w_slot + 1024) = odd;
  };

  float16_t acc[8];
  float16_t dd;
#pragma unroll
  for (int l = 0; l < 8; ++l) acc[l] = float16_t{};
  const float16_t zero{};
  auto step = [&](uint32_t kb, auto cls) JMA_INL {
    constexpr int l = decltype(cls)::value;
    _Float16* const ring[4] = {a0, a1, a2, a3};
    const _Float16* const as = ring[l % 4];
    const _Float16* const ws = l % 2 ? w1 : w0;
    load_a(l < 5 ? kb : kb + 1, (l + 3) % 8, ring[(l + 3) % 4]);
    if constexpr (l == 1) load_w(kb + 1);
    if constexpr (l == 5) {
#pragma unroll
      for (uint32_t i = 0; i < kScales; ++i) dma4(scales, s_as + 64 * i, scale_off[i], min(kb + 1, KB - 1u) * 128u);
    }
    half8_t av[2], we[2], wo[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      av[c] = *(const half8_t*)(as + wb * 1024 + c * 512 + lane * 8);
      we[c] = *(const half8_t*)(ws + ww * 2048 + c * 512 + lane * 8);
      wo[c] = *(const half8_t*)(ws + ww * 2048 + 1024 + c * 512 + lane * 8);
    }
    if constexpr (l == 0) {
      const float wd = s_d[ww * 32 + j];
#pragma unroll
      for (int e = 0; e < 16; ++e) dd[e] = wd * s_as[wb * 32 + 8 * (e / 4) + 4 * h + e % 4];
    }
    float16_t dot = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[0], we[0], zero, 0, 0, 0);
    dot = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[0], wo[0], dot, 0, 0, 0);
    dot = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[1], we[1], dot, 0, 0, 0);
    dot = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[1], wo[1], dot, 0, 0, 0);
    if constexpr (l == 7) take_w();
    put(std::integral_constant<int, (l + 1) % 8>{}, l % 2 ? w0 : w1);
    if constexpr (l == 7) s_d[su_row] = (float)__builtin_bit_cast(_Float16, d16);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[l][e] = __builtin_fmaf(dd[e], dot[e], acc[l][e]);
    wait_barrier<loads(l) + loads((l + 7) % 8)>();  // the next step's activations have arrived
    __builtin_amdgcn_sched_barrier(0);
  };

  load_w(0);
#pragma unroll
  for (uint32_t i = 0; i < kScales; ++i) dma4(scales, s_as + 64 * i, scale_off[i], 0u);
  load_a(0, 0, a0);
  load_a(0, 1, a1);
  load_a(0, 2, a2);
  take_w();
  put(std::integral_constant<int, 0>{}, w0);
  s_d[su_row] = (float)__builtin_bit_cast(_Float16, d16);
  wait_barrier<0>();
  for (uint32_t kb = 0; kb < KB; ++kb) static_for<8>([&](auto l) JMA_INL { step(kb, l); });
  // No load into this workgroup's LDS may outlive it.
  __builtin_amdgcn_s_waitcnt((0 & 15) | (7 << 4) | (15 << 8));

  const uint32_t r = r0 + ww * 32u + j;
  if (r >= rows) return;
  float16_t sum{};
#pragma unroll
  for (int l = 0; l < 8; ++l) sum += acc[l];
  store_tile(sum, b0 + wb * 32u + 4u * h, a.batch, r, rows, a.m[mi].out, a.m[mi].addend, a.addend_mode);
}

namespace {
template <int FMT, uint32_t kBt, uint32_t kWt, uint32_t kNb, uint32_t kNw>
void launch_tile(const QMatArgs& a, uint32_t tiles_w, const void* act, const void* sums, const void* scales,
                 hipStream_t stream) {
  constexpr QGemmShape s{kBt, kWt, kNb, kNw};
  const uint32_t total = tiles_w * ((a.batch + qgemm_rows_b(s) - 1) / qgemm_rows_b(s));
  if constexpr (FMT == 2 || FMT == 4)
    hipLaunchKernelGGL((qkgemm_kernel<FMT, kBt, kWt, kNb, kNw>), dim3(total), dim3(qgemm_threads(s)), 0, stream, a,
                       (const _Float16*)act, (const _Float16*)sums, (const float*)scales, tiles_w,
                       qgemm_recip(tiles_w), total);
  else
    hipLaunchKernelGGL((qgemm_kernel<FMT, kBt, kWt, kNb, kNw>), dim3(total), dim3(qgemm_threads(s)), 0, stream, a,
                       (const _Float16*)act, (const uint16_t*)scales, tiles_w, qgemm_recip(tiles_w), total);
}
template <int FMT>
hipError_t launch_fmt(const QMatArgs& a, uint32_t shape, uint32_t tiles_w, const void* act, const void* sums,
                      const void* scales, hipStream_t stream) {
  constexpr QGemmShape large = FMT == 4 ? kQ5KLargeShape : kQGemmShape[0];
  constexpr QGemmShape s1 = kQGemmShape[1], s2 = kQGemmShape[2];
  switch (shape) {
    case 0: launch_tile<FMT, large.bt, large.wt, large.nb, large.nw>(a, tiles_w, act, sums, scales, stream); break;
    case 1: launch_tile<FMT, s1.bt, s1.wt, s1.nb, s1.nw>(a, tiles_w, act, sums, scales, stream); break;
    case 2: launch_tile<FMT, s2.bt, s2.wt, s2.nb, s2.nw>(a, tiles_w, act, sums, scales, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_qgemm(const QMatArgs& a, uint32_t fmt, uint32_t shape, uint32_t tiles_w,
                        const void* act, const void* act_scale, hipStream_t stream) {
  if (fmt == 0) return launch_fmt<0>(a, shape, tiles_w, act, nullptr, act_scale, stream);
  if (fmt == 1) return launch_fmt<1>(a, shape, tiles_w, act, nullptr, act_scale, stream);
  if (fmt == 5) return launch_fmt<5>(a, shape, tiles_w, act, nullptr, act_scale, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_qkgemm(const QMatArgs& a, uint32_t fmt, uint32_t shape, uint32_t tiles_w,
                         const void* act, const void* sums, const void* scales, hipStream_t stream) {
  if (fmt == 2) return launch_fmt<2>(a, shape, tiles_w, act, sums, scales, stream);
  if (fmt == 4) return launch_fmt<4>(a, shape, tiles_w, act, sums, scales, stream);
  if (fmt != 3) return hipErrorInvalidValue;
  const uint32_t total = tiles_w * ((a.batch + qgemm_rows_b(kQ6KShape) - 1) / qgemm_rows_b(kQ6KShape));
  hipLaunchKernelGGL(q6gemm_kernel, dim3(total), dim3(qgemm_threads(kQ6KShape)), 0, stream, a,
                     (const _Float16*)act, (const float*)scales, tiles_w, qgemm_recip(tiles_w), total);
  return hipGetLastError();
}

}  // namespace jma
