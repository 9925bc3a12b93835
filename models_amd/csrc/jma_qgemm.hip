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

// Bytes 0 and 1 (or 2 and 3) of x, unsigned, as two halves less `bias`: 0x6400 | u is 1024 + u.
template <int kBias>
__device__ __forceinline__ uint32_t bytes_to_half2(uint32_t x, uint32_t sel) {
  const half2_t off = {(_Float16)(-1024.0f - kBias), (_Float16)(-1024.0f - kBias)};
  const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, x, sel)) + off;
  return __builtin_bit_cast(uint32_t, v);
}
template <int kBias>
__device__ __forceinline__ half8_t bytes_to_half8(uint32_t x0, uint32_t x1) {
  u32x4_t r;
  r[0] = bytes_to_half2<kBias>(x0, 0x04010400u);
  r[1] = bytes_to_half2<kBias>(x0, 0x04030402u);
  r[2] = bytes_to_half2<kBias>(x1, 0x04010400u);
  r[3] = bytes_to_half2<kBias>(x1, 0x04030402u);
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
    if constexpr (FMT == 1) {  // int8: the sign bit flipped makes v + 128
      return bytes_to_half8<128>(q[c].x ^ 0x80808080u, q[c].y ^ 0x80808080u);
    } else {
      uint32_t x0 = (q[0].x >> (4 * c)) & 0x0F0F0F0Fu;
      uint32_t x1 = (q[0].y >> (4 * c)) & 0x0F0F0F0Fu;
      if constexpr (FMT == 5) {
        x0 |= fifth_bits((qh >> (16 * c)) & 15u);
        x1 |= fifth_bits((qh >> (16 * c + 4)) & 15u);
        return bytes_to_half8<16>(x0, x1);
      } else {
        return bytes_to_half8<8>(x0, x1);
      }
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

// Barrier once at most N of this wave's loads are in flight and its LDS writes are done.
template <int N>
__device__ __forceinline__ void wait_barrier() {
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
// unpacking, on one SIMD; the two overlap only partly (matrix unit busy 30% of the time, vector
// issue about 40%). 3072 + 1024 + 1024 rows of 3072 inputs, 2048 activation rows, Q4_0: 519 us
// with integer dots on the vector unit, 140 us with this kernel (459 TOPS).
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

namespace {
template <int FMT, uint32_t I>
void launch_shape(const QMatArgs& a, uint32_t tiles_w, const _Float16* act, const uint16_t* scales, hipStream_t stream) {
  constexpr QGemmShape s = kQGemmShape[I];
  const uint32_t tiles_b = (a.batch + qgemm_rows_b(s) - 1) / qgemm_rows_b(s);
  hipLaunchKernelGGL((qgemm_kernel<FMT, s.bt, s.wt, s.nb, s.nw>), dim3(tiles_w * tiles_b),
                     dim3(qgemm_threads(s)), 0, stream, a, act, scales, tiles_w, qgemm_recip(tiles_w),
                     tiles_w * tiles_b);
}
template <int FMT>
hipError_t launch_fmt(const QMatArgs& a, uint32_t shape, uint32_t tiles_w, const _Float16* act,
                      const uint16_t* scales, hipStream_t stream) {
  switch (shape) {
    case 0: launch_shape<FMT, 0>(a, tiles_w, act, scales, stream); break;
    case 1: launch_shape<FMT, 1>(a, tiles_w, act, scales, stream); break;
    case 2: launch_shape<FMT, 2>(a, tiles_w, act, scales, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_qgemm(const QMatArgs& a, uint32_t fmt, uint32_t shape, uint32_t tiles_w,
                        const void* act, const void* act_scale, hipStream_t stream) {
  const _Float16* x = (const _Float16*)act;
  const uint16_t* s = (const uint16_t*)act_scale;
  if (fmt == 0) return launch_fmt<0>(a, shape, tiles_w, x, s, stream);
  if (fmt == 1) return launch_fmt<1>(a, shape, tiles_w, x, s, stream);
  if (fmt == 5) return launch_fmt<5>(a, shape, tiles_w, x, s, stream);
  return hipErrorInvalidValue;
}

}  // namespace jma
