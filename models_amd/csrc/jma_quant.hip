// GGUF block-quantized matrix-vector products for the projections around attention (the Q/K/V
// projection before the append, llama/LlamaForwardPass.java:1043-1067, and the output projection
// plus residual after it, :1131-1138), on gfx950.
//
// Arithmetic (the definition backend-native's tests hold its Q4_0 kernel to exactly,
// backend-native/src/test/java/com/integrallis/models/backend/nativekernel/
// NativeKernelLibraryTest.java:909-1023): each 32-element block of an activation row is quantized
// to Q8_0 (absmax, inverse 127 / absmax, element = nearest integer of x * inverse by the 1.5 * 2^23
// trick, scale = f16-rounded absmax / 127); each output is the in-order chain over the row's
// blocks of fma(weightScale * activationScale, integer block dot, sum). Integer dots are exact and
// every float operation is the reference's, in its order, so the outputs are the oracle's bit for
// bit.
//
// Work: one 256-thread workgroup per tile of R rows of one matrix. It quantizes the activation
// rows itself into LDS (a few KB at decode sizes: no separate launch), forms every (row, block)
// term of its tile in parallel (coalesced 16-bit weight loads: 18- and 34-byte blocks are only
// 2-byte aligned; 4-element integer dots with v_dot4_i32_i8), then one thread per (activation row,
// output row) runs the block chain from LDS. The bytes are the weights (HBM-bound at large
// shapes); at decode shapes a launch is latency-bound.
#include <hip/hip_runtime.h>

#include "jma_kernels.h"

namespace jma {
namespace {

constexpr uint32_t kQThreads = 256;
typedef short short2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

template <int kCtrl>
__device__ __forceinline__ int dpp_int(int x) {
  return __builtin_amdgcn_mov_dpp(x, kCtrl, 0xF, 0xF, false);
}
constexpr int kQuadXor1 = 0xB1;  // quad_perm [1, 0, 3, 2]
constexpr int kQuadXor2 = 0x4E;  // quad_perm [2, 3, 0, 1]
// Once the quads of 8 consecutive lanes hold equal values, row_half_mirror (lane 7 - i within
// each half row) pairs quad 0 with quad 1 as i ^ 4 would; once those 8-lane groups are equal,
// row_mirror (lane 15 - i within each row of 16) pairs them as i ^ 8 would.
constexpr int kHalfMirror = 0x141;
constexpr int kRowMirror = 0x140;

// A value of the other row of 16 lanes in a 32-lane group (the lane 16 away): v_permlane16_swap
// with both operands x leaves rows {0, 0, 2, 2} and {1, 1, 3, 3} of x in its two results, so a
// lane of row 0 finds its partner in the second and a lane of row 1 in the first. Symmetric
// combinations of the two results give both partners the same bits without choosing.
__device__ __forceinline__ void rows16(uint32_t x, uint32_t& r0, uint32_t& r1) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  r0 = r[0];
  r1 = r[1];
}

// Sum over the 8 consecutive lanes of a group (exact in integers, so the pairing order is free).
__device__ __forceinline__ int sum8(int x) {
  x += dpp_int<kQuadXor1>(x);
  x += dpp_int<kQuadXor2>(x);
  return x + dpp_int<kHalfMirror>(x);
}

// ggmlNearestInt (NativeKernelLibraryTest.java:1019-1022): x + 1.5 * 2^23 rounds x to an integer
// (nearest, ties to even) in the low mantissa bits.
__device__ __forceinline__ int nearest_int(float v) {
#pragma clang fp contract(off)
  const float s = v + 12582912.0f;
  return (int)(__float_as_uint(s) & 0x007FFFFFu) - 0x00400000;
}

__device__ __forceinline__ float f16_bits_to_float(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// Bits 0..3 of x moved to bit 4 of bytes 0..3 (the four shifted copies of x do not overlap, so
// the product has no carries).
__device__ __forceinline__ uint32_t fifth_bits(uint32_t x) { return ((x * 0x00204081u) & 0x01010101u) << 4; }

// Weight block of a format (backend-native's codes: 0 Q4_0, 1 Q8_0, 5 Q5_0): a 16-bit scale,
// then 16 bytes of nibbles (Q4_0), a 32-bit word of fifth bits and 16 bytes of nibbles (Q5_0) or
// 32 int8 (Q8_0), read as 16-bit halves (the blocks are 2-byte aligned only).
template <int FMT>
struct QBlock {
  static constexpr uint32_t kHalves = FMT == 0 ? 9u : FMT == 5 ? 11u : 17u;
  uint32_t h[kHalves];
  __device__ __forceinline__ void load(const uint16_t* rec) {
#pragma unroll
    for (uint32_t i = 0; i < kHalves; ++i) h[i] = rec[i];
  }
  __device__ __forceinline__ uint32_t word(uint32_t j) const { return h[1 + 2 * j] | (h[2 + 2 * j] << 16); }
  // Integer dot of the block with Q8_0 activations aq (8 words of 4 int8) whose element sum is
  // asum. Q4_0: byte i holds element i in its low nibble and element i + 16 in its high one, each
  // offset by 8; the offset is applied as -8 * asum. Q5_0: the same nibbles with bit j of the
  // word at byte 2 as element j's fifth bit, offset by 16 (dot_q5_0_q8_0_row_scalar,
  // backend-native/src/main/rust/model-kernels/src/lib.rs:3204-3252): elements 0..31 as bytes.
  __device__ __forceinline__ int dot(const int* aq, int asum) const {
    int d = 0;
    if constexpr (FMT == 0) {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t w = word(j);
        d = __builtin_amdgcn_sdot4((int)(w & 0x0F0F0F0Fu), aq[j], d, false);
        d = __builtin_amdgcn_sdot4((int)((w >> 4) & 0x0F0F0F0Fu), aq[4 + j], d, false);
      }
      d -= 8 * asum;
    } else if constexpr (FMT == 5) {
      const uint32_t high = word(0);
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t w = h[3 + 2 * j] | (h[4 + 2 * j] << 16);
        const uint32_t lo = (w & 0x0F0F0F0Fu) | fifth_bits((high >> (4 * j)) & 15u);
        const uint32_t hi = ((w >> 4) & 0x0F0F0F0Fu) | fifth_bits((high >> (16 + 4 * j)) & 15u);
        d = __builtin_amdgcn_sdot4((int)lo, aq[j], d, false);
        d = __builtin_amdgcn_sdot4((int)hi, aq[4 + j], d, false);
      }
      d -= 16 * asum;
    } else {
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) d = __builtin_amdgcn_sdot4((int)word(j), aq[j], d, false);
    }
    return d;
  }
};

// Q8_0 quantization of one eighth of a 32-element activation block (quantizeInputs,
// NativeKernelLibraryTest.java:998-1017): the four consecutive lanes of a quad each take eight
// elements and meet for the block maximum and the element sum through DPP quad exchanges. The
// block's absolute maximum (NaN skipped) gives inverse = 127 / absmax, each element the nearest
// integer of x * inverse (the reference's 1.5 * 2^23 addition), the scale the f16-rounded
// absmax / 127. All four lanes of a quad must call it together.
__device__ __forceinline__ void q8_0_eighth(const float* xs, uint2& packed, float& scale, int& sum) {
  const float4 x0 = *(const float4*)xs, x1 = *(const float4*)(xs + 4);
  const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
  float am = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(xv[i]));  // a NaN element is skipped
  am = fmaxf(am, __int_as_float(dpp_int<kQuadXor1>(__float_as_int(am))));
  am = fmaxf(am, __int_as_float(dpp_int<kQuadXor2>(__float_as_int(am))));
  const float inverse = am == 0.0f ? 0.0f : 127.0f / am;
  uint32_t pk[2] = {0u, 0u};
  int s = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float scaled;
    {
#pragma clang fp contract(off)
      scaled = xv[i] * inverse;
    }
    const int q = nearest_int(scaled);
    s += (int)(int8_t)q;
    pk[i >> 2] |= ((uint32_t)q & 0xFFu) << (8 * (i & 3));
  }
  packed = make_uint2(pk[0], pk[1]);
  s += dpp_int<kQuadXor1>(s);
  s += dpp_int<kQuadXor2>(s);
  sum = s;
  scale = (float)(_Float16)(am / 127.0f);
}

// Q8_K quantization of one thirty-second of a 256-element activation block (eight elements;
// quantize_q8_k_batch, backend-native/src/main/rust/model-kernels/src/lib.rs:3906-3952): the 32
// consecutive lanes of the block find the element of largest magnitude (the first on ties, NaN
// skipped) with shuffles; inverse = -127 / that element, each element min(nearest(inverse * x),
// 127). sum16: the 16-element sum of this lane's pair (valid on even parts); scale: 1 / inverse
// (0 for an all-zero block). All 32 lanes of a block must call it together.
__device__ __forceinline__ void q8_k_part(const float* xs, uint32_t part, uint2& packed, int& sum16,
                                          float& scale) {
  const float4 x0 = *(const float4*)xs, x1 = *(const float4*)(xs + 4);
  const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
  float best = 0.0f, bval = 0.0f;
  uint32_t bidx = 0xFFFFFFFFu;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float m = fabsf(xv[i]);
    if (m > best) {  // strict: the first of equal magnitudes; a NaN compares false
      best = m;
      bval = xv[i];
      bidx = part * 8u + i;
    }
  }
  // The block maximum over its 32 lanes under the total order (magnitude, then the lower index
  // first): the same winner whatever the pairing, so DPP exchanges within rows of 16, then the
  // two rows of the group through v_permlane16_swap.
  auto take = [&](float ob, float ov, uint32_t oi) {
    if (ob > best || (ob == best && oi < bidx)) {
      best = ob;
      bval = ov;
      bidx = oi;
    }
  };
  auto step = [&](auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    take(__int_as_float(dpp_int<c>(__float_as_int(best))), __int_as_float(dpp_int<c>(__float_as_int(bval))),
         (uint32_t)dpp_int<c>((int)bidx));
  };
  step(std::integral_constant<int, kQuadXor1>{});
  step(std::integral_constant<int, kQuadXor2>{});
  step(std::integral_constant<int, kHalfMirror>{});
  step(std::integral_constant<int, kRowMirror>{});
  {
    uint32_t b0, b1, v0, v1, i0, i1;
    rows16(__float_as_uint(best), b0, b1);
    rows16(__float_as_uint(bval), v0, v1);
    rows16(bidx, i0, i1);
    const float fb0 = __uint_as_float(b0), fb1 = __uint_as_float(b1);
    const bool second = fb1 > fb0 || (fb1 == fb0 && i1 < i0);
    best = second ? fb1 : fb0;
    bval = __uint_as_float(second ? v1 : v0);
    bidx = second ? i1 : i0;
  }
  int s = 0;
  if (best == 0.0f) {
    packed = make_uint2(0u, 0u);
  } else {
    const float inverse = -127.0f / bval;
    uint32_t pk[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float scaled;
      {
#pragma clang fp contract(off)
        scaled = inverse * xv[i];
      }
      const int q = min(nearest_int(scaled), 127);
      s += (int)(int8_t)q;
      pk[i >> 2] |= ((uint32_t)q & 0xFFu) << (8 * (i & 3));
    }
    packed = make_uint2(pk[0], pk[1]);
  }
  s += dpp_int<kQuadXor1>(s);  // two threads make one 16-element sum
  sum16 = s;
  scale = best == 0.0f ? 0.0f : 1.0f / (-127.0f / bval);
}

}  // namespace

template <int FMT>
__global__ __launch_bounds__(kQThreads) void qmatvec_kernel(const QMatArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char q_lds[];
  // LDS holds one pass of nc activation rows; the workgroup's rows (blockIdx.y's group) pass
  // through it in turn while the weight tile stays in registers.
  const uint32_t nc = a.chunk, cols = a.cols, K = a.blocks, R = a.rows_per_tile, Kp = K + 1;
  int8_t* act_q = (int8_t*)q_lds;                                   // [nc][cols]
  float* act_scale = (float*)(q_lds + ((nc * cols + 15u) & ~15u));  // [nc][K]
  int* act_sum = (int*)(act_scale + nc * K);                        // [nc][K]
  float* t_scale = (float*)(act_sum + nc * K);                      // [nc][R][Kp]
  float* t_dot = t_scale + nc * R * Kp;                             // [nc][R][Kp]

  uint32_t mi = 0;
  for (uint32_t i = 1; i < a.count; ++i) mi = blockIdx.x >= a.m[i].tile0 ? i : mi;
  const uint8_t* w = a.m[mi].w;
  float* out = a.m[mi].out;
  const float* addend = a.m[mi].addend;
  const uint32_t rows = a.m[mi].rows;
  const uint32_t r0 = (blockIdx.x - a.m[mi].tile0) * R;
  const uint32_t nrows = min(R, rows - r0);
  const uint32_t nunits = nrows * K;
  constexpr uint32_t kRecHalves = QBlock<FMT>::kHalves;  // block bytes / 2
  const uint16_t* wrec = (const uint16_t*)(w + (uint64_t)r0 * K * (2u * kRecHalves));
  const uint32_t tid = threadIdx.x;

  // A thread's first kU units (every unit of a tile of up to 1024 terms) are loaded once, in
  // flight while the first activations are quantized, and serve every pass.
  constexpr uint32_t kU = 4;
  QBlock<FMT> unit[kU];
#pragma unroll
  for (uint32_t i = 0; i < kU; ++i)
    if (tid + i * kQThreads < nunits) unit[i].load(wrec + (uint64_t)(tid + i * kQThreads) * kRecHalves);

  const uint32_t g0 = blockIdx.y * a.group_rows, g1 = min(a.batch, g0 + a.group_rows);
  for (uint32_t b0 = g0; b0 < g1; b0 += nc) {
    const uint32_t nb = min(nc, g1 - b0);
    const float* xb = a.x + (uint64_t)b0 * cols;
    // Q8_0 activations: four threads per 32-element block, eight elements each.
    for (uint32_t t = tid; t < nb * K * 4u; t += kQThreads) {
      const uint32_t b = t / (K * 4u), rem = t % (K * 4u), blk = rem >> 2, qtr = rem & 3u;
      uint2 packed;
      float scale;
      int s;
      q8_0_eighth(xb + (uint64_t)b * cols + blk * 32u + qtr * 8u, packed, scale, s);
      *(uint2*)(act_q + (uint64_t)b * cols + blk * 32u + qtr * 8u) = packed;
      if (qtr == 0) {
        act_scale[b * K + blk] = scale;
        act_sum[b * K + blk] = s;
      }
    }
    __syncthreads();

    // Every (row, block) term of the tile: the scale product and the integer dot, per activation
    // row. Tiles of more than kU * 256 terms (rows over 32768 inputs) load further units in turn.
    auto terms = [&](const QBlock<FMT>& wb, uint32_t u) {
      const uint32_t row = u / K, blk = u % K;
      const float wscale = f16_bits_to_float(wb.h[0]);
      for (uint32_t b = 0; b < nb; ++b) {
        const int* aq = (const int*)(act_q + (uint64_t)b * cols + blk * 32u);
        const int d = wb.dot(aq, act_sum[b * K + blk]);
        const uint32_t at = (b * R + row) * Kp + blk;
        t_scale[at] = wscale * act_scale[b * K + blk];
        t_dot[at] = (float)d;
      }
    };
#pragma unroll
    for (uint32_t i = 0; i < kU; ++i)
      if (tid + i * kQThreads < nunits) terms(unit[i], tid + i * kQThreads);
    for (uint32_t u = tid + kU * kQThreads; u < nunits; u += kQThreads) {
      QBlock<FMT> wb;
      wb.load(wrec + (uint64_t)u * kRecHalves);
      terms(wb, u);
    }
    __syncthreads();

    // One thread per (activation row, output row): sum = fma(scale, dot, sum) over the blocks in
    // order, then the optional bias or residual (one float add, as addOptionalBias and the
    // residual loop do).
    for (uint32_t t = tid; t < nb * nrows; t += kQThreads) {
      const uint32_t b = t / nrows, row = t % nrows;
      const float* ps = t_scale + (b * R + row) * Kp;
      const float* pd = t_dot + (b * R + row) * Kp;
      float sum = 0.0f;
      uint32_t blk = 0;
      for (; blk + 8 <= K; blk += 8) {  // the LDS reads of eight steps ahead of their fma chain
        float sc[8], dt[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sc[i] = ps[blk + i], dt[i] = pd[blk + i];
#pragma unroll
        for (int i = 0; i < 8; ++i) sum = __builtin_fmaf(sc[i], dt[i], sum);
      }
      for (; blk < K; ++blk) sum = __builtin_fmaf(ps[blk], pd[blk], sum);
      const uint32_t r = r0 + row;
      const uint64_t o = (uint64_t)(b0 + b) * rows + r;
      if (a.addend_mode == 1) sum = sum + addend[r];
      else if (a.addend_mode == 2) sum = sum + addend[o];
      out[o] = sum;
    }
  }
}

// ---------------------------------------------------------------- K-quants (Q4_K, Q5_K, Q6_K)
//
// Q8_K activations (quantize_q8_k_batch, backend-native/src/main/rust/model-kernels/src/lib.rs:
// 3906-3952): per 256-element block, the element of largest magnitude (the first on ties, NaN
// skipped) sets inverse = -127 / max, element = min(nearest(inverse * x), 127), sums of 16
// elements, scale = 1 / inverse. Rows as backend-native's scalar row kernels form them
// (dot_q4_k_q8_k_row_scalar :3410-3459, dot_q5_k_q8_k_row_scalar :3461-3518,
// dot_q6_k_q8_k_row_scalar :3519-3577); the integer parts are exact in any order, so eight
// threads share each (row, block) and only the float chains keep the reference's order. Q5_K is
// Q4_K with a 32-byte array of fifth bits ahead of the nibbles (bit g of byte i: element i of
// group g), so the two share their code and float chain.
template <int FMT>
__global__ __launch_bounds__(kQThreads) void qkmatvec_kernel(const QMatArgs a) {
  constexpr bool kQ45 = FMT == 2 || FMT == 4;          // Q4_K or Q5_K
  constexpr uint32_t kNT = kQ45 ? 4u : 9u;             // floats per (row, block) term
  constexpr uint32_t kBlockBytes = FMT == 2 ? 144u : FMT == 4 ? 176u : 210u;
  extern __shared__ __attribute__((aligned(16))) unsigned char q_lds[];
  // One pass of nc activation rows in LDS at a time (qmatvec_kernel); the tile's weight blocks
  // come from memory in the first pass and from the caches in later ones.
  const uint32_t nc = a.chunk, cols = a.cols, KB = a.blocks, R = a.rows_per_tile;
  const uint32_t rs = KB * kNT + 1;  // floats per (activation row, output row) of terms
  int8_t* act_q = (int8_t*)q_lds;                                   // [nc][cols]
  float* act_scale = (float*)(q_lds + ((nc * cols + 15u) & ~15u));  // [nc][KB]
  int* act_sum = (int*)(act_scale + nc * KB);                       // [nc][cols / 16]
  float* terms = (float*)(act_sum + nc * (cols / 16u));             // [nc][R][rs]

  uint32_t mi = 0;
  for (uint32_t i = 1; i < a.count; ++i) mi = blockIdx.x >= a.m[i].tile0 ? i : mi;
  const uint8_t* w = a.m[mi].w;
  float* out = a.m[mi].out;
  const float* addend = a.m[mi].addend;
  const uint32_t rows = a.m[mi].rows;
  const uint32_t r0 = (blockIdx.x - a.m[mi].tile0) * R;
  const uint32_t nrows = min(R, rows - r0);
  const uint32_t nunits = nrows * KB;
  const uint8_t* wtile = w + (uint64_t)r0 * KB * kBlockBytes;
  const uint32_t tid = threadIdx.x, sub = tid & 7u;

  const uint32_t g0 = blockIdx.y * a.group_rows, g1 = min(a.batch, g0 + a.group_rows);
  for (uint32_t b0 = g0; b0 < g1; b0 += nc) {
    const uint32_t nb = min(nc, g1 - b0);
    const float* xb = a.x + (uint64_t)b0 * cols;
    // Q8_K activations: 32 threads per block, eight consecutive elements each.
    for (uint32_t t = tid; t < nb * KB * 32u; t += kQThreads) {
      const uint32_t b = t / (KB * 32u), blk = (t / 32u) % KB, part = t & 31u;
      uint2 packed;
      int s;
      float scale;
      q8_k_part(xb + (uint64_t)b * cols + blk * 256u + part * 8u, part, packed, s, scale);
      *(uint2*)(act_q + (uint64_t)b * cols + blk * 256u + part * 8u) = packed;
      if ((part & 1u) == 0) act_sum[b * (cols / 16u) + blk * 16u + part / 2u] = s;
      if (part == 0) act_scale[b * KB + blk] = scale;
    }
    __syncthreads();

    // Terms: eight threads per (row, block); every thread of a unit runs the same batch loop.
    for (uint32_t t = tid; t < ((nunits * 8u + 63u) & ~63u); t += kQThreads) {
      const uint32_t u = min(t / 8u, nunits - 1u);  // the last wave's spare lanes repeat a unit
      const bool real = t / 8u < nunits;
      const uint32_t row = u / KB, blk = u % KB;
      const uint8_t* wb = wtile + (uint64_t)u * kBlockBytes;
      if constexpr (kQ45) {
        const uint16_t* h = (const uint16_t*)wb;
        const float wd = f16_bits_to_float(h[0]), wdmin = f16_bits_to_float(h[1]);
        uint32_t scb[12];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
          const uint32_t x = h[2 + i];
          scb[2 * i] = x & 0xFFu;
          scb[2 * i + 1] = x >> 8;
        }
        const uint32_t g = sub;
        const int sc = g < 4 ? (int)(scb[g] & 63u) : (int)((scb[g + 4] & 15u) | ((scb[g - 4] >> 6) << 4));
        const int mn = g < 4 ? (int)(scb[g + 4] & 63u) : (int)((scb[g + 4] >> 4) | ((scb[g] >> 6) << 4));
        // The group's 32 quants as 8 words of 4 bytes: nibbles (Q5_K: plus bit g of each qh byte
        // as the byte's bit 4).
        uint32_t nib[8];
        const uint16_t* qn16 = h + (FMT == 4 ? 24 : 8) + (g >> 1) * 16;
        const uint32_t shift = (g & 1u) * 4u;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          nib[i] = (((uint32_t)qn16[2 * i] | ((uint32_t)qn16[2 * i + 1] << 16)) >> shift) & 0x0F0F0F0Fu;
        if constexpr (FMT == 4) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const uint32_t qh = (uint32_t)h[8 + 2 * i] | ((uint32_t)h[9 + 2 * i] << 16);
            nib[i] |= ((qh >> g) & 0x01010101u) << 4;
          }
        }
        for (uint32_t b = 0; b < nb; ++b) {
          const int* aq = (const int*)(act_q + (uint64_t)b * cols + blk * 256u + g * 32u);
          int dot = 0;
#pragma unroll
          for (int i = 0; i < 8; ++i) dot = __builtin_amdgcn_sdot4((int)nib[i], aq[i], dot, false);
          const int* s16 = act_sum + b * (cols / 16u) + blk * 16u;
          const int qs = sum8(sc * dot), ms = sum8(mn * (s16[2 * g] + s16[2 * g + 1]));
          if (real && sub == 0) {
            const float as = act_scale[b * KB + blk];
            float* tt = terms + (b * R + row) * rs + blk * kNT;
            tt[0] = wd * as;
            tt[1] = (float)qs;
            tt[2] = -(wdmin * as);
            tt[3] = (float)ms;
          }
        }
      } else {
        // Lane class l = sub: elements i, i + 8, i + 16, i + 24 of each 32-run, both halves, all
        // four quarters (ql low / high nibble, qh bit pairs), each times its int8 group scale.
        const int8_t* sc = (const int8_t*)(wb + 192);
        const float wd = (float)__builtin_bit_cast(_Float16, (uint16_t)(wb[208] | (wb[209] << 8)));
        int ql1[8], ql2[8], qhh[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t hf = k >> 2, i = sub + 8u * (k & 3);
          ql1[k] = wb[hf * 64u + i];
          ql2[k] = wb[hf * 64u + 32u + i];
          qhh[k] = wb[128u + hf * 32u + i];
        }
        for (uint32_t b = 0; b < nb; ++b) {
          const int8_t* aq = act_q + (uint64_t)b * cols + blk * 256u;
          int acc = 0;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const uint32_t hf = k >> 2, i = sub + 8u * (k & 3), si = i / 16u;
            const int q1 = ((ql1[k] & 15) | ((qhh[k] & 3) << 4)) - 32;
            const int q2 = ((ql2[k] & 15) | (((qhh[k] >> 2) & 3) << 4)) - 32;
            const int q3 = ((ql1[k] >> 4) | (((qhh[k] >> 4) & 3) << 4)) - 32;
            const int q4 = ((ql2[k] >> 4) | (((qhh[k] >> 6) & 3) << 4)) - 32;
            const int8_t* aa = aq + hf * 128u;
            acc += sc[hf * 8u + si] * q1 * aa[i];
            acc += sc[hf * 8u + si + 2u] * q2 * aa[i + 32u];
            acc += sc[hf * 8u + si + 4u] * q3 * aa[i + 64u];
            acc += sc[hf * 8u + si + 6u] * q4 * aa[i + 96u];
          }
          if (real) {
            float* tt = terms + (b * R + row) * rs + blk * kNT;
            if (sub == 0) tt[0] = wd * act_scale[b * KB + blk];
            tt[1 + sub] = (float)acc;
          }
        }
      }
    }
    __syncthreads();

    for (uint32_t t = tid; t < nb * nrows; t += kQThreads) {
      const uint32_t b = t / nrows, row = t % nrows;
      const float* tt = terms + (b * R + row) * rs;
      float sum = 0.0f;
      if constexpr (kQ45) {
        for (uint32_t blk = 0; blk < KB; ++blk) {
          sum = __builtin_fmaf(tt[blk * 4], tt[blk * 4 + 1], sum);
          sum = __builtin_fmaf(tt[blk * 4 + 2], tt[blk * 4 + 3], sum);
        }
      } else {
        float ls[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (uint32_t blk = 0; blk < KB; ++blk)
#pragma unroll
          for (int l = 0; l < 8; ++l) ls[l] = __builtin_fmaf(tt[blk * 9], tt[blk * 9 + 1 + l], ls[l]);
#pragma unroll
        for (int l = 0; l < 8; ++l) sum = sum + ls[l];
      }
      const uint32_t r = r0 + row;
      const uint64_t o = (uint64_t)(b0 + b) * rows + r;
      if (a.addend_mode == 1) sum = sum + addend[r];
      else if (a.addend_mode == 2) sum = sum + addend[o];
      out[o] = sum;
    }
  }
}

// ---------------------------------------------------------------- prefill-sized batches
//
// Batches of kQGemmMinBatch activation rows and more run as matrix products on activations
// quantized once into scratch, in the matrix ops' operand order (qact_index, qact_scale_index).

// Eight int8 as halves in the order of a run of qact_index.
__device__ __forceinline__ half8_t act_run(uint2 packed) {
  half8_t v;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    v[(i & ~3) | ((i & 1) << 1) | ((i >> 1) & 1)] =
        (_Float16)(short)(int8_t)((i < 4 ? packed.x : packed.y) >> (8 * (i & 3)));
  return v;
}

// Q8_0 activations of the 32-element formats: a wave takes one block of 16 rows, a quad of lanes
// per row. Rows past the batch (up to a multiple of 32) get zeros.
__global__ __launch_bounds__(kQThreads) void q8_0_quant_kernel(const float* x, uint32_t batch,
                                                               uint32_t cols, _Float16* act,
                                                               uint16_t* scales) {
  const uint32_t K = cols / 32u, pairs = (K + 1u) / 2u;
  const uint32_t tile = blockIdx.x / pairs, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t blk = blockIdx.x % pairs * 2u + (wave >> 1);
  if (blk >= K) return;
  const uint32_t b = tile * 32u + (wave & 1u) * 16u + lane / 4u, qtr = lane & 3u;
  uint2 packed;
  float scale;
  int s;
  q8_0_eighth(x + (uint64_t)min(b, batch - 1u) * cols + blk * 32u + qtr * 8u, packed, scale, s);
  half8_t v = act_run(packed);
  if (b >= batch) {
    v = half8_t{};
    scale = 0.0f;
  }
  *(half8_t*)(act + qact_index(b, blk * 32u + qtr * 8u, cols)) = v;
  if (qtr == 0)
    scales[qact_scale_index(b, blk, K)] = __builtin_bit_cast(uint16_t, (_Float16)scale);
}

// Q8_K activations of the K-quants: a workgroup takes one 256-element block of 8 rows, 32 threads
// a row with 8 elements each. Rows past the batch (up to a multiple of 32) get zeros. The block's
// sixteen 16-element sums (below 2048 in magnitude, exact in f16) and its scale go beside them;
// `classes` (null = not needed) gets the values in Q6_K's order too; act null: only that order.
__global__ __launch_bounds__(kQThreads) void q8_k_quant_kernel(const float* x, uint32_t batch,
                                                               uint32_t cols, _Float16* act,
                                                               _Float16* classes, _Float16* sums,
                                                               float* scales) {
  const uint32_t KB = cols / 256u, blk = blockIdx.x % KB;
  const uint32_t b = blockIdx.x / KB * 8u + threadIdx.x / 32u, part = threadIdx.x & 31u;
  uint2 packed;
  int s;
  float scale;
  q8_k_part(x + (uint64_t)min(b, batch - 1u) * cols + blk * 256u + part * 8u, part, packed, s, scale);
  if (b >= batch) {
    packed = make_uint2(0u, 0u);
    s = 0;
    scale = 0.0f;
  }
  if (act != nullptr) {
    *(half8_t*)(act + qact_index(b, blk * 256u + part * 8u, cols)) = act_run(packed);
    if ((part & 1u) == 0) sums[qact_sum_index(b, blk, part / 2u, KB)] = (_Float16)(short)s;
  }
  if (part == 0) scales[qact_scale_index(b, blk, KB)] = scale;
  if (classes == nullptr) return;
  // The four lanes of a quad hold elements l, l + 8, l + 16, l + 24 of one 32-element run for every
  // class l: lane m takes classes 2 m and 2 m + 1, bytes 2 m and 2 m + 1 of all four lanes.
  const uint32_t m = part & 3u, sel = (m & 1u) ? 16u : 0u;
  half2_t lo[2], hi[2];
  auto take = [&](auto from) {
    constexpr int f = decltype(from)::value, ctrl = f * 0x55;  // quad_perm [f, f, f, f]
    const uint32_t px = (uint32_t)dpp_int<ctrl>((int)packed.x), py = (uint32_t)dpp_int<ctrl>((int)packed.y);
    const uint32_t two = (m < 2u ? px : py) >> sel;
    lo[f / 2][f % 2] = (_Float16)(short)(int8_t)two;
    hi[f / 2][f % 2] = (_Float16)(short)(int8_t)(two >> 8);
  };
  take(std::integral_constant<int, 0>{});
  take(std::integral_constant<int, 1>{});
  take(std::integral_constant<int, 2>{});
  take(std::integral_constant<int, 3>{});
  const uint32_t e = blk * 256u + part / 4u * 32u + 2u * m;  // element 2 m of the run: class 2 m
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i) {
    *(half2_t*)(classes + qact_class_index(b, e + 16u * i, cols)) = lo[i];
    *(half2_t*)(classes + qact_class_index(b, e + 1u + 16u * i, cols)) = hi[i];
  }
}

hipError_t launch_q8_k_quant(const float* x, uint32_t batch, uint32_t cols, void* act, void* classes,
                             void* sums, void* scales, hipStream_t stream) {
  const uint32_t blocks = qact_tiles(batch) * 4u * (cols / 256u);
  hipLaunchKernelGGL(q8_k_quant_kernel, dim3(blocks), dim3(kQThreads), 0, stream, x, batch, cols,
                     (_Float16*)act, (_Float16*)classes, (_Float16*)sums, (float*)scales);
  return hipGetLastError();
}

hipError_t launch_q8_0_quant(const float* x, uint32_t batch, uint32_t cols, void* act, void* scales,
                             hipStream_t stream) {
  const uint32_t blocks = qact_tiles(batch) * ((cols / 32u + 1u) / 2u);
  hipLaunchKernelGGL(q8_0_quant_kernel, dim3(blocks), dim3(kQThreads), 0, stream, x, batch, cols,
                     (_Float16*)act, (uint16_t*)scales);
  return hipGetLastError();
}

hipError_t launch_qmatvec(const QMatArgs& a, uint32_t fmt, uint32_t tiles, hipStream_t stream) {
  const size_t lds = qmatvec_lds_bytes(a.chunk, a.cols, a.rows_per_tile);
  const dim3 grid(tiles, (a.batch + a.group_rows - 1) / a.group_rows);
  if (fmt == 0)
    hipLaunchKernelGGL(qmatvec_kernel<0>, grid, dim3(kQThreads), lds, stream, a);
  else if (fmt == 1)
    hipLaunchKernelGGL(qmatvec_kernel<1>, grid, dim3(kQThreads), lds, stream, a);
  else if (fmt == 2)
    hipLaunchKernelGGL(qkmatvec_kernel<2>, grid, dim3(kQThreads),
                       qkmatvec_lds_bytes(2, a.chunk, a.cols, a.rows_per_tile), stream, a);
  else if (fmt == 3)
    hipLaunchKernelGGL(qkmatvec_kernel<3>, grid, dim3(kQThreads),
                       qkmatvec_lds_bytes(3, a.chunk, a.cols, a.rows_per_tile), stream, a);
  else if (fmt == 4)
    hipLaunchKernelGGL(qkmatvec_kernel<4>, grid, dim3(kQThreads),
                       qkmatvec_lds_bytes(4, a.chunk, a.cols, a.rows_per_tile), stream, a);
  else if (fmt == 5)
    hipLaunchKernelGGL(qmatvec_kernel<5>, grid, dim3(kQThreads), lds, stream, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace jma
