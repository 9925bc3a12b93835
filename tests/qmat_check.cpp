// CPU bounds check of the quantized-projection launches (models_amd/csrc/jma_quant.hip and
// models_amd/csrc/jma_qgemm.hip), built
// with g++ and AddressSanitizer / UndefinedBehaviorSanitizer by tests/test_plan_cpu.py.
//
// For each call below it routes every weight format the way quantized_matmul_impl does and plans
// its launch with the runtime's own planner (jma_plan.h): prefill-sized batches run the
// matrix-core product (qgemm_kernel, qkgemm_kernel, q6gemm_kernel) in the workgroup tiles that
// plan_qgemm picks, over activations quantized once into scratch; the others run the matrix-vector
// kernels (plan_qmat, qmat_group_rows), whose workgroups take `chunk` activation rows per pass. It then walks every workgroup (x, y) of every launch the way the kernels index
// memory: the matrix a workgroup serves (the last with tile0 <= x), its weight blocks, the
// activations (or the quantized activation scratch) it reads, its LDS arrays, and every output,
// bias and residual element it reads or writes. Every access touches an exactly sized heap array,
// so an index past an extent is a sanitizer error; every output element must be written exactly
// once across the call's launches.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <string>
#include <vector>

#include "jma_plan.h"

namespace {

int failures = 0;

void expect(bool ok, const std::string& what) {
  if (!ok) {
    ++failures;
    fprintf(stderr, "FAIL: %s\n", what.c_str());
  }
}

struct Call {
  std::string name;
  std::vector<uint32_t> formats, rows;
  uint32_t batch, cols, addend_mode;
};

// The routing of quantized_matmul_impl.
bool gemm_format(uint32_t, uint32_t batch) { return batch >= jma::kQGemmMinBatch; }

struct Buffers {
  std::vector<uint8_t*> w;
  std::vector<float*> add;
  float* x = nullptr;           // activations [batch][cols]
  // quantized activations, their scales and (Q8_K) the values in class order and the sums
  std::vector<uint16_t> act, act_scale, act_class, act_sum;
  std::vector<float> act_scale_k;
  std::vector<uint8_t> written;  // per output element
};

volatile float sink = 0.0f;

// Launch table of one format: (matrix, first tile, output offset) in matrix order.
struct M { uint32_t idx, tile0; uint64_t out_off; };

std::vector<M> table(const Call& c, uint32_t fmt, uint32_t R, uint32_t& tiles) {
  std::vector<M> ms;
  tiles = 0;
  uint64_t out_off = 0;
  for (uint32_t i = 0; i < c.formats.size(); ++i) {
    if (c.formats[i] == fmt) {
      ms.push_back({i, tiles, out_off});
      tiles += (c.rows[i] + R - 1) / R;
    }
    out_off += (uint64_t)c.batch * c.rows[i];
  }
  return ms;
}

// qgemm_kernel: workgroups in qgemm_tile's order, each thread stages one weight block per step (rows
// and blocks clamped to the last valid one), each wave its 1 KB pieces of the activation stage and
// its scales; outputs in 32 x 32 tiles. Every access at its first and last byte.
void walk_qgemm(const Call& c, uint32_t fmt, const jma::QGemmShape s, Buffers& B) {
  const uint32_t K = c.cols / 32u, kB = jma::qgemm_rows_b(s), kW = jma::qgemm_rows_w(s);
  const uint32_t threads = jma::qgemm_threads(s), waves = s.nb * s.nw, units = kW * 2;
  uint32_t tiles;
  const std::vector<M> ms = table(c, fmt, kW, tiles);
  const uint32_t bb = jma::qmat_block_bytes(fmt), tiles_b = (c.batch + kB - 1) / kB;
  const uint32_t total = tiles * tiles_b, btiles = jma::qact_tiles(c.batch);
  const uint32_t pieces = kB / 32 * 2, ppw = (pieces + waves - 1) / waves;
  std::vector<uint8_t> seen(total, 0);
  expect(units <= threads, c.name + ": at most one staged half block per thread");
  std::vector<uint16_t> w_lds(kW * 32), a_lds(kB * 32), c_lds(kW);
  for (uint32_t id = 0; id < total; ++id) {
    uint32_t tx, ty;
    jma::qgemm_tile(id, tiles, jma::qgemm_recip(tiles), total, tx, ty);
    expect(tx < tiles && ty < tiles_b, c.name + ": product tile in range");
    seen[ty * tiles + tx]++;
    uint32_t mi = 0;
    for (uint32_t i = 1; i < ms.size(); ++i) mi = tx >= ms[i].tile0 ? i : mi;
    const uint32_t idx = ms[mi].idx, rows = c.rows[idx];
    const uint32_t r0 = (tx - ms[mi].tile0) * kW, b0 = ty * kB;
    expect(r0 < rows, c.name + ": product tile past its matrix");
    auto a_tile = [&](uint32_t i) { return std::min(b0 / 32u + i, btiles - 1u); };
    for (uint32_t step = 0; step < (K + 3) / 4 * 4 + 3; ++step) {  // loads run three steps ahead
      const uint64_t k = std::min(step, K - 1u);
      std::vector<uint8_t> w_put(kW * 4, 0), a_put(pieces, 0);
      for (uint32_t tid = 0; tid < threads; ++tid) {
        const uint32_t su_row = tid % units / 2u, h = tid & 1u;
        const uint64_t row = std::min(r0 + su_row, rows - 1u);
        const uint8_t* blk = B.w[idx] + (row * K + k) * bb;
        const uint32_t q = (fmt == 5 ? 6u : 2u) + 8u * h;
        sink = sink + blk[0] + blk[1] + blk[q] + blk[q + 7u] + blk[fmt == 1 ? 18u + 8u * h + 7u : 5u];
        const uint32_t slot = (su_row / 32u) * 1024u + h * 256u + (su_row % 32u) * 8u;
        for (uint32_t i = 0; i < 2; ++i) {
          w_lds[slot + i * 512] = 0;
          w_lds[slot + i * 512 + 7] = 0;
          w_put[(slot + i * 512) / 256] = 1;  // one of the 32-row runs of 8
        }
        c_lds[su_row] = 0;
      }
      for (uint32_t wv = 0; wv < waves; ++wv) {
        for (uint32_t i = 0; i < ppw; ++i) {
          const uint32_t p = (wv + waves * i) % pieces;
          const uint64_t off = (uint64_t)a_tile(p / 2u) * 32u * c.cols + p % 2u * 512u + k * 1024u;
          sink = sink + B.act[off] + B.act[off + 511];
          a_lds[p * 512] = 0;
          a_lds[p * 512 + 511] = 0;
          a_put[p] = 1;
        }
        for (uint32_t i = 0; i < s.bt; ++i) {
          const uint32_t t = wv / s.nw * s.bt + i;
          sink = sink + B.act_scale[((uint64_t)a_tile(t) * K + k) * 32u + 31u] + a_lds[t * 1024 + 512 + 63 * 8 + 7];
        }
        for (uint32_t i = 0; i < s.wt; ++i) {
          const uint32_t t = wv % s.nw * s.wt + i;
          sink = sink + w_lds[t * 1024 + 512 + 63 * 8 + 7] + c_lds[t * 32 + 31];
        }
      }
      for (uint32_t i = 0; i < kW * 4 / 32; ++i) expect(w_put[i] == 1, c.name + ": every weight run staged");
      for (uint8_t n : a_put) expect(n == 1, c.name + ": every activation piece loaded");
    }
    for (uint32_t r = r0; r < std::min(r0 + kW, rows); ++r)
      for (uint32_t b = b0; b < std::min(b0 + kB, c.batch); ++b) {
        const uint64_t o = (uint64_t)b * rows + r;
        if (c.addend_mode == 1) sink = sink + B.add[idx][r];
        if (c.addend_mode == 2) sink = sink + B.add[idx][o];
        B.written[ms[mi].out_off + o]++;
      }
  }
  for (uint8_t n : seen) expect(n == 1, c.name + ": every product tile once");
}

// The activation quantization of the products: every element and scale of every 32-row tile once.
void walk_quant(const Call& c, Buffers& B) {
  const uint32_t K = c.cols / 32u, rows = jma::qact_tiles(c.batch) * 32u;
  for (uint32_t b = 0; b < rows; ++b)
    for (uint32_t k = 0; k < c.cols; k += 8) {
      const uint64_t at = jma::qact_index(b, k, c.cols);
      expect(at % 8 == 0, c.name + ": activation run aligned");
      for (uint32_t i = 0; i < 8; ++i) B.act[jma::qact_index(b, k + i, c.cols)]++;
      if (k % 32 == 0) B.act_scale[jma::qact_scale_index(b, k / 32, K)]++;
    }
  for (uint64_t i = 0; i < (uint64_t)rows * c.cols; i += 8)
    expect(B.act[i] == 1 && B.act[i + 3] == 1 && B.act[i + 7] == 1, c.name + ": every activation run once");
  for (uint64_t i = 0; i < (uint64_t)rows * K; ++i)
    expect(B.act_scale[i] == 1, c.name + ": every activation scale once");
  const jma::QactLayout o = jma::qact_layout(jma::qact_elements(c.batch, c.cols), jma::kQactBlocks);
  expect(o.act == 0 && o.scales >= (uint64_t)rows * c.cols * 2 && o.total - o.scales >= (uint64_t)rows * K * 2,
         c.name + ": activation scratch regions");
}

// qkgemm_kernel (Q4_K, Q5_K) and q6gemm_kernel (Q6_K): as walk_qgemm, a step one 32-element group
// (or class) of a block; the block's header, quants, sums and scales at their first and last bytes.
void walk_qkgemm(const Call& c, uint32_t fmt, const jma::QGemmShape s, Buffers& B) {
  const uint32_t KB = c.cols / 256u, kB = jma::qgemm_rows_b(s), kW = jma::qgemm_rows_w(s);
  const uint32_t threads = jma::qgemm_threads(s), waves = s.nb * s.nw;
  const bool q6 = fmt == 3;
  uint32_t tiles;
  const std::vector<M> ms = table(c, fmt, kW, tiles);
  const uint32_t bb = jma::qmat_block_bytes(fmt), tiles_b = (c.batch + kB - 1) / kB;
  const uint32_t total = tiles * tiles_b, btiles = jma::qact_tiles(c.batch);
  const uint32_t pieces = kB / 32 * 2, ppw = (pieces + waves - 1) / waves;
  const uint32_t scale_pieces = (kB + 63) / 64;
  const std::vector<uint16_t>& act = q6 ? B.act_class : B.act;
  std::vector<uint8_t> seen(total, 0);
  std::vector<uint16_t> w_lds(kW * (q6 ? 64 : 32)), a_lds(kB * 32), s_lds(kW * 16);
  std::vector<float> as_lds(scale_pieces * 64), d_lds(kW);
  if (q6) expect(threads == kW * 8 && pieces == waves, c.name + ": Q6_K staging");
  else expect(kW * 2 <= threads, c.name + ": at most one staged half block per thread");
  for (uint32_t id = 0; id < total; ++id) {
    uint32_t tx, ty;
    jma::qgemm_tile(id, tiles, jma::qgemm_recip(tiles), total, tx, ty);
    expect(tx < tiles && ty < tiles_b, c.name + ": product tile in range");
    seen[ty * tiles + tx]++;
    uint32_t mi = 0;
    for (uint32_t i = 1; i < ms.size(); ++i) mi = tx >= ms[i].tile0 ? i : mi;
    const uint32_t idx = ms[mi].idx, rows = c.rows[idx];
    const uint32_t r0 = (tx - ms[mi].tile0) * kW, b0 = ty * kB;
    expect(r0 < rows, c.name + ": product tile past its matrix");
    auto a_tile = [&](uint32_t i) { return std::min(b0 / 32u + i, btiles - 1u); };
    for (uint32_t kbx = 0; kbx <= KB; ++kbx) {  // loads run up to one block ahead
      const uint64_t kb = std::min(kbx, KB - 1u);
      std::vector<uint8_t> w_put(kW * (q6 ? 16 : 4), 0);
      for (uint32_t tid = 0; tid < threads; ++tid) {
        const uint32_t su_row = q6 ? tid / 8u : tid % (kW * 2) / 2u;
        const uint8_t* blk = B.w[idx] + ((uint64_t)std::min(r0 + su_row, rows - 1u) * KB + kb) * bb;
        if (q6) {
          const uint32_t hf = tid >> 2 & 1u, rr = tid >> 1 & 1u, sp = tid & 1u;
          const uint32_t ql = 64u * hf + 32u * rr + 16u * sp, qh = 128u + 32u * hf + 16u * sp;
          sink = sink + blk[ql] + blk[ql + 15u] + blk[qh] + blk[qh + 15u] + blk[192u + 8u * hf] + blk[199u + 8u * hf] + blk[209];
          const uint32_t slot = (su_row / 32u) * 2048u + hf * 512u + rr * 256u + (su_row % 32u) * 8u + sp * 4u;
          for (uint32_t o = 0; o < 2; ++o) {
            w_lds[slot + o * 1024u + 3u] = 0;
            w_put[(slot + o * 1024u) / 4u]++;
          }
        } else {
          const uint32_t h = tid & 1u, q = fmt == 4 ? 48u : 16u;
          sink = sink + blk[0] + blk[15];
          for (uint32_t p = 0; p < 4; ++p) sink = sink + blk[q + 32u * p + 8u * h] + blk[q + 32u * p + 16u + 8u * h + 7u];
          if (fmt == 4) sink = sink + blk[16u + 8u * h] + blk[32u + 8u * h + 7u];
          const uint32_t slot = (su_row / 32u) * 1024u + h * 256u + (su_row % 32u) * 8u;
          w_lds[slot + 7u] = w_lds[slot + 512u + 7u] = 0;
          w_put[slot / 8u] = w_put[(slot + 512u) / 8u] = 1;
          s_lds[(su_row / 32u) * 512u + h * 256u + (su_row % 32u) * 8u + 7u] = 0;
        }
        d_lds[su_row] = 0;
      }
      for (uint32_t i = 0; i < (q6 ? kW * 16u : kW * 4u); ++i) expect(w_put[i] == 1, c.name + ": every weight run staged once");
      for (uint32_t g = 0; g < 8; ++g)
        for (uint32_t wv = 0; wv < waves; ++wv)
          for (uint32_t i = 0; i < ppw; ++i) {
            const uint32_t p = (wv + waves * i) % pieces;
            const uint64_t off = (uint64_t)a_tile(p / 2u) * 32u * c.cols + p % 2u * 512u + (kb * 8u + g) * 1024u;
            sink = sink + act[off] + act[off + 511];
            a_lds[p * 512 + 511] = 0;
          }
      for (uint32_t i = 0; i < scale_pieces; ++i)
        for (uint32_t h = 0; h < 2; ++h) {
          sink = sink + B.act_scale_k[((uint64_t)a_tile(2u * i + h) * KB + kb) * 32u + 31u];
          as_lds[64 * i + 32 * h + 31] = 0;
        }
      for (uint32_t t = 0; t < kB / 32 && !q6; ++t) sink = sink + B.act_sum[((uint64_t)a_tile(t) * KB + kb) * 512u + 511u];
    }
    for (uint32_t r = r0; r < std::min(r0 + kW, rows); ++r)
      for (uint32_t b = b0; b < std::min(b0 + kB, c.batch); ++b) {
        const uint64_t o = (uint64_t)b * rows + r;
        if (c.addend_mode == 1) sink = sink + B.add[idx][r];
        if (c.addend_mode == 2) sink = sink + B.add[idx][o];
        B.written[ms[mi].out_off + o]++;
      }
  }
  for (uint8_t n : seen) expect(n == 1, c.name + ": every product tile once");
}

// q8_k_quant_kernel: every value in both orders, sum and scale of every 32-row tile once.
void walk_quant_k(const Call& c, Buffers& B) {
  const uint32_t KB = c.cols / 256u, rows = jma::qact_tiles(c.batch) * 32u;
  for (uint32_t b = 0; b < rows; ++b)
    for (uint32_t k = 0; k < c.cols; ++k) {
      B.act[jma::qact_index(b, k, c.cols)]++;
      B.act_class[jma::qact_class_index(b, k, c.cols)]++;
      if (k % 16 == 0) B.act_sum[jma::qact_sum_index(b, k / 256u, k % 256u / 16u, KB)]++;
      if (k % 256 == 0) B.act_scale_k[jma::qact_scale_index(b, k / 256u, KB)]++;
    }
  bool once = true;
  for (uint64_t i = 0; i < (uint64_t)rows * c.cols; ++i) once &= B.act[i] == 1 && B.act_class[i] == 1;
  for (uint64_t i = 0; i < (uint64_t)rows * KB * 16u; ++i) once &= B.act_sum[i] == 1;
  for (uint64_t i = 0; i < (uint64_t)rows * KB; ++i) once &= B.act_scale_k[i] == 1.0f;
  expect(once, c.name + ": every quantized activation, sum and scale once");
  const uint64_t values = (uint64_t)rows * c.cols * 2;
  for (uint32_t kind : {jma::kQactK, jma::kQactQ6, jma::kQactKAndQ6}) {
    const jma::QactLayout o = jma::qact_layout(jma::qact_elements(c.batch, c.cols), kind);
    const uint64_t after_act = kind & jma::kQactK ? values : 0, after_classes = kind & jma::kQactQ6 ? values : 0;
    expect(o.act == 0 && o.classes >= after_act && o.sums - o.classes >= after_classes &&
               o.scales - o.sums >= (kind & jma::kQactK ? (uint64_t)rows * KB * 32 : 0) &&
               o.total - o.scales >= (uint64_t)rows * KB * 4 && o.classes % 16 == 0 && o.sums % 16 == 0 &&
               o.scales % 16 == 0,
           c.name + ": activation scratch regions");
  }
}

// qmatvec_kernel / qkmatvec_kernel: the tile's weight units, the activation rows of each pass,
// the LDS arrays at their largest indices, every output.
void walk_pass(const Call& c, uint32_t fmt, const jma::QMatPlan& qp, Buffers& B) {
  const uint32_t K = c.cols / jma::qmat_block_elems(fmt);
  uint32_t tiles;
  const std::vector<M> ms = table(c, fmt, qp.rows_per_tile, tiles);
  const uint32_t R = qp.rows_per_tile, nc = qp.chunk;
  const uint32_t group_rows = jma::qmat_group_rows(c.batch, nc, tiles);
  const uint32_t gy = (c.batch + group_rows - 1) / group_rows;
  expect(group_rows % nc == 0 && gy <= 65535u, c.name + ": grid rows");
  const bool kq = jma::qmat_kquant(fmt);
  const uint64_t lds = kq ? jma::qkmatvec_lds_bytes(fmt, nc, c.cols, R) : jma::qmatvec_lds_bytes(nc, c.cols, R);
  expect(lds <= jma::kQMatLds, c.name + ": LDS");
  unsigned char* smem = new unsigned char[lds];
  const uint32_t nt = fmt == 3 ? 9u : 4u;
  for (uint32_t bx = 0; bx < tiles; ++bx) {
    uint32_t mi = 0;
    for (uint32_t i = 1; i < ms.size(); ++i) mi = bx >= ms[i].tile0 ? i : mi;
    const uint32_t idx = ms[mi].idx, rows = c.rows[idx];
    const uint32_t r0 = (bx - ms[mi].tile0) * R;
    expect(r0 < rows, c.name + ": tile past its matrix");
    const uint32_t nrows = std::min(R, rows - r0);
    const uint32_t bb = jma::qmat_block_bytes(fmt);
    for (uint32_t u = 0; u < nrows * K; ++u) {
      const uint64_t off = ((uint64_t)r0 * K + u) * bb;
      sink = sink + B.w[idx][off] + B.w[idx][off + bb - 1];
    }
    for (uint32_t by = 0; by < gy; ++by) {
      const uint32_t g0 = by * group_rows, g1 = std::min(c.batch, g0 + group_rows);
      for (uint32_t b0 = g0; b0 < g1; b0 += nc) {
        const uint32_t nb = std::min(nc, g1 - b0);
        for (uint32_t b = 0; b < nb; ++b)
          sink = sink + B.x[(uint64_t)(b0 + b) * c.cols] + B.x[(uint64_t)(b0 + b) * c.cols + c.cols - 1];
        uint64_t top;
        if (!kq) {
          const uint64_t Kp = K + 1;
          const uint64_t act = ((uint64_t)nc * c.cols + 15u) / 16u * 16u;
          top = act + (uint64_t)nc * K * 8u + ((uint64_t)(nb - 1) * R + (nrows - 1)) * Kp * 4u +
                (uint64_t)nc * R * Kp * 4u + K * 4u;  // t_dot[(b * R + row) * Kp + blk]
        } else {
          const uint64_t rs = (uint64_t)K * nt + 1;
          const uint64_t act = ((uint64_t)nc * c.cols + 15u) / 16u * 16u;
          top = act + (uint64_t)nc * K * 4u + (uint64_t)nc * (c.cols / 16u) * 4u +
                (((uint64_t)(nb - 1) * R + (nrows - 1)) * rs + (K - 1) * nt + nt - 1) * 4u + 4u;
        }
        expect(top <= lds, c.name + ": LDS index");
        smem[top - 1] = 0;
        for (uint32_t b = 0; b < nb; ++b)
          for (uint32_t row = 0; row < nrows; ++row) {
            const uint32_t r = r0 + row;
            const uint64_t o = (uint64_t)(b0 + b) * rows + r;
            if (c.addend_mode == 1) sink = sink + B.add[idx][r];
            if (c.addend_mode == 2) sink = sink + B.add[idx][o];
            B.written[ms[mi].out_off + o]++;
          }
      }
    }
  }
  delete[] smem;
}

void walk(const Call& c) {
  const uint32_t n = (uint32_t)c.formats.size();
  const bool kq = jma::qmat_kquant(c.formats[0]);
  const uint32_t K = c.cols / jma::qmat_block_elems(c.formats[0]);
  Buffers B;
  B.w.resize(n);
  B.add.assign(n, nullptr);
  uint64_t total_rows = 0;
  for (uint32_t i = 0; i < n; ++i) {
    B.w[i] = new uint8_t[(uint64_t)c.rows[i] * K * jma::qmat_block_bytes(c.formats[i])];
    if (c.addend_mode == 1) B.add[i] = new float[c.rows[i]];
    if (c.addend_mode == 2) B.add[i] = new float[(uint64_t)c.batch * c.rows[i]];
    total_rows += c.rows[i];
  }
  B.x = new float[(uint64_t)c.batch * c.cols];
  B.written.assign(c.batch * total_rows, 0);
  if (gemm_format(c.formats[0], c.batch)) {
    const uint64_t rows32 = (uint64_t)jma::qact_tiles(c.batch) * 32u;
    B.act.assign(rows32 * c.cols, 0);
    if (kq) {
      B.act_class.assign(rows32 * c.cols, 0);
      B.act_sum.assign(rows32 * K * 16u, 0);
      B.act_scale_k.assign(rows32 * K, 0.0f);
      walk_quant_k(c, B);
    }
  }
  if (!kq && gemm_format(c.formats[0], c.batch)) {
    const uint64_t rows32 = (uint64_t)jma::qact_tiles(c.batch) * 32u;
    B.act_scale.assign(rows32 * K, 0);
    walk_quant(c, B);
  }
  std::vector<uint32_t> pass_fmts;
  for (uint32_t f : c.formats)
    if (!gemm_format(f, c.batch)) pass_fmts.push_back(f);
  jma::QMatPlan qp;
  if (!pass_fmts.empty()) {
    qp = jma::plan_qmat(pass_fmts.data(), (uint32_t)pass_fmts.size(), c.cols);
    expect(qp.rows_per_tile > 0 && qp.chunk >= 1 && qp.chunk <= jma::kQMatMaxChunk, c.name + ": plan");
  }
  std::string how;
  for (uint32_t fmt = 0; fmt <= 5; ++fmt) {
    if (std::find(c.formats.begin(), c.formats.end(), fmt) == c.formats.end()) continue;
    if (gemm_format(fmt, c.batch)) {
      {
        // Every workgroup tile the planner may choose, the chosen one into the written counts.
        std::vector<uint32_t> fmt_rows;
        for (uint32_t i = 0; i < n; ++i)
          if (c.formats[i] == fmt) fmt_rows.push_back(c.rows[i]);
        const uint32_t chosen = jma::plan_qgemm(fmt_rows.data(), (uint32_t)fmt_rows.size(), c.batch, 256);
        expect(chosen < jma::kQGemmShapes, c.name + ": product shape");
        for (uint32_t s = 0; s < jma::kQGemmShapes; ++s) {
          const std::vector<uint8_t> before = B.written;
          if (jma::qmat_kquant(fmt)) walk_qkgemm(c, fmt, jma::qgemm_shape(fmt, s), B);
          else walk_qgemm(c, fmt, jma::qgemm_shape(fmt, s), B);
          if (s != chosen) B.written = before;
        }
      }
      how += " fmt " + std::to_string(fmt) + ": product;";
    } else if (qp.rows_per_tile > 0) {
      walk_pass(c, fmt, qp, B);
      how += " fmt " + std::to_string(fmt) + ": " + std::to_string(qp.rows_per_tile) +
             " rows per tile, " + std::to_string(qp.chunk) + " per pass;";
    }
  }
  for (uint64_t i = 0; i < B.written.size(); ++i)
    if (B.written[i] != 1) {
      expect(false, c.name + ": output " + std::to_string(i) + " written " +
                        std::to_string(B.written[i]) + " times");
      break;
    }
  printf("%s (batch %u, cols %u):%s\n", c.name.c_str(), c.batch, c.cols, how.c_str());
  (void)kq;
  for (uint32_t i = 0; i < n; ++i) {
    delete[] B.w[i];
    delete[] B.add[i];
  }
  delete[] B.x;
}

// The product's tile: no batch of at most 32 rows pads its activation rows past 32, none of at most 64
// past 64 while that many 64 x 64 tiles fit the compute units; large launches keep the large tile.
void check_tiles() {
  auto rows_b = [](uint32_t batch, uint32_t rows) {
    return jma::qgemm_rows_b(jma::kQGemmShape[jma::plan_qgemm(&rows, 1, batch, 256)]);
  };
  for (uint32_t rows : {1u, 64u, 2048u, 16300u, 16384u, 20000u, 131072u})
    for (uint32_t batch : {16u, 17u, 31u, 32u})
      expect(rows_b(batch, rows) == 32, "32-row tiles: " + std::to_string(batch) + " x " + std::to_string(rows));
  for (uint32_t rows : {1u, 64u, 2048u, 16300u, 16384u})
    for (uint32_t batch : {33u, 48u, 64u})
      expect(rows_b(batch, rows) == 64, "64-row tiles: " + std::to_string(batch) + " x " + std::to_string(rows));
  expect(rows_b(64, 32768) == 128 && rows_b(65, 16384) == 128 && rows_b(1000, 3072) == 128 &&
             rows_b(512, 3072) == 64 && rows_b(77, 2048) == 64,
         "tiles of larger launches");
}

// Scratch held after a product call: enough for itself and for any of at most as many activations (up to
// 65536 inputs), of any kind of K-quants after one of them; from 64 MiB on no more than that, with 31 rows
// of 65536 inputs to spare.
void check_scratch() {
  const uint32_t shapes[][2] = {{16, 256}, {17, 4096}, {31, 65536}, {77, 2048}, {1000, 3072}, {2048, 8192}, {4096, 8192}, {16384, 8192}};
  for (bool kq : {false, true})
    for (const auto& a : shapes) {
      const std::string at = "scratch of " + std::to_string(a[0]) + " x " + std::to_string(a[1]) + (kq ? ", K" : "");
      const uint64_t held = jma::qact_reserve_bytes(a[0], a[1], kq), n = (uint64_t)a[0] * a[1];
      for (uint32_t cols = 256; cols <= 65536; cols += 256) {
        const uint64_t batch = n / cols;
        if (batch < jma::kQGemmMinBatch) break;
        for (uint32_t kind = 0; kind <= (kq ? 3u : 0u); ++kind) {
          const uint64_t need = jma::qact_layout(jma::qact_elements((uint32_t)batch, cols), kind).total;
          expect(need <= held, at + ": room for " + std::to_string(batch) + " x " + std::to_string(cols));
        }
      }
      const uint64_t per64 = kq ? 265 : 132;  // bytes per 64 activations
      expect(held <= std::max<uint64_t>(64u << 20, (n + 31 * 65536) * per64 / 64 + 4096), at + ": no more than needed");
    }
}

}  // namespace

int main() {
  check_tiles();
  check_scratch();
  const std::vector<Call> calls = {
      // decode shapes: Llama-3.2-1B Q/K/V and wo, Qwen2 with biases
      {"llama1b qkv decode", {1, 0, 0}, {2048, 512, 512}, 1, 2048, 0},
      {"llama1b wo + residual", {0}, {2048}, 1, 2048, 2},
      {"qwen2 qkv biases", {1, 1, 1}, {896, 128, 128}, 1, 896, 1},
      // prefill-sized grouped calls with biases and residuals (the 200-row shape included)
      {"grouped 200 rows, biases", {1, 0, 0}, {1024, 256, 256}, 200, 1024, 1},
      {"wo 200 rows, residual", {0}, {1024}, 200, 1024, 2},
      {"grouped 2048 rows, biases", {1, 5, 0}, {3072, 1024, 1024}, 2048, 3072, 1},
      {"Q5_K_M 300 rows", {4, 4, 3}, {2048, 512, 512}, 300, 2048, 0},
      {"Q4_K_M 129 rows, residual", {2, 2, 3}, {1536, 256, 256}, 129, 1536, 2},
      {"Q4_K_M 2048 rows, biases", {2, 2, 3}, {3072, 1024, 1024}, 2048, 3072, 1},
      // edges: one block, one row, ragged batches, wide rows, 16 matrices
      {"one block", {0}, {1}, 1, 32, 0},
      {"odd blocks", {5}, {17}, 13, 2080, 1},
      {"wide row", {3}, {64}, 9, 14336, 2},
      {"wide row 32-element", {1}, {64}, 9, 14336, 0},
      {"wide row K-quant product", {2, 4}, {70, 3}, 40, 14336, 1},
      {"sixteen matrices", std::vector<uint32_t>(16, 0), std::vector<uint32_t>(16, 100), 33, 512, 1},
      {"batch 8", {0, 1}, {3072, 3}, 8, 2048, 0},
      {"batch 9", {0, 1}, {3072, 3}, 9, 2048, 0},
      {"batch 16 (product)", {5, 1}, {17, 65}, 16, 2080, 2},
      {"batch 15 (passes)", {5, 1}, {17, 65}, 15, 2080, 2},
      {"ragged product 100 x 200", {0, 5}, {200, 7}, 100, 96, 1},
      {"K-quant product 17 x 65 rows", {4, 2}, {17, 65}, 17, 512, 2},
      {"Q6_K product 33 x 70 rows", {3, 2, 3}, {70, 33, 1}, 33, 768, 1},
      {"wide row Q6_K product", {3}, {65}, 20, 14336, 2},
  };
  for (const Call& c : calls) walk(c);
  if (failures) {
    printf("%d failures\n", failures);
    return 1;
  }
  printf("ok\n");
  return 0;
}
