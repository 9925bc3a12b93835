// Decode launch planning and the index formulas of the decode split exchange, shared by the host
// runtime (jma_runtime.cpp), the kernels (jma_kernels.hip) and a CPU bounds check
// (tests/plan_check.cpp); and the launch planning of the quantized projections (jma_quant.hip,
// checked by tests/qmat_check.cpp). Plain C++: no HIP types, so it also builds with g++ alone.
#pragma once

#include <stdint.h>

#include <algorithm>

#if defined(__HIPCC__)
#define JMA_HD __host__ __device__ inline
#else
#define JMA_HD inline
#endif

namespace jma {

// Rows handled by one launch when their (sequence, position) pairs are passed as kernel
// arguments; larger batches are split into several launches by the runtime.
constexpr int kMaxRows = 128;
// Waves per decode workgroup at head dimension dk: the waves of one workgroup share a split and
// combine in LDS. Two waves per SIMD hide each other's instruction latency; at dk = 256 two tile
// buffers take half the register file, so one wave per SIMD.
constexpr int decode_waves(int dk) { return dk >= 256 ? 4 : 8; }
// Most splits one decode row may be cut into when the decode kernel reduces them itself (the
// reducing workgroup loads every split's partial); and when a separate reduce_kernel does
// (partials in part_acc / part_ml, reduced by one workgroup per head and 64 output elements).
constexpr int kMaxSplits = 32;
constexpr int kMaxWideSplits = 1024;
// Query heads one decode workgroup serves (the 16 MFMA columns); partial buffers reserve this
// many head slots per work item.
constexpr int kHeadSlots = 16;
// Fewest K/V bytes a decode split streams when the planner chooses its size (plan_decode).
constexpr uint64_t kMinSplitBytes = 96 * 1024;

// Storage block (slots) of the transposed V layout, and of the K tiles.
JMA_HD int v_block(bool f16) { return f16 ? 32 : 16; }

// K layout inside one (sequence, layer, kv head) region of cap * key_length elements: blocks of
// B = v_block slots, each stored as key_length / W column panels of B rows x W elements, where a
// panel row is 64 bytes (W = 32 f16 or 16 f32 elements). One matrix-core operand load of a tile
// (16 or 32 rows x 64 bytes across a wave) is then 1 KB of contiguous memory; row-major rows
// would spread it over 16 separate 64-byte pieces, which a compute unit issues 2-3x slower. A
// key length that is not a multiple of W keeps the rows whole (W = key_length).
JMA_HD uint32_t k_panel(uint32_t key_length, bool f16) {
  const uint32_t w = f16 ? 32u : 16u;
  return key_length % w == 0 ? w : key_length;
}
// Element offset of K element e of slot `slot` in its region.
JMA_HD uint64_t k_index(uint32_t slot, uint32_t e, uint32_t key_length, bool f16) {
  const uint32_t b = (uint32_t)v_block(f16), w = k_panel(key_length, f16);
  return (uint64_t)(slot - slot % b) * key_length + (uint64_t)(e / w) * (b * w) +
         (uint64_t)(slot % b) * w + e % w;
}

JMA_HD uint32_t first_visible(uint32_t position, uint32_t window) {
  // LlamaConfig.attentionStartPosition, causal branch (llama/LlamaConfig.java:184-195).
  return (window == 0 || position + 1 <= window) ? 0u : position + 1 - window;
}

// First work item of the group (row, rest = kv head * head groups + head group) whose ns splits
// are items item0 .. item0 + ns - 1. ns_uniform > 0: every row has ns_uniform splits; else row
// `row` starts at item_start_row.
JMA_HD uint64_t group_item0(uint32_t ns_uniform, uint32_t item_start_row, uint32_t row,
                            uint32_t hkv, uint32_t hgroups, uint32_t rest, uint32_t ns) {
  return ns_uniform ? ((uint64_t)row * hkv * hgroups + rest) * ns
                    : (uint64_t)item_start_row + (uint64_t)rest * ns;
}

// Arrival-ticket counter of a group: [row][kv head][head group].
JMA_HD uint64_t group_counter(uint32_t row, uint32_t hkv, uint32_t kvh, uint32_t hgroups, uint32_t hg) {
  return ((uint64_t)row * hkv + kvh) * hgroups + hg;
}

// Fused exchange: float index of element e (e < dv; e = dv is m, dv + 1 is l) of head slot hs of
// work item `item`; each (item, head slot) holds dv + 4 floats.
JMA_HD uint64_t fused_part_float(uint64_t item, uint32_t hs, uint32_t dv, uint32_t e) {
  return (item * kHeadSlots + hs) * (dv + 4) + e;
}
// Separate reduction: element e of head slot hs of item in part_acc, and its (m, l) in part_ml.
// With column slices, the slices of one head group write their columns into a single DV-wide
// item: the item of (row, kv head, head group, split) in the plan without slices, which is the
// group's virtual item numbering with `hgroups` / slices groups and the row's first item / slices
// (every row holds slices times the items it would hold unsliced). reduce_kernel reads it as an
// unsliced plan's.
JMA_HD uint64_t sep_item(uint32_t ns_uniform, uint32_t item_start_row, uint32_t row, uint32_t hkv,
                         uint32_t hgroups, uint32_t slices, uint32_t kvh, uint32_t hg, uint32_t ns,
                         uint32_t split) {
  const uint32_t hgr = hgroups / slices;
  return group_item0(ns_uniform, item_start_row / slices, row, hkv, hgr, kvh * hgr + hg, ns) + split;
}
JMA_HD uint64_t sep_acc_float(uint64_t item, uint32_t hs, uint32_t dv, uint32_t e) {
  return (item * kHeadSlots + hs) * dv + e;
}
JMA_HD uint64_t sep_ml_float(uint64_t item, uint32_t hs) { return (item * kHeadSlots + hs) * 2; }

// Split plan of one decode launch of `count` <= kMaxRows rows at positions[]: every workgroup
// streams tiles_per_split tiles, at least tiles_per_wave per wave, raised until the launch is near
// target_blocks workgroups and no row needs more than kMaxSplits splits (the decode kernel then
// reduces the splits itself). When that cap would leave the launch with fewer than a quarter of
// the target workgroups (few long rows: one sequence at a long context with few KV heads), rows
// are cut wider, up to kMaxWideSplits splits, and reduce_kernel combines them (`separate`); a
// context running separate kernels (`unfused`) always does.
//
// Column slices: at head dim 256 or 512 a launch of few workgroups (short rows: a sliding-window
// layer) cuts each head's value columns among `slices` = 4 workgroups, each computing q.K over its
// tiles and V and the output for a quarter of the columns. That gives four times the workgroups,
// each streaming K and a quarter of V (instead of all of V), with a quarter of the partials to
// exchange per split. The slices are virtual head groups: `hgroups` is head groups x slices. At
// head dim 512 a plan takes four slices when the sliced launch stays within half the target,
// else none (two slices, which read K twice, measured 27.5 against 22.6 us for one row at
// 32 704 positions); wide plans' slices share the separate reduction's items (sep_item).
struct DecodePlan {
  uint32_t hgroups = 0, slices = 1, tiles_per_split = 0, total_items = 0, max_splits = 0, ns_uniform = 0;
  bool any_split = false, separate = false;
  uint32_t nsplit[kMaxRows] = {};
  uint32_t item_start[kMaxRows + 1] = {};
  uint64_t part_f_bytes = 0, counter_bytes = 0, acc_bytes = 0, ml_bytes = 0;
};

inline DecodePlan plan_decode(uint32_t count, const uint32_t* positions, uint32_t window,
                              uint32_t hkv, uint32_t group, int dk, int dv, bool f16,
                              int target_blocks, int tiles_per_wave, bool unfused,
                              int min_split_tiles = 0) {
  DecodePlan p;
  const uint32_t blk = (uint32_t)v_block(f16);
  p.hgroups = (group + kHeadSlots - 1) / kHeadSlots;
  uint32_t ntiles[kMaxRows];
  uint64_t units = 0;
  uint32_t max_tiles = 0;
  for (uint32_t i = 0; i < count; ++i) {
    const uint32_t pos = positions[i];
    const uint32_t first = first_visible(pos, window);
    ntiles[i] = pos / blk - first / blk + 1;
    max_tiles = std::max(max_tiles, ntiles[i]);
    units += (uint64_t)ntiles[i] * hkv * p.hgroups;
  }
  const uint64_t target = (uint64_t)std::max(target_blocks, 1);
  const uint64_t tile_bytes = (uint64_t)blk * (uint64_t)(dk + dv) * (f16 ? 2u : 4u);
  uint64_t tps = min_split_tiles > 0 ? (uint64_t)min_split_tiles
                                     : (uint64_t)decode_waves(dk) * (uint64_t)std::max(tiles_per_wave, 1);
  // Every split streams at least kMinSplitBytes: a split's exchange (its partial stored, polled and
  // combined) costs about as much as streaming that many bytes through one compute unit, so
  // smaller splits add exchange work without saving time. One tile per wave already streams that
  // much at head dim 128 and above; at 64 and below the split takes more tiles (C2, d 64: 12
  // tiles, 11 splits, 7.6 against 8.1 us per launch with 8 tiles, 17 splits).
  if (min_split_tiles == 0) tps = std::max<uint64_t>(tps, (kMinSplitBytes + tile_bytes - 1) / tile_bytes);
  const uint64_t base_tps = tps;
  tps = std::max<uint64_t>(tps, (units + target - 1) / target);
  const uint64_t tps_fused = std::max<uint64_t>(tps, (max_tiles + kMaxSplits - 1) / kMaxSplits);
  bool wide = false;
  if (tps_fused > tps && !unfused) {
    uint64_t fused_items = 0;
    for (uint32_t i = 0; i < count; ++i)
      fused_items += (ntiles[i] + tps_fused - 1) / tps_fused * hkv * p.hgroups;
    wide = fused_items * 4 < target;
  }
  tps = wide ? std::max<uint64_t>(tps, (max_tiles + kMaxWideSplits - 1) / kMaxWideSplits)
             : tps_fused;
  // Short rows: a launch of few workgroups (under an eighth of the target) that each stream more
  // than 64 KB waits on the per-CU load issue rate (~64 KB per us), so it takes half the tiles
  // per split (at least one per two waves) and twice the workgroups, as long as each extra
  // split's partial (dv + 4 floats per query head, read back by the reducer) stays within 2 KB.
  const uint64_t part_bytes = (uint64_t)std::min<uint32_t>(group, kHeadSlots) * (dv + 4) * 4;
  if (min_split_tiles == 0 && !wide && tps == base_tps && tps >= 2 && tps * tile_bytes > 65536 &&
      part_bytes <= 2048 && (max_tiles + tps / 2 - 1) / (tps / 2) <= (uint64_t)kMaxSplits) {
    uint64_t few = 0;
    for (uint32_t i = 0; i < count; ++i) few += (ntiles[i] + tps - 1) / tps * hkv * p.hgroups;
    if (few * 8 < target) tps /= 2;
  }
  // Column slices (above): fused plans of at most one tile per wave at head dim 256 (the sliced
  // instance keeps one tile buffer) whose sliced launch stays within half the target; at 512, four
  // slices under the same rule.
  if (!unfused && dk == dv &&
      (dk == 512 || (!wide && dk == 256 && tps <= (uint64_t)decode_waves(dk)))) {
    uint64_t n = 0;
    for (uint32_t i = 0; i < count; ++i) n += (ntiles[i] + tps - 1) / tps * hkv * p.hgroups;
    if (n * 4 * 2 <= target) {
      p.slices = 4;
      p.hgroups *= 4;
    }
  }
  p.tiles_per_split = (uint32_t)tps;
  uint32_t items = 0;
  bool uniform = true;
  for (uint32_t i = 0; i < count; ++i) {
    p.item_start[i] = items;
    p.nsplit[i] = (uint32_t)((ntiles[i] + tps - 1) / tps);
    p.any_split |= p.nsplit[i] > 1;
    uniform &= p.nsplit[i] == p.nsplit[0];
    p.max_splits = std::max(p.max_splits, p.nsplit[i]);
    items += p.nsplit[i] * hkv * p.hgroups;
  }
  p.item_start[count] = items;
  p.total_items = items;
  p.ns_uniform = uniform ? p.nsplit[0] : 0u;
  p.separate = p.any_split && (unfused || wide);
  if (p.separate) {
    p.acc_bytes = (uint64_t)items / p.slices * kHeadSlots * dv * 4;
    p.ml_bytes = (uint64_t)items / p.slices * kHeadSlots * 2 * 4;
  } else if (p.any_split) {
    p.part_f_bytes = (uint64_t)items * kHeadSlots * (dv / p.slices + 4) * 4;
    p.counter_bytes = (uint64_t)count * hkv * p.hgroups * 4;
  }
  return p;
}

// ---------------------------------------------------------------- split prefill units
//
// Work items of a prefill launch whose units (kernel 3b's stripes, kernel 3c's stripe pairs) run
// last-first (the longest causal ranges first), the trailing split_units of them as two items each
// (they come first), one per half of the unit's kv tiles [t0, t1); the first half is kPairLead
// tiles shorter (at least one tile; a split unit has two or more). Shared by the kernels, their
// launches (grid size) and a CPU check that every unit's tiles are covered exactly once.
constexpr uint32_t kPairLead = 2;  // tiles by which a split unit's first half is the shorter

struct SplitItem {
  uint32_t unit, half;
  bool split;
};
JMA_HD uint64_t split_items(uint32_t units, uint32_t split_units) {
  return (uint64_t)units + split_units;
}
JMA_HD SplitItem split_item(uint32_t units, uint32_t split_units, uint32_t item) {
  SplitItem r;
  r.split = item < 2 * split_units;
  r.half = r.split ? item & 1u : 0u;
  r.unit = units - 1 - (r.split ? item / 2 : item - split_units);
  return r;
}
// The item's tiles [tb, te) of its unit's [t0, t1).
JMA_HD void split_range(uint32_t t0, uint32_t t1, const SplitItem& it, uint32_t& tb, uint32_t& te) {
  const uint32_t n = t1 - t0;
  const uint32_t lead = n < kPairLead ? n : kPairLead;
  const uint32_t first = (n - lead) / 2 > 1u ? (n - lead) / 2 : 1u;
  const uint32_t tm = t0 + first;
  tb = it.split && it.half != 0u ? tm : t0;
  te = it.split && it.half == 0u ? tm : t1;
}

// ---------------------------------------------------------------- quantized projections
//
// Launch planning of the block-quantized projections (jma_quant.hip), shared by the runtime and a
// CPU bounds check (tests/qmat_check.cpp). A launch serves every matrix of one weight format:
// workgroup (x, y) takes rows_per_tile rows of one matrix (tiles in matrix order) and the
// activation rows y * group_rows .. + group_rows - 1, which pass through its LDS chunk rows at a
// time while the tile's weight blocks stay in its registers or caches.

// backend-native's weight codes (RS:150-161): 0 Q4_0, 1 Q8_0, 2 Q4_K, 3 Q6_K, 4 Q5_K, 5 Q5_0.
JMA_HD bool qmat_kquant(uint32_t fmt) { return fmt == 2 || fmt == 3 || fmt == 4; }
JMA_HD uint32_t qmat_block_elems(uint32_t fmt) { return qmat_kquant(fmt) ? 256u : 32u; }
// GGUF block bytes (RS:87-92).
JMA_HD uint32_t qmat_block_bytes(uint32_t fmt) {
  return fmt == 0 ? 18u : fmt == 1 ? 34u : fmt == 2 ? 144u : fmt == 3 ? 210u : fmt == 4 ? 176u : 22u;
}

// Dynamic LDS of one workgroup for `chunk` activation rows: Q8_0 activations, their scales and
// block sums, then the tile's (scale product, integer dot) terms per (activation row, tile row).
JMA_HD uint64_t qmatvec_lds_bytes(uint32_t chunk, uint32_t cols, uint32_t rows_per_tile) {
  const uint64_t K = cols / 32u;
  return ((uint64_t)chunk * cols + 15u) / 16u * 16u + (uint64_t)chunk * K * 8u +
         2u * (uint64_t)chunk * rows_per_tile * (K + 1u) * 4u;
}
// K-quants: Q8_K activations, scales and 16-element sums, then 4 (Q4_K, Q5_K) or 9 (Q6_K)
// floats per (activation row, tile row, 256-block).
JMA_HD uint64_t qkmatvec_lds_bytes(uint32_t fmt, uint32_t chunk, uint32_t cols, uint32_t rows_per_tile) {
  const uint64_t KB = cols / 256u, nt = fmt == 3 ? 9u : 4u;
  return ((uint64_t)chunk * cols + 15u) / 16u * 16u + (uint64_t)chunk * KB * 4u +
         (uint64_t)chunk * (cols / 16u) * 4u + (uint64_t)chunk * rows_per_tile * (KB * nt + 1u) * 4u;
}

constexpr uint64_t kQMatLds = 64u * 1024u;   // dynamic LDS a projection workgroup may take
constexpr uint32_t kQMatMaxChunk = 8;        // activation rows per pass
constexpr uint32_t kQMatTargetBlocks = 1024;  // workgroups a projection launch aims for

// Batches of at least kQGemmMinBatch activation rows run as a matrix product on the matrix cores
// (jma_qgemm.hip) over activations quantized once into scratch. The line is right for the square
// projections of small models (2048 x 2048, 15 rows: Q4_0 15 us in the matrix-vector kernel against 27, Q4_K
// 19 against 23); matrices of 4096 x 4096 cross between 8 and 15 rows (Q4_K 48 against 39 us at 8, Q4_0
// 64 against 48 at 15), and wide outputs gain from 2 rows on (28672 x 4096, 15 rows: Q4_0 409 against 51).
constexpr uint32_t kQGemmMinBatch = 16;

// Quantized activations of a product, as halves (the int8 values exactly) in the order the matrix
// ops read them: tiles of 32 activation rows; per tile, chunks of 16 inputs, each [k half h][row]
// [8 inputs], so the 64 lanes (32 h + row) of one operand load read 1 KB in order. Inside a run of
// 8 the second and third of every four inputs change places, the order in which nibbles and bytes
// of a word come out as pairs of halves. Element index of input k of row b:
JMA_HD uint64_t qact_index(uint32_t b, uint32_t k, uint32_t cols) {
  const uint32_t i = k % 8u, at = (i & ~3u) | ((i & 1u) << 1) | ((i >> 1) & 1u);
  return (uint64_t)(b / 32u) * 32u * cols + (uint64_t)(k / 16u) * 512u + ((k / 8u) % 2u) * 256u +
         (b % 32u) * 8u + at;
}
// The same for Q6_K weights: per 256-element block, the eight classes l of elements whose index
// within their 32-element run is l + 8 m, m < 4; per class, the block's two 128-element halves as
// chunks, each [run % 2][row][m / 2][run / 2][m % 2].
JMA_HD uint64_t qact_class_index(uint32_t b, uint32_t k, uint32_t cols) {
  const uint32_t e = k % 256u, hf = e / 128u, run = e / 32u % 4u, l = e % 8u, m = e / 8u % 4u;
  return (uint64_t)(b / 32u) * 32u * cols + (uint64_t)(k / 256u) * 8192u + (l * 2u + hf) * 512u +
         (run % 2u) * 256u + (b % 32u) * 8u + (m / 2u) * 4u + (run / 2u) * 2u + m % 2u;
}
// Scale of block blk (of K per row) of row b.
JMA_HD uint64_t qact_scale_index(uint32_t b, uint32_t blk, uint32_t K) {
  return (uint64_t)(b / 32u) * 32u * K + (uint64_t)blk * 32u + b % 32u;
}
// Q8_K: sum i (of 16 elements each) of block blk, a matrix operand of 16 inputs per block.
JMA_HD uint64_t qact_sum_index(uint32_t b, uint32_t blk, uint32_t i, uint32_t KB) {
  return ((uint64_t)(b / 32u) * KB + blk) * 512u + (i / 8u) * 256u + (b % 32u) * 8u + i % 8u;
}
JMA_HD uint32_t qact_tiles(uint32_t batch) { return (batch + 31u) / 32u; }
// What a product call keeps of its activations in scratch, as offsets: the values (for any format but
// Q6_K), the values in Q6_K's order, the 16-element sums (Q4_K, Q5_K) and the scales. 32-element
// formats take 2 1/16 bytes per activation, Q4_K and Q5_K 2 9/64, Q6_K 2 1/64, a call of Q6_K and
// others 4 9/64, with the batch rounded up to 32 rows.
struct QactLayout {
  uint64_t act, classes, sums, scales, total;
};
enum QactKind : uint32_t { kQactBlocks = 0, kQactK = 1, kQactQ6 = 2, kQactKAndQ6 = 3 };  // bits: Q4_K / Q5_K, Q6_K
JMA_HD QactLayout qact_layout(uint64_t elements, uint32_t kind) {  // elements: 32-row tiles x cols
  const auto up = [](uint64_t bytes) { return (bytes + 255u) / 256u * 256u; };
  const uint64_t values = up(elements * 2u);
  QactLayout o;
  o.act = 0;
  o.classes = kind == kQactQ6 ? 0 : values;
  o.sums = o.classes + (kind & kQactQ6 ? values : 0);
  o.scales = o.sums + (kind & kQactK ? up(elements / 8u) : 0);
  o.total = o.scales + up(kind == kQactBlocks ? elements / 16u : elements / 64u);
  return o;
}
JMA_HD uint64_t qact_elements(uint32_t batch, uint32_t cols) { return (uint64_t)qact_tiles(batch) * 32u * cols; }
// Scratch to hold after a call where it can be had, so that a captured call of no more activations than
// an eager one before it, of up to kQactMaxCols inputs, never has to grow it: rounding a batch up to 32
// rows adds at most 31 rows and, from 16 rows on, at most doubles it. K-quant calls hold room for any
// mix of them, 32-element calls for these, within kQactAnyKind bytes for K-quants too.
constexpr uint64_t kQactMaxCols = 65536, kQactAnyKind = 64u << 20;
JMA_HD uint64_t qact_reserve_bytes(uint32_t batch, uint32_t cols, bool kq) {
  const uint64_t n = (uint64_t)batch * cols, own = qact_elements(batch, cols);
  const uint64_t others = n < 31u * kQactMaxCols ? 2u * n : n + 31u * kQactMaxCols;
  const uint64_t elements = own > others ? own : others;
  const uint64_t blocks = qact_layout(elements, kQactBlocks).total, any = qact_layout(elements, kQactKAndQ6).total;
  return kq || any <= kQactAnyKind ? any : blocks > kQactAnyKind ? blocks : kQactAnyKind;
}

// Workgroup tiles of the product: 32 bt nb activation rows x 32 wt nw weight rows on nb x nw
// waves of bt x wt 32 x 32 tiles each, half a weight block staged per thread and step.
struct QGemmShape {
  uint32_t bt, wt, nb, nw;
};
constexpr uint32_t qgemm_rows_b(QGemmShape s) { return 32u * s.bt * s.nb; }
constexpr uint32_t qgemm_rows_w(QGemmShape s) { return 32u * s.wt * s.nw; }
constexpr uint32_t qgemm_threads(QGemmShape s) { return 64u * s.nb * s.nw; }
constexpr uint32_t kQGemmShapes = 3;
constexpr QGemmShape kQGemmShape[kQGemmShapes] = {
    {2, 2, 2, 2},  // 128 x 128
    {1, 1, 2, 2},  // 64 x 64
    {1, 1, 1, 4},  // 32 x 128
};
// The tile of a format: Q5_K keeps a second set of integer sums, so its large tile is 128 x 64;
// Q6_K eight float chains per output, one 32 x 32 tile per wave (128 x 64 on eight waves).
constexpr QGemmShape kQ5KLargeShape{2, 1, 2, 2};
constexpr QGemmShape kQ6KShape{1, 1, 4, 2};
JMA_HD QGemmShape qgemm_shape(uint32_t fmt, uint32_t shape) {
  return fmt == 3 ? kQ6KShape : fmt == 4 && shape == 0 ? kQ5KLargeShape : kQGemmShape[shape];
}

// Tile (tx, ty) of workgroup `id` of a launch of `total` = tiles_w x batch tiles: the workgroups
// of one XCD (dispatch order modulo 8) take consecutive tiles, the weight tiles fastest, so that
// an XCD's L2 keeps the activations of few batch tiles. recip = qgemm_recip(tiles_w): the quotient
// by it is exact or one short, and stays on the scalar unit (a division goes through the vector
// unit's reciprocal, and the buffer descriptors made from it would be built in vector registers).
inline uint32_t qgemm_recip(uint32_t tiles_w) {
  return tiles_w <= 1 ? 0xFFFFFFFFu : (uint32_t)(((uint64_t)1 << 32) / tiles_w);
}
JMA_HD void qgemm_tile(uint32_t id, uint32_t tiles_w, uint32_t recip, uint32_t total, uint32_t& tx,
                       uint32_t& ty) {
  const uint32_t xcd = id % 8u, per = total / 8u, rem = total % 8u;
  const uint32_t t = xcd * per + (xcd < rem ? xcd : rem) + id / 8u;
  ty = (uint32_t)(((uint64_t)t * recip) >> 32);
  tx = t - ty * tiles_w;
  if (tx >= tiles_w) {
    tx -= tiles_w;
    ++ty;
  }
}

// The workgroup tile (index of kQGemmShape) of a product launch, of 4096 inputs in these times:
// 32-row tiles for batches that fit them, however many outputs (32 rows: 2048 outputs, Q5_0, 55 us,
// as 64 x 64 tiles; 16384 outputs 59 against 94 with 128 x 128 tiles; 128256 outputs 231 against 273,
// Q4_K 112 against 203, Q5_K 139 against 310); else 64 x 64 tiles while they fit the compute units once
// (64 rows, 16384 outputs, 256 tiles: Q5_0 57 us against 95, Q4_K 42 against 62); else the largest
// once they cover half the units. (Twice as many 64 x 64 tiles as units are level with the large ones
// or better in Q4_0 and Q4_K, 72 against 86 us and 57 against 63 at 128 x 16384, but slower in Q8_0
// and Q5_K by up to 14%; 1024 of them are slower in each, 1.26 to 1.82 times.) Q6_K has one tile.
inline uint32_t plan_qgemm(const uint32_t* rows, uint32_t count, uint32_t batch, uint32_t cus) {
  if (batch <= 32) return 2;
  uint64_t small = 0, large = 0;
  for (uint32_t i = 0; i < count; ++i) {
    small += (rows[i] + 63u) / 64u;
    large += (rows[i] + 127u) / 128u;
  }
  if (small * ((batch + 63u) / 64u) <= cus) return 1;
  return large * ((batch + 127u) / 128u) * 2 >= cus ? 0 : 1;
}

// Threads of a product launch over tiles_w weight tiles; one launch holds fewer than 2^32.
inline uint64_t qgemm_launch_threads(uint32_t fmt, uint32_t shape, uint64_t tiles_w, uint32_t batch) {
  const QGemmShape s = qgemm_shape(fmt, shape);
  return tiles_w * ((batch + (uint64_t)qgemm_rows_b(s) - 1) / qgemm_rows_b(s)) * qgemm_threads(s);
}

struct QMatPlan {
  uint32_t rows_per_tile = 0, chunk = 0;  // 0: cols too large for one workgroup's LDS
};

// Rows per tile (up to 512 (row, block) terms for the 32-element formats, two per thread; 64 for
// the K-quants, eight threads each) and activation rows per pass, the largest that keep every
// format of the call within kQMatLds.
inline QMatPlan plan_qmat(const uint32_t* formats, uint32_t count, uint32_t cols) {
  QMatPlan p;
  if (count == 0) return p;
  const bool kq = qmat_kquant(formats[0]);
  const uint32_t K = cols / qmat_block_elems(formats[0]);
  if (K == 0) return p;
  auto lds = [&](uint32_t chunk, uint32_t tile) {
    uint64_t m = 0;
    for (uint32_t i = 0; i < count; ++i)
      m = std::max(m, kq ? qkmatvec_lds_bytes(formats[i], chunk, cols, tile)
                         : qmatvec_lds_bytes(chunk, cols, tile));
    return m;
  };
  uint32_t tile = std::max<uint32_t>(1u, std::min<uint32_t>(64u, (kq ? 64u : 512u) / K));
  while (tile > 1 && lds(1, tile) > kQMatLds) tile /= 2;
  if (lds(1, tile) > kQMatLds) return p;
  uint32_t chunk = kQMatMaxChunk;
  while (chunk > 1 && lds(chunk, tile) > kQMatLds) --chunk;
  p.rows_per_tile = tile;
  p.chunk = chunk;
  return p;
}

// Activation rows per workgroup of a launch with `tiles` weight tiles: whole passes, as few as
// keep the launch near kQMatTargetBlocks workgroups (one pass each at decode batches).
JMA_HD uint32_t qmat_group_rows(uint32_t batch, uint32_t chunk, uint32_t tiles) {
  const uint64_t passes = (batch + chunk - 1) / chunk;
  uint64_t per = (passes * tiles + kQMatTargetBlocks - 1) / kQMatTargetBlocks;
  per = per < 1 ? 1 : (per > passes ? passes : per);
  return (uint32_t)(per * chunk);
}

}  // namespace jma
