// Definitions shared by the decode kernels (partitioned and balanced schedules).
#pragma once

#include "gk_mfma.hpp"
#include "work_order.hpp"

namespace gk {

// The MFMA kernels re-base their running max when a score exceeds it by more
// than this (log2 units), so probabilities stay <= 2^slack. At 0 every new
// maximum re-bases: the largest probability is exactly 1 and the bf16
// rounding of the others tracks the reference's normalised probabilities
// closely enough for its relative-L2 gate against the tiled reference
// (5e-3) on rows of a few keys; a slack of 8 (rarer re-bases) reached 6.4e-3
// there. GK_DECODE_RESCALE_SLACK selects another slack at build time.
#ifndef GK_DECODE_RESCALE_SLACK
#define GK_DECODE_RESCALE_SLACK 0
#endif
constexpr float kDecodeRescaleSlack = GK_DECODE_RESCALE_SLACK;

struct DecodeArgs {
  const uint16_t* query;
  int64_t q_stride;
  const uint16_t* pool;
  int64_t slots;
  const int32_t* block_tables;
  int64_t bt_stride;
  int32_t block_shift;
  const int32_t* row_request;
  const int32_t* row_context;
  const int32_t* row_map;
  int32_t rows, q_heads, kv_heads, group, head_groups, heads_per_group;
  float score_scale;  // scale * log2(e), or scale / softcap when capping
  float softcap_log2; // softcap * log2(e) when capping
  int32_t window, partition, max_parts;
  uint16_t* out;
  int64_t out_stride;
  float* part_o;
  float* part_ml;
  uint16_t* pool_out;  // the pool as a store target (decode_unit.hip)
};

template <int D>
struct MfmaShape {
  static constexpr int TS = D == 256 ? 16 : 32;   // keys per step
  static constexpr int TG = TS / 16;              // 16-key groups per step (QK tiles)
  static constexpr int NC = D / 32;               // 32-dim k chunks of Q.K
  static constexpr int CPR = D / 8;               // 16-byte chunks per head row
  static constexpr int LOADS = TS * CPR / 64;     // 16-byte loads per lane per tile
  static constexpr int NO = D / 16;               // 16-dim output chunks of P.V
  static constexpr int TILE = TS * D * 2;         // bytes of one K or V tile in LDS
};

// A row's tiles: visible keys [left, ctx) occupy tiles first .. first + count - 1.
// An empty row still owns one (fully masked) tile, so every unit is finalised.
struct RowTiles {
  int first, count, left, ctx;
};

template <int TS>
__device__ __forceinline__ RowTiles row_tiles(int ctx, int window) {
  RowTiles r;
  r.ctx = ctx > 0 ? ctx : 0;
  r.left = visible_left(r.ctx, window);
  r.first = r.left / TS;
  r.count = stream_row_tile_count(r.ctx, window, TS);
  return r;
}

// One workgroup per unit (decode_unit.hip): rows of at most this many visible
// keys (1 MiB of keys and values; at head_dim 64 what lets two workgroups share
// a CU's LDS), whose block-table entries, one more when a window starts inside
// a page, lie in LDS; and as many new rows with a fused store.
constexpr int unit_max_keys(int head_dim) { return head_dim == 64 ? 3072 : (1 << 18) / head_dim; }
constexpr int unit_short_keys(int waves) { return 128 * waves; }  // with fewer than eight waves
constexpr int kUnitMaxNewRows = 256;
bool unit_decode_fits(const gk_decode_params* params, int64_t units);
int launch_unit_decode(const DecodeArgs& a, bool softcap, int head_dim, const gk_decode_params* params, bool store,
                       hipStream_t stream);

// Balanced ("stream") decode schedule, head dims 64/128/256, GQA group >= 4,
// any block size. Workspace layout: part_o[2 * wgs][hpw][D],
// part_ml[2 * wgs][hpw][2] and unit_span[units] (int32 pairs).
int stream_decode_wgs(int head_dim, bool softcap, int block_size);
size_t stream_decode_workspace_bytes(int head_dim, int heads_per_group, int64_t units, int wgs);
int launch_stream_decode(const DecodeArgs& a, bool softcap, int head_dim, int wgs, void* workspace,
                         hipStream_t stream);

}  // namespace gk
