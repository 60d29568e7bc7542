// Chunked / prefix-shared paged prefill attention for gfx950 (bf16 MFMA).
//
// A sequence contributes a chunk of consecutive query rows at positions
// prefix .. prefix + rows - 1; row i attends keys [left_i, prefix + i] of its
// request (causal; left_i = prefix + i - window + 1 with a sliding window).
// The chunk's own K/V rows are already in the pool (the store runs first), so
// every key is read through the block table.
//
// Work decomposition. A workgroup of eight waves owns one (sequence, kv head,
// tile of rows), or with a work list (prefill_schedule.hpp) a range of such a
// tile's keys, whose partial result prefill_merge_kernel combines. The GQA group is folded into the tile: its 256 "query rows"
// (128 at head_dim 256) are (row, head) pairs, so one K/V tile serves every
// head of the group. Each wave computes 32 query rows (two 16-column MFMA
// tiles; one, 16 rows, at head_dim 256) against the keys of a step (64 at
// head_dim 128, 32 at head_dim 64 and 256):
//   S^T[key][qrow] = K . Q^T      v_mfma_f32_16x16x32_bf16, K from LDS
//   O[qrow][dim]  += P . V        P straight from S^T's registers, V read
//                                 transposed from LDS (ds_read_b64_tr_b16)
// A step's K and V tiles are shared by the eight waves through LDS: 16-byte
// buffer->LDS loads issued by the whole workgroup, XOR-swizzled by token,
// double-buffered so the next tile streams in while the current one is used.
// Online softmax runs in log2 units with a lazily re-based running maximum.
//
// Numerics versus the reference (the tile chain of
// src/bridge/paged_attention_tiles.cpp:57-195): fp32 scores times scale,
// probabilities rounded to bf16 before P.V (relative to the running maximum),
// fp32 accumulation, one normalisation at the end by the sum of those bf16
// probabilities, bf16 output.
#include "gk_mfma.hpp"
#include "prefill_schedule.hpp"
#include "work_order.hpp"

#include <algorithm>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

namespace gk {
namespace {

// Waves per workgroup (each owns 16 * kNT query rows). Eight, one workgroup
// per CU (two waves per SIMD): each K/V tile is loaded into LDS once for 256
// query rows instead of twice for two 128-row workgroups (C4, 64-key steps,
// same box: 180.0 -> 174.1 us with four -> eight waves; 168.8 us together with
// the early V reads below).
constexpr int kPrefillWaves = 8;
// 16-column query tiles per wave. Two at head_dim 64 and 128: three fit in 256
// VGPRs only without the early V reads, and four spill; both also quantise
// C4's rows badly (48- or 64-row tiles of 512-row chunks leave a partial round
// of workgroups). One at head_dim 256, whose output accumulators alone take 64
// VGPRs per tile: with two, every head_dim 256 instance spills 536-588 bytes
// per lane; four waves of two tiles (one wave per SIMD, accumulators in AGPRs,
// no spills) measured 163.6-164.7 -> 227.4-227.5 us on C4's shapes at head_dim
// 256: the second wave of a SIMD matters more than halving the operand reads.
constexpr int kNT = 2;
constexpr int kQrowsPerWave = 16 * kNT;
template <int D>
constexpr int prefill_nt() { return D > 128 ? 1 : kNT; }
static_assert(prefill_tile_qrows(64) == kPrefillWaves * 16 * prefill_nt<64>() &&
                  prefill_tile_qrows(128) == kPrefillWaves * 16 * prefill_nt<128>() &&
                  prefill_tile_qrows(256) == kPrefillWaves * 16 * prefill_nt<256>(),
              "the schedule's row tiles are the kernel's");
// Keys per step: 64 at head_dim 128 (half the per-step barriers, cross-lane
// maxima, re-base checks and load setup of 32-key steps: C4 178.1 -> 166.8
// us); 32 at head_dim 64, whose 64-key form needs 130 VGPRs and so would drop
// from four waves per SIMD to three, and at head_dim 256, where a 64-key K
// and V tile pair takes 64 KiB of LDS per stage.
template <int D>
constexpr int prefill_keys() { return prefill_step_keys(D); }
// K/V pipeline depth. Two: three and four stages measured the same on C4 (the
// kernel is bound by its instruction stream, not by load latency).
constexpr int kStages = 2;
constexpr float kLazyRescale = 8.f;
// XCDs of an MI355X: consecutive workgroups of a launch go to consecutive XCDs.
constexpr int kXcds = 8;

struct PrefillArgs {
  const uint16_t* query;
  int64_t q_stride;
  const uint16_t* pool;
  int64_t slots;
  const int32_t* block_tables;
  int64_t bt_stride;
  int32_t block_shift;
  const int32_t* seq_request;
  const int32_t* seq_first_row;
  const int32_t* seq_rows;
  const int32_t* seq_prefix;
  int32_t q_heads, kv_heads, group, rows_per_tile;
  int32_t tiles, seqs;  // row tiles per sequence; sequences
  float score_scale;   // scale * log2(e), or scale / softcap when capping
  float softcap_log2;  // softcap * log2(e) when capping
  int32_t window;
  uint16_t* out;
  int64_t out_stride;
  DivMagic tiles_div, seqs_div, group_div;  // division by tiles, seqs and group (work_order.hpp)
  // Work list (prefill_schedule.hpp) instead of the sequence arrays when not null.
  const int32_t* items;
  const int32_t* row_request;  // block-table row of each query row
  int32_t item_count;
  // XCD x serves the kv heads h with h % classes == x % classes, classes =
  // gcd(kv_heads, 8): class_heads = kv_heads / classes heads on class_xcds =
  // 8 / classes XCDs (class_shift = log2 classes).
  int32_t class_shift, class_heads, class_xcds;
  DivMagic class_heads_div;
  int32_t part_slots;          // partial slots of one kv head
  float* part_o;               // [kv head, slot][wave][query tile][16-dim chunk][lane] x 4 output rows
  float* part_ml;              // [kv head, slot][wave][query tile][2][16]: base (log2 units), sum
};

template <int D>
struct PrefillShape {
  static constexpr int NC = D / 32;                 // 32-dim k chunks of Q.K
  static constexpr int CPR = D / 8;                 // 16-byte chunks per head row
  static constexpr int NO = D / 16;                 // 16-dim output chunks
  static constexpr int TILE = prefill_keys<D>() * D * 2;  // bytes of one K or V tile
  static constexpr int NI = TILE / 1024;            // 1 KiB load instructions per tile
};

// How a step's slots are found (the MODE template argument):
//  kStepBlocks  blocks of at least a step's keys: one scalar block-table entry per step;
//  kLoadBlocks  blocks of >= 64 / (D / 8) keys (one load instruction's): one
//               scalar entry per load instruction;
//  kKeyBlocks   shorter blocks, down to the token-granular map (block 1): each
//               lane reads its own key's entry with a vector load.
constexpr int kStepBlocks = 0, kLoadBlocks = 1, kKeyBlocks = 2;

template <int D, bool SOFTCAP, int MODE>
__global__ __launch_bounds__(kPrefillWaves * 64, 1) void prefill_kernel(PrefillArgs a) {
  using S = PrefillShape<D>;
  // This head dimension's query tiles per wave (in place of the namespace's).
  constexpr int kNT = prefill_nt<D>(), kQrowsPerWave = 16 * kNT;
  constexpr int kKeys = prefill_keys<D>();
  static_assert(kKeys == 32 || kKeys == 64, "a step is one or two 32-key halves");
  constexpr int kKG = kKeys / 16;  // 16-key groups per step (Q.K tiles)
  constexpr int kKH = kKeys / 32;  // 32-key halves per step (P.V k chunks)
  // Load instructions per wave per K (or V) tile; wave w issues instructions w, w + waves, ...
  constexpr int LPW = (S::NI + kPrefillWaves - 1) / kPrefillWaves;
  constexpr int NE = MODE == kStepBlocks ? 1 : LPW;  // block-table entries per wave (per lane) per step
  constexpr int KPL = kKeys / S::NI;                 // keys of one load instruction
  constexpr bool CLAMPED = MODE != kStepBlocks;      // entries of keys outside [key_begin, key_end) clamped
  static_assert(MODE != kKeyBlocks || kStages == 2, "per-lane entries rely on the step's full drain");
  // kStages K/V stages. The direct loads are asm statements the compiler does
  // not track, so one array serves every stage; reads are ordered by the
  // explicit vmcnt wait and the barrier of each step.
  // A region of its own (after the stages) holds, after the step loop, each
  // wave's output rows in bf16 (rows padded by 16 bytes so that the four
  // q-groups' rows of a write fall on different banks), read back as 16-byte
  // pieces for the global stores. Being separate from the stages, a wave
  // starts its output as soon as its own last step ends, with no barrier
  // (132 KiB at head_dim 128, one workgroup per CU either way).
  constexpr int kOutRowBytes = 2 * D + 16;
  constexpr int kKvBytes = kStages * 2 * S::TILE,
                kOutBytes = kPrefillWaves * kQrowsPerWave * kOutRowBytes;
  __shared__ __attribute__((aligned(16))) char lds[kKvBytes + kOutBytes];
  auto kv = reinterpret_cast<char(*)[2][S::TILE]>(lds);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (LDS bases of the direct loads)
  const int q = lane >> 4, c16 = lane & 15;
  // Work item (row tile, sequence, kv head), row tiles fastest, kv heads
  // slowest. Workgroup b runs on XCD b % 8, so b is mapped to items with each
  // XCD taking one contiguous eighth of that order: the workgroups sharing a
  // kv head's K/V (every row tile of every sequence, which share the prefix)
  // run under one L2 instead of fetching it into all eight. Inside its share
  // an XCD takes the row tiles highest first (heavy_first_item).
  //
  // The prologue is a chain of scalar loads: the arguments, the sequence's
  // fields, its first block-table entry, then the first K/V tile. Each link is
  // a memory round trip, so every argument is materialised in one batch at the
  // top and the four sequence fields are loaded together ahead of the
  // early-exit test (the compiler would otherwise fetch the sequence pointers
  // after the work-item arithmetic and the fields one by one: six round trips
  // before the first K/V load instead of three).
  // A work list's record holds all of that in one load.
  const int g = a.group;
  const auto div_group = [&](int x) { return (int)fast_div((uint32_t)x, a.group_div); };
  int kvh, request, first_row, nr, pos_lo, key_begin, kb0, nsteps, slot = -1;
  if (a.items) {
    asm volatile("" ::"s"(a.items), "s"(a.row_request), "s"(a.item_count), "s"(a.class_shift), "s"(a.class_heads),
                 "s"(a.class_xcds), "s"(a.class_heads_div.mul), "s"(a.class_heads_div.shift), "s"(a.part_slots),
                 "s"(a.block_tables), "s"(a.query), "s"(a.pool), "s"(a.out), "s"(a.group), "s"(a.bt_stride),
                 "s"(a.block_shift), "s"(a.window), "s"(a.q_stride), "s"(a.slots), "s"(a.kv_heads),
                 "s"(a.group_div.mul), "s"(a.group_div.shift));
    // Item j of this XCD: the list is dealt out over the XCDs of the class,
    // longest items first, the class's kv heads side by side.
    const int xcd = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    const int jl = (int)fast_div((uint32_t)j, a.class_heads_div);
    const int li = jl * a.class_xcds + (xcd >> a.class_shift);
    kvh = (xcd & ((1 << a.class_shift) - 1)) + ((j - jl * a.class_heads) << a.class_shift);
    if (li >= a.item_count) return;
    const int32_t* rec = a.items + (int64_t)li * kPrefillItemWords;
    first_row = scalar_load(rec, 0);
    nr = scalar_load(rec, 1);
    pos_lo = scalar_load(rec, 2);
    const int key0 = scalar_load(rec, 3);
    nsteps = scalar_load(rec, 4);
    slot = scalar_load(rec, 5);
    request = scalar_load(a.row_request, first_row);
    // The list may be made for a wider window than the call's: steps that lie
    // before every row's window are skipped.
    const int left = a.window > 0 ? max(0, pos_lo - a.window + 1) : 0;
    kb0 = max(key0, left & ~(kKeys - 1));
    nsteps -= (kb0 - key0) / kKeys;
    key_begin = max(left, kb0);
    if (nsteps <= 0) {
      // No visible key in this piece (never a whole item): an empty partial,
      // whose output the merge does not read into its sums.
      if (slot >= 0 && lane < 16) {
        float* ml = a.part_ml + (((int64_t)kvh * a.part_slots + slot) * kPrefillWaves + wave) * (kNT * 32);
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) {
          ml[nt * 32 + lane] = -INFINITY;
          ml[nt * 32 + 16 + lane] = 0.f;
        }
      }
      return;
    }
  } else {
    asm volatile("" ::"s"(a.seq_rows), "s"(a.seq_prefix), "s"(a.seq_first_row), "s"(a.seq_request),
                 "s"(a.block_tables), "s"(a.query), "s"(a.pool), "s"(a.out), "s"(a.tiles), "s"(a.seqs),
                 "s"(a.rows_per_tile), "s"(a.group), "s"(a.bt_stride), "s"(a.block_shift), "s"(a.window),
                 "s"(a.q_stride), "s"(a.slots), "s"(a.kv_heads), "s"(gridDim.x), "s"(a.tiles_div.mul),
                 "s"(a.tiles_div.shift), "s"(a.seqs_div.mul), "s"(a.seqs_div.shift), "s"(a.group_div.mul),
                 "s"(a.group_div.shift));
    const int nitems = gridDim.x, xcd = blockIdx.x % kXcds, per_xcd = nitems / kXcds, extra = nitems % kXcds;
    // Divisions by runtime values go through the host's multiply-shift pairs.
    const auto div_tiles = [&](int x) { return (int)fast_div((uint32_t)x, a.tiles_div); };
    const int item = heavy_first_item(xcd * per_xcd + min(xcd, extra), per_xcd + (xcd < extra), a.tiles,
                                      (int)blockIdx.x / kXcds, div_tiles);
    const int item_seq = div_tiles(item), tile = item - item_seq * a.tiles;
    kvh = (int)fast_div((uint32_t)item_seq, a.seqs_div);
    const int seq = item_seq - kvh * a.seqs;
    const int rows = a.seq_rows[seq], prefix = a.seq_prefix[seq], seq_first = a.seq_first_row[seq];
    request = a.seq_request[seq];
    asm volatile("" ::"s"(rows), "s"(prefix), "s"(seq_first), "s"(request));
    const int r0 = tile * a.rows_per_tile;
    if (r0 >= rows) return;
    nr = min(a.rows_per_tile, rows - r0);
    first_row = seq_first + r0;
    pos_lo = prefix + r0;
    key_begin = a.window > 0 ? max(0, pos_lo - a.window + 1) : 0;
    kb0 = key_begin & ~(kKeys - 1);
    nsteps = (pos_lo + nr - kb0 + kKeys - 1) / kKeys;
  }
  const int32_t* __restrict__ bt = a.block_tables + (int64_t)request * a.bt_stride;
  // Keys of this workgroup: [key_begin, key_end), a whole item's or a piece's.
  const int key_end = min(pos_lo + nr, kb0 + nsteps * kKeys);

  // This lane's query rows (one per 16-column tile): qrow = (row, head).
  int qpos[kNT], qleft[kNT];
  bool qvalid[kNT];
  bf16x8_t qb[kNT][S::NC];
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt) {
    const int qr = wave * kQrowsPerWave + nt * 16 + c16;
    const int row = div_group(qr), head = qr - row * g;
    qvalid[nt] = row < nr;
    qpos[nt] = qvalid[nt] ? pos_lo + row : -1;
    qleft[nt] = a.window > 0 ? qpos[nt] - a.window + 1 : 0;
    const uint16_t* src = a.query + (int64_t)(first_row + row) * a.q_stride + (int64_t)(kvh * g + head) * D;
#pragma unroll
    for (int c = 0; c < S::NC; ++c) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (qvalid[nt]) v = load16(src + (4 * c + q) * 8);
      qb[nt][c] = __builtin_bit_cast(bf16x8_t, v);
    }
  }

  // Smallest query position and largest window start over this wave's valid rows.
  const int wave_pos_min = pos_lo + div_group(wave * kQrowsPerWave);
  const int wave_left_max =
      a.window > 0 ? pos_lo + min(nr - 1, div_group(wave * kQrowsPerWave + kQrowsPerWave - 1)) - a.window + 1 : 0;

  // At d 128 the row sums of the bf16 probabilities run on one more MFMA per
  // half step against an all-ones operand, in the output layout (rows 4q + r).
  // At d 64 the registers would drop the kernel from four waves per SIMD to
  // three, which costs more than it saves: each lane sums its query row on the
  // VALU (component 0 of l_run).
  constexpr bool kMfmaSum = D >= 128;
  // Step loop (below): at d 64 two groups of waves alternate between MFMA and
  // softmax phases (C4 shapes: 113.7 -> 104.8 us); at d 128 the same order
  // measured 158.9 -> 181.0 us, with or without the phase offset, so d 128
  // keeps one barrier per step with every wave in Q.K -> softmax -> P.V order.
  constexpr bool kPingPong = D < 128;
  f32x4_t o[kNT][S::NO];
  float m_run[kNT];
  // Without softcap the re-base check compares the raw score maximum with
  // (m_run + kLazyRescale) / scale, kept per tile and updated at each re-base:
  // the step's maximum is scaled only when a re-base is due.
  float m_thr[kNT];
  const float inv_scale = 1.f / a.score_scale;
  // The base the probabilities are formed against: m_run, or 0 while the row
  // has no maximum yet (kept with m_run, so a step does not select it).
  float m_base[kNT];
  f32x4_t l_run[kNT];
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt) {
#pragma unroll
    for (int c = 0; c < S::NO; ++c) o[nt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    m_run[nt] = -INFINITY;
    m_thr[nt] = -INFINITY;
    m_base[nt] = 0.f;
    l_run[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const uint16_t* kbase = a.pool + (int64_t)kvh * a.slots * D;
  const uint16_t* vbase = kbase + (int64_t)a.kv_heads * a.slots * D;
  const uint32_t region = (uint32_t)(a.slots * D * 2);
  // The unrolled d 128 loop passes the resources to the direct-load asm as
  // words made uniform with readfirstlane (the compiler keeps the opaque
  // resource in VGPRs there); d 64 keeps the builtin resource (1.8% faster).
  auto make_rsrc = [&](const uint16_t* base) {
    if constexpr (D < 128) return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, region, kBufferDword3);
    else return buffer_words(base, region);
  };
  using Rsrc = decltype(make_rsrc(kbase));
  const Rsrc krs = make_rsrc(kbase), vrs = make_rsrc(vbase);
  const int shift = a.block_shift, bmask = (1 << shift) - 1;

  // Block-table entries of the step at key tb (scalar loads, or per-lane
  // vector loads for kKeyBlocks, fetched a step ahead: the loop's wait before
  // its closing barrier covers them). With CLAMPED a key outside
  // [key_begin, key_end) takes the entry of the nearest such key.
  struct Entries {
    int e[NE];
  };
  auto entry_of = [&](int tb) __attribute__((always_inline)) {
    Entries en;
#pragma unroll
    for (int k = 0; k < NE; ++k) {
      int key = tb;
      if constexpr (MODE == kLoadBlocks) key += (wave + k * kPrefillWaves) * KPL;
      if constexpr (MODE == kKeyBlocks) key += (wave + k * kPrefillWaves) * KPL + lane / S::CPR;
      if constexpr (CLAMPED) key = min(max(key, key_begin), key_end - 1);
      if constexpr (MODE == kKeyBlocks) en.e[k] = bt[key >> shift];
      else en.e[k] = scalar_load(bt, key >> shift);
    }
    return en;
  };
  // Byte offsets of this wave's direct loads for the step at tb, the same for
  // its K and its V tile. Steps are kKeys-aligned. Piece p = 64 ins + lane of
  // load instruction ins (wave ins % waves): token p / CPR, stored chunk
  // p % CPR holding the token's chunk (p % CPR) ^ swz(token, D / 8). A token
  // outside [key_begin, key_end) reads the row of the nearest token inside:
  // every row read is a stored token, so the masked keys' V rows are finite
  // and their zero probabilities contribute exactly zero (no zeroing pass).
  // The clamped token stays in the block of the entry used for it: blocks of
  // kKeys or more hold the whole step, shorter blocks whole load instructions
  // or (kKeyBlocks) the lane's own token, and clamping is monotone.
  struct Offsets {
    uint32_t v[LPW];
  };
  auto offsets_of = [&](int tb, const Entries& en) __attribute__((always_inline)) {
    Offsets of{};
    // One block holds the whole step: the clamped key's offset in the step
    // stays in [0, kKeys) (the first step starts at or below key_begin, the
    // last holds key_end - 1), so the slot is a scalar base plus that offset.
    const int lo = key_begin - tb, hi = key_end - 1 - tb;
    const uint32_t step_slot = ((uint32_t)en.e[0] << shift) + (uint32_t)(tb & bmask);
#pragma unroll
    for (int k = 0; k < LPW; ++k) {
      const int ins = wave + k * kPrefillWaves;
      if (S::NI % kPrefillWaves != 0 && ins >= S::NI) break;  // wave-uniform
      const int p = ins * 64 + lane, tt = p / S::CPR, pc = p % S::CPR;
      uint32_t slot;
      if constexpr (MODE == kStepBlocks) {
        slot = step_slot + (uint32_t)min(max(tt, lo), hi);
      } else {
        const int key = min(max(tb + tt, key_begin), key_end - 1);
        slot = (uint32_t)((en.e[k] << shift) | (key & bmask));
      }
      of.v[k] = slot * (2 * D) + ((pc ^ swz(tt, D / 8)) << 4);
    }
    return of;
  };
  auto issue = [&](const Offsets& of, Rsrc rs, char* tile) __attribute__((always_inline)) {
    // Per-lane entries are vector loads of the previous step, already complete
    // (the loop waits for every load before its closing barrier); say so to
    // the compiler.
    if constexpr (MODE == kKeyBlocks) wait_vmem_visible();
    const uint32_t base = lds_addr(tile);
#pragma unroll
    for (int k = 0; k < LPW; ++k) {
      const int ins = wave + k * kPrefillWaves;
      if (S::NI % kPrefillWaves != 0 && ins >= S::NI) break;  // wave-uniform
      if constexpr (D < 128) lds_dma16(base + ins * 1024, rs, of.v[k]);
      else lds_dma16_w(base + ins * 1024, rs, of.v[k]);
    }
  };

  // Scores of the current step and probabilities of the previous one.
  f32x4_t sc[kKG][kNT];
  bf16x8_t pa[kKH][kNT];

  // S^T = K.Q^T into sc: lane (q, c16) gets qrow c16 (+16 nt), keys tb + 16h + 4q + r.
  auto scores = [&](const char* kt) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < kKG; ++h) {
      const int tt = 16 * h + c16;
      bf16x8_t kr[S::NC];
#pragma unroll
      for (int c = 0; c < S::NC; ++c)
        kr[c] = *reinterpret_cast<const bf16x8_t*>(kt + tt * (2 * D) + (((4 * c + q) ^ swz(tt, D / 8)) << 4));
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        sc[h][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < S::NC; ++c) sc[h][nt] = mfma32(kr[c], qb[nt][c], sc[h][nt]);
      }
    }
  };

  // V operand c of P . V for the 32-key half hh of the V tile vt: keys
  // 32hh + 4q + (c16 >> 2) and 32hh + 16 + 4q + (c16 >> 2), dims
  // 16c + 4 (c16 & 3), read transposed.
  auto read_v = [&](const char* vt, int hh, int c) __attribute__((always_inline)) {
    const int lc = 2 * c + ((c16 & 3) >> 1);
    const int t0 = 32 * hh + 4 * q + (c16 >> 2), t1 = t0 + 16;
    const bf16x4_t v0 = lds_read_tr4(vt + t0 * (2 * D) + ((lc ^ swz(t0, D / 8)) << 4) + ((c16 & 1) << 3));
    const bf16x4_t v1 = lds_read_tr4(vt + t1 * (2 * D) + ((lc ^ swz(t1, D / 8)) << 4) + ((c16 & 1) << 3));
    return __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // O[qrow][dim] += P . V with pa and the V tile vt, and the row sums. The
  // first half's operands come from vfirst when the caller read them earlier.
  auto accumulate = [&](const char* vt, const bf16x8_t* vfirst, int nfirst = S::NO) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < S::NO; ++c) {
#pragma unroll
      for (int hh = 0; hh < kKH; ++hh) {
        const bf16x8_t v = (hh == 0 && vfirst && c < nfirst) ? vfirst[c] : read_v(vt, hh, c);
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) o[nt][c] = mfma32(pa[hh][nt], v, o[nt][c]);
      }
    }
    if constexpr (kMfmaSum) {
      const bf16x8_t ones = {(__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f,
                             (__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f};
#pragma unroll
      for (int hh = 0; hh < kKH; ++hh)
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) l_run[nt] = mfma32(pa[hh][nt], ones, l_run[nt]);
    }
  };

  // Online softmax of the step at tb: mask sc, form pa, re-base o and l_run.
  // A step whose keys every valid query row of this wave sees (below the
  // causal diagonal, inside the window) needs no per-element mask. Without
  // softcap the scale folds into the exponent: masked scores become -inf in
  // place (the same registers on both paths), the row maximum is taken on raw
  // scores (scale > 0), and p = exp2(fma(s, scale, -max)).
  auto softmax = [&](int tb) __attribute__((always_inline)) {
    const bool full = tb + kKeys - 1 <= wave_pos_min && tb >= wave_left_max;
    if constexpr (!SOFTCAP) mfma_results_ready(sc);
    // Mask, and each tile's row maximum over this lane's 4 kKG scores.
    float mx[kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      if constexpr (SOFTCAP) {
#pragma unroll
        for (int h = 0; h < kKG; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[h][nt][r] = soft_cap(sc[h][nt][r] * a.score_scale, a.softcap_log2);
      }
      if (!full) {
#pragma unroll
        for (int h = 0; h < kKG; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = tb + 16 * h + 4 * q + r;
            sc[h][nt][r] = (key <= qpos[nt] && key >= qleft[nt]) ? sc[h][nt][r] : -INFINITY;
          }
      }
      float t[4 * kKG];
#pragma unroll
      for (int i = 0; i < 4 * kKG; ++i) t[i] = sc[i >> 2][nt][i & 3];
      mx[nt] = tree_max(t);  // log2 units with softcap, raw scores without
    }
    // The probabilities of both tiles are formed right away against the
    // running maxima, before the cross-lane reduction of the steps' maxima,
    // which only decides afterwards whether a (rare) re-base is due; that
    // recomputes them against the new maximum. Same values as re-basing
    // first. Empty asm uses keep them above the re-base branch, which the
    // compiler would otherwise sink them into, behind the reduction (C4 shapes
    // at head_dim 64: 107.2 -> 105.4 us). One branch serves both tiles, so the
    // common path of a step is one basic block (head_dim 128: 156.3 ->
    // 154.9 us against a branch per tile).
    auto probabilities = [&](int nt, float base) __attribute__((always_inline)) {
      float ps[4 * kKG];
#pragma unroll
      for (int i = 0; i < 4 * kKG; ++i) {
        if constexpr (SOFTCAP) ps[i] = fast_exp2(sc[i >> 2][nt][i & 3] - base);
        else ps[i] = fast_exp2(__builtin_fmaf(sc[i >> 2][nt][i & 3], a.score_scale, -base));
      }
#pragma unroll
      for (int i = 0; i < 4 * kKG; ++i) pa[i >> 3][nt][i & 7] = (__bf16)ps[i];
      if constexpr (!kMfmaSum) {
        float l = 0.f;
#pragma unroll
        for (int i = 0; i < 4 * kKG; ++i) l += ps[i];
        return l;
      }
      return 0.f;
    };
    float lsum[kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      lsum[nt] = probabilities(nt, m_base[nt]);
#pragma unroll
      for (int hh = 0; hh < kKH; ++hh) {
        const auto w = __builtin_bit_cast(u32x4_t, pa[hh][nt]);
        asm volatile("" ::"v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
      }
    }
#pragma unroll
    for (int nt = 0; nt + 1 < kNT; nt += 2) col4_max2(mx[nt], mx[nt + 1]);
    if constexpr (kNT % 2) mx[kNT - 1] = col4_max(mx[kNT - 1]);
    bool any = false;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) any = any || (mx[nt] > (SOFTCAP ? m_run[nt] + kLazyRescale : m_thr[nt]));
    if (__builtin_amdgcn_ballot_w64(any)) {
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        if (!__builtin_amdgcn_ballot_w64(mx[nt] > (SOFTCAP ? m_run[nt] + kLazyRescale : m_thr[nt]))) continue;
        const float m_new = fmaxf(m_run[nt], SOFTCAP ? mx[nt] : mx[nt] * a.score_scale);
        const float alpha = m_run[nt] == -INFINITY ? 0.f : fast_exp2(m_run[nt] - m_new);
        m_run[nt] = m_new;
        m_thr[nt] = (m_new + kLazyRescale) * inv_scale;
        m_base[nt] = m_new == -INFINITY ? 0.f : m_new;
        if constexpr (!kMfmaSum) l_run[nt][0] *= alpha;
        // o rows are qrows 4q + r; qrow h's factor lives in lanes with c16 == h.
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float f = __int_as_float(__builtin_amdgcn_ds_bpermute((4 * q + r) << 2, __float_as_int(alpha)));
#pragma unroll
          for (int c = 0; c < S::NO; ++c) o[nt][c][r] *= f;
          if constexpr (kMfmaSum) l_run[nt][r] *= f;
        }
        lsum[nt] = probabilities(nt, m_base[nt]);
      }
    }
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      if constexpr (!kMfmaSum) l_run[nt][0] += lsum[nt];
  };

  static_assert(kStages == 2, "K and V alternate between two stages");
  if constexpr (!kPingPong) {
    // One barrier per step: before it each wave waits for its own loads of
    // the current stage; after it every wave's loads of the stage have landed
    // and every wave has finished the previous step, whose stage is refilled
    // with the next step. The first half's V operands are read before the
    // softmax, their LDS latency behind its arithmetic.
    Entries e_next{};
    {
      const Offsets first = offsets_of(kb0, entry_of(kb0));
      issue(first, krs, kv[0][0]);
      issue(first, vrs, kv[0][1]);
    }
    if (1 < nsteps) e_next = entry_of(kb0 + kKeys);
    if (__builtin_expect(div_group(wave * kQrowsPerWave) >= nr, 0)) {
      // All rows of this wave lie past the tile's last: it only loads its share
      // and keeps step, and the other wave of its SIMD has the matrix cores and
      // the LDS to itself (256 workgroups of 64 steps, half the waves active:
      // head_dim 128 113.9 -> 82.6 us, with softcap 189.8 -> 120.0; three
      // quarters 116.6 -> 110.6. A branch inside the loop below instead cost full
      // tiles 2%).
      for (int step = 0; step < nsteps; ++step) {
        wait_vmem<0>();
        __syncthreads();
        wait_vmem_visible();
        if (step + 1 < nsteps) {
          const int tb = kb0 + step * kKeys, next = (step + 1) & 1;
          const Offsets of = offsets_of(tb + kKeys, e_next);
          issue(of, krs, kv[next][0]);
          issue(of, vrs, kv[next][1]);
          if (step + 2 < nsteps) e_next = entry_of(tb + 2 * kKeys);
        }
      }
      return;
    }
    // The loop is unrolled over the two stages, so that every LDS address of a
    // step is a per-lane offset plus an immediate (stage, 16-key group, half):
    // ~44 fewer VALU instructions per wave and step (C4: 148.6 -> 138.0 us).
    // The lambdas are forced inline (with three call sites the compiler made
    // the softmax a real call with a stack frame) and the buffer resources go
    // to the direct-load asm as scalar words (make_rsrc).
    auto body = [&](int step, auto stage) __attribute__((always_inline)) {
      constexpr int cur = decltype(stage)::value, next = cur ^ 1;
      const int tb = kb0 + step * kKeys;
      wait_vmem<0>();
      __syncthreads();
      // Every load of this wave has landed; tell the compiler. Its wait-count
      // model does not see the asm direct loads or waits, so it still counts
      // the query loads before the loop (and, with per-lane entries, the entry
      // loads) as outstanding, and would put an s_waitcnt vmcnt(0) before
      // their first use in the step: after this step's direct loads, which it
      // would then wait for (C4: 185.2 -> 183.9 us).
      wait_vmem_visible();
      if (step + 1 < nsteps) {
        const Offsets of = offsets_of(tb + kKeys, e_next);
        issue(of, krs, kv[next][0]);
        issue(of, vrs, kv[next][1]);
        if (step + 2 < nsteps) e_next = entry_of(tb + 2 * kKeys);
      }
      scores(kv[cur][0]);
      if constexpr (D <= 128) {
        bf16x8_t vfirst[S::NO];
#pragma unroll
        for (int c = 0; c < S::NO; ++c) vfirst[c] = read_v(kv[cur][1], 0, c);
        softmax(tb);
        accumulate(kv[cur][1], vfirst);
      } else {
        // head_dim 256: half the V operands are read early (32 VGPRs; C4's
        // shapes at head_dim 256, same box: none 162.7-164.2 us, a quarter
        // 160.5-162.8, half 158.2-158.7, all 164.9-166.0).
        constexpr int NF = S::NO / 2;
        bf16x8_t vfirst[NF];
#pragma unroll
        for (int c = 0; c < NF; ++c) vfirst[c] = read_v(kv[cur][1], 0, c);
        softmax(tb);
        accumulate(kv[cur][1], vfirst, NF);
      }
    };
    int step = 0;
    for (; step + 1 < nsteps; step += 2) {
      body(step, std::integral_constant<int, 0>{});
      body(step + 1, std::integral_constant<int, 1>{});
    }
    if (step < nsteps) body(step, std::integral_constant<int, 0>{});
  } else {
    // Two groups of waves, one wave of each on every SIMD (waves w and w + 4
    // share a SIMD), take turns between the matrix cores and the vector ALU.
    // A wave's work per step is an MFMA phase M(i) (scores of step i, then
    // P.V of step i - 1) and a VALU phase S(i) (the softmax of step i), run as
    // M(0) S(0) M(1) S(1) ... M(n) with a barrier after each phase. The
    // second group passes one barrier before its first phase and the first
    // group one after its last, so the second runs every phase one barrier
    // interval later: between two barriers one wave of each SIMD is in an
    // MFMA phase while the other is in a softmax phase.
    //
    // LDS: a wave's iteration i reads K(i) (stage i % 2) and V(i - 1) (stage
    // (i - 1) % 2). At its start each wave issues its share of the direct
    // loads of K(i + 1) and V(i), into the stages that both groups last read
    // in iteration i - 1, and waits for them before the barrier that ends
    // interval 2i + 1 (the first group's second barrier of the iteration, the
    // second group's first), after which the first group reads them.
    const bool lead = wave < kPrefillWaves / 2;
    Entries e_next = entry_of(kb0);
    Offsets off_v = offsets_of(kb0, e_next);  // offsets of the step whose V is issued next
    issue(off_v, krs, kv[0][0]);
    if (1 < nsteps) e_next = entry_of(kb0 + kKeys);
    wait_vmem<0>();
    __syncthreads();
    wait_vmem_visible();  // as in the other loop: the query (and entry) loads have landed
    if (!lead) __syncthreads();
    for (int i = 0; i <= nsteps; ++i) {
      const int tb = kb0 + i * kKeys;
      if (i + 1 < nsteps) {
        const Offsets off_k = offsets_of(tb + kKeys, e_next);
        issue(off_k, krs, kv[(i + 1) & 1][0]);
        issue(off_v, vrs, kv[i & 1][1]);
        off_v = off_k;
        if (i + 2 < nsteps) e_next = entry_of(tb + 2 * kKeys);
      } else if (i + 1 == nsteps) {
        issue(off_v, vrs, kv[i & 1][1]);
      }
      if (i < nsteps) scores(kv[i & 1][0]);
      if (i > 0) accumulate(kv[(i - 1) & 1][1], nullptr);
      if (!lead) wait_vmem<0>();
      __syncthreads();
      if (i < nsteps) softmax(tb);
      if (lead) wait_vmem<0>();
      __syncthreads();
      wait_vmem_visible();
    }
    if (lead) __syncthreads();
  }

  if (slot >= 0) {
    // A piece: its accumulators, bases and sums as they stand in registers
    // (1 KiB stores; the merge kernel reads them back in the same layout).
    const int64_t pslot = (int64_t)kvh * a.part_slots + slot;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      const int t = wave * kNT + nt;  // 16-row tile of the workgroup
      if (div_group(16 * t) >= nr) break;
      f32x4_t* po = reinterpret_cast<f32x4_t*>(a.part_o) + ((pslot * (kPrefillWaves * kNT) + t) * S::NO) * 64 + lane;
#pragma unroll
      for (int c = 0; c < S::NO; ++c) po[c * 64] = o[nt][c];
      float* ml = a.part_ml + (pslot * (kPrefillWaves * kNT) + t) * 32;
      if (lane < 16) ml[lane] = m_run[nt];
      if constexpr (kMfmaSum) {
        if (c16 == 0) *reinterpret_cast<f32x4_t*>(ml + 16 + 4 * q) = l_run[nt];
      } else {
        const float l = col4_sum(l_run[nt][0]);
        if (lane < 16) ml[16 + lane] = l;
      }
    }
    return;
  }
  // Normalise into bf16 rows in LDS: o row 4q + r of tile nt, its sum in
  // l_run[nt][r] (MFMA sums) or in lane c16 == 4q + r after the cross-row sum
  // (VALU sums). Then each wave stores its own rows as 16-byte pieces: the
  // wave's LDS operations complete in order, so it reads back what it wrote.
  // (Stored straight from the MFMA layout, a lane's values are 2-byte
  // elements 32 bytes apart: 64 narrow stores per lane.)
  char* rows_lds = lds + kKvBytes + wave * kQrowsPerWave * kOutRowBytes;
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt) {
    float l = 0.f;
    if constexpr (!kMfmaSum) l = col4_sum(l_run[nt][0]);
    // The hardware reciprocal (within one fp32 ulp, far below the bf16
    // rounding that follows) instead of a full division; every row sum is at
    // least 1 (the row's maximum contributes at least 1).
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lr = kMfmaSum ? l_run[nt][r]
                                : __int_as_float(__builtin_amdgcn_ds_bpermute((4 * q + r) << 2, __float_as_int(l)));
      const float inv = lr > 0.f ? __builtin_amdgcn_rcpf(lr) : 0.f;
      __bf16* dst = reinterpret_cast<__bf16*>(rows_lds + (nt * 16 + 4 * q + r) * kOutRowBytes) + c16;
#pragma unroll
      for (int c = 0; c < S::NO; ++c) dst[16 * c] = (__bf16)(o[nt][c][r] * inv);
    }
  }
  constexpr int kPieces = kQrowsPerWave * D / 8;  // 16-byte pieces of the wave's rows
  static_assert(kPieces % 64 == 0, "whole pieces per lane");
#pragma unroll
  for (int i = 0; i < kPieces / 64; ++i) {
    const int piece = i * 64 + lane, ql = piece / (D / 8), part = piece % (D / 8);
    const int qr = wave * kQrowsPerWave + ql;
    const int row = div_group(qr), head = qr - row * g;
    const uint4 v = *reinterpret_cast<const uint4*>(rows_lds + ql * kOutRowBytes + part * 16);
    if (row < nr)
      *reinterpret_cast<uint4*>(a.out + (int64_t)(first_row + row) * a.out_stride + (int64_t)(kvh * g + head) * D +
                                part * 8) = v;
  }
}

// ---------------------------------------------------------------------------
// Merge of the items that a work list splits
// ---------------------------------------------------------------------------
struct PrefillMergeArgs {
  const int32_t* merges;  // PrefillMerge records
  int32_t part_slots, group, q_heads;
  DivMagic group_div;
  const float* part_o;
  const float* part_ml;
  uint16_t* out;
  int64_t out_stride;
};

// Bound by reading the partials (from the last-level cache mostly) and, for few
// of them, by the launch: 8 us for 256 partials of 128 KiB (4.2 TB/s), 15 us for
// 496 (4.4 TB/s), 7 us for 258 of 64 KiB. One wave per (split item, kv head, 16 query rows, 32
// dims): the partials are read as the pieces' lanes stored them, 1 KiB a load,
// the loads of up to eight parts in one memory round trip.
template <int D>
__global__ __launch_bounds__(64) void prefill_merge_kernel(PrefillMergeArgs a) {
  constexpr int kTiles = prefill_tile_qrows(D) / 16, NO = D / 16, CC = 2, kGroups = NO / CC;
  constexpr int kRowBytes = 16 * CC * 2 + 16;
  __shared__ __attribute__((aligned(16))) char lds[16 * kRowBytes];
  const int lane = threadIdx.x, q = lane >> 4, c16 = lane & 15;
  const int mi = blockIdx.x / (kTiles * kGroups), rest = blockIdx.x % (kTiles * kGroups);
  const int t = rest / kGroups, cg = rest % kGroups, kvh = blockIdx.y;
  const int32_t* rec = a.merges + (int64_t)mi * kPrefillMergeWords;
  const int first_row = scalar_load(rec, 0), nr = scalar_load(rec, 1), slot = scalar_load(rec, 2),
            parts = scalar_load(rec, 3);
  if ((int)fast_div((uint32_t)(16 * t), a.group_div) >= nr) return;
  const int64_t tile0 = ((int64_t)kvh * a.part_slots + slot) * kTiles + t;  // part p: + p kTiles
  f32x4_t m_run, l_run{0.f, 0.f, 0.f, 0.f}, acc[CC];
#pragma unroll
  for (int r = 0; r < 4; ++r) m_run[r] = -INFINITY;
#pragma unroll
  for (int c = 0; c < CC; ++c) acc[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto merge_parts = [&](auto batch) {
    constexpr int BATCH = decltype(batch)::value;
    for (int p0 = 0; p0 < parts; p0 += BATCH) {
      f32x4_t mp[BATCH], lp[BATCH], op[BATCH][CC];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        const int64_t tile = tile0 + (int64_t)min(p0 + u, parts - 1) * kTiles;
        mp[u] = *reinterpret_cast<const f32x4_t*>(a.part_ml + tile * 32 + 4 * q);
        lp[u] = *reinterpret_cast<const f32x4_t*>(a.part_ml + tile * 32 + 16 + 4 * q);
        const f32x4_t* po = reinterpret_cast<const f32x4_t*>(a.part_o) + (tile * NO + cg * CC) * 64 + lane;
#pragma unroll
        for (int c = 0; c < CC; ++c) op[u][c] = po[c * 64];
      }
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // Parts past the last (clamped duplicates) weigh nothing. A part
          // without a visible key has no output: its slot is not read into
          // the sum.
          const float mu = p0 + u < parts ? mp[u][r] : -INFINITY;
          const float mn = fmaxf(m_run[r], mu);
          const float fa = m_run[r] == -INFINITY ? 0.f : fast_exp2(m_run[r] - mn);
          const float fb = mu == -INFINITY ? 0.f : fast_exp2(mu - mn);
          l_run[r] = l_run[r] * fa + (mu == -INFINITY ? 0.f : lp[u][r] * fb);
#pragma unroll
          for (int c = 0; c < CC; ++c) acc[c][r] = acc[c][r] * fa + (mu == -INFINITY ? 0.f : op[u][c][r] * fb);
          m_run[r] = mn;
        }
      }
    }
  };
  if (parts <= 4) merge_parts(std::integral_constant<int, 4>{});
  else merge_parts(std::integral_constant<int, 8>{});
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float inv = l_run[r] > 0.f ? 1.f / l_run[r] : 0.f;
    __bf16* dst = reinterpret_cast<__bf16*>(lds + (4 * q + r) * kRowBytes) + c16;
#pragma unroll
    for (int c = 0; c < CC; ++c) dst[16 * c] = (__bf16)(acc[c][r] * inv);
  }
  // The wave's own LDS operations complete in order: 16 rows x 4 pieces of 16 bytes.
  static_assert(CC == 2, "one 16-byte piece per lane");
  const int ql = lane >> 2, part = lane & 3;
  const uint4 v = *reinterpret_cast<const uint4*>(lds + ql * kRowBytes + part * 16);
  const int qr = 16 * t + ql, row = (int)fast_div((uint32_t)qr, a.group_div), head = qr - row * a.group;
  if (row < nr)
    *reinterpret_cast<uint4*>(a.out + (int64_t)(first_row + row) * a.out_stride +
                              (int64_t)(kvh * a.group + head) * D + cg * (16 * CC) + part * 8) = v;
}

template <int D, int MODE>
void launch_mode(const PrefillArgs& a, bool softcap, dim3 grid, hipStream_t stream) {
  if (softcap) prefill_kernel<D, true, MODE><<<grid, kPrefillWaves * 64, 0, stream>>>(a);
  else prefill_kernel<D, false, MODE><<<grid, kPrefillWaves * 64, 0, stream>>>(a);
}

template <int D>
void launch(const PrefillArgs& a, bool softcap, int block_size, dim3 grid, hipStream_t stream) {
  constexpr int keys = prefill_keys<D>();
  if (block_size >= keys) launch_mode<D, kStepBlocks>(a, softcap, grid, stream);
  else if (block_size >= keys / PrefillShape<D>::NI) launch_mode<D, kLoadBlocks>(a, softcap, grid, stream);
  else launch_mode<D, kKeyBlocks>(a, softcap, grid, stream);
}

}  // namespace

namespace {

int validate(const gk_prefill_params* p, bool listed) {
  if (!p) return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: null parameters");
  if (p->struct_size != sizeof(gk_prefill_params))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: struct_size does not match this library's gk_prefill_params");
  if (p->head_dim != 64 && p->head_dim != 128 && p->head_dim != 256)
    return fail(GK_ERR_UNSUPPORTED, "gk_paged_prefill: head dimension must be 64, 128 or 256");
  if (p->q_heads <= 0 || p->kv_heads <= 0 || p->q_heads % p->kv_heads || p->q_heads / p->kv_heads > 128)
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: invalid head geometry (GQA group at most 128)");
  if (!is_pow2(p->block_size) || p->block_size > (1 << 20))
    return fail(GK_ERR_UNSUPPORTED, "gk_paged_prefill: block_size must be a power of two of at most 2^20");
  if (p->seqs < 0 || p->seqs > 65535 || p->max_rows < 0 || p->slots <= 0)
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: sequence count, rows or slots out of range");
  if (p->slots > (int64_t)(UINT32_MAX / 2) / p->head_dim)
    return fail(GK_ERR_UNSUPPORTED, "gk_paged_prefill: one kv head's K or V region must stay below 4 GiB");
  if (!(p->scale > 0.f) || !(p->scale < INFINITY) || !(p->softcap >= 0.f) || !(p->softcap < INFINITY))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: invalid scale or softcap");
  if (!listed && (p->seqs == 0 || p->max_rows == 0)) return GK_OK;
  if (!p->query || !p->pool || !p->block_tables || !p->out ||
      (!listed && (!p->seq_request || !p->seq_first_row || !p->seq_rows || !p->seq_prefix)))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: null pointer");
  const auto misaligned = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) != 0; };
  if (misaligned(p->query) || misaligned(p->pool) || misaligned(p->out) || (p->q_row_stride & 7) ||
      (p->out_row_stride & 7) || p->q_row_stride < (int64_t)p->q_heads * p->head_dim ||
      p->out_row_stride < (int64_t)p->q_heads * p->head_dim)
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: query/pool/out must be 16-byte aligned with full rows");
  return GK_OK;
}

// The arguments that do not depend on where the work comes from.
PrefillArgs common_args(const gk_prefill_params* p) {
  PrefillArgs a{};
  a.query = static_cast<const uint16_t*>(p->query);
  a.q_stride = p->q_row_stride;
  a.pool = static_cast<const uint16_t*>(p->pool);
  a.slots = p->slots;
  a.block_tables = p->block_tables;
  a.bt_stride = p->bt_stride;
  a.block_shift = log2_int(p->block_size);
  a.q_heads = p->q_heads;
  a.kv_heads = p->kv_heads;
  a.group = p->q_heads / p->kv_heads;
  a.rows_per_tile = prefill_tile_qrows(p->head_dim) / a.group;
  const bool softcap = p->softcap > 0.f;
  a.score_scale = softcap ? p->scale / p->softcap : p->scale * kLog2e;
  a.softcap_log2 = p->softcap * kLog2e;
  a.window = p->sliding_window > 0 ? p->sliding_window : 0;
  a.out = static_cast<uint16_t*>(p->out);
  a.out_stride = p->out_row_stride;
  a.group_div = div_magic((uint32_t)a.group);
  return a;
}

int launch_prefill(const gk_prefill_params* p, const PrefillArgs& a, int64_t workgroups, hipStream_t stream) {
  const dim3 grid((unsigned)workgroups);
  const bool softcap = p->softcap > 0.f;
  if (p->head_dim == 64) launch<64>(a, softcap, p->block_size, grid, stream);
  else if (p->head_dim == 128) launch<128>(a, softcap, p->block_size, grid, stream);
  else launch<256>(a, softcap, p->block_size, grid, stream);
  return hip_status(hipGetLastError(), "gk_paged_prefill launch");
}

// Workspace of a work list: the partial outputs, then (base, sum) of every row.
size_t list_output_bytes(const gk_prefill_params* p, const gk_prefill_list* list) {
  return (size_t)p->kv_heads * list->part_slots * prefill_tile_qrows(p->head_dim) * p->head_dim * sizeof(float);
}
size_t list_workspace_bytes(const gk_prefill_params* p, const gk_prefill_list* list) {
  return list_output_bytes(p, list) +
         (size_t)p->kv_heads * list->part_slots * prefill_tile_qrows(p->head_dim) * 2 * sizeof(float);
}

}  // namespace

int device_cus();

int paged_prefill(const gk_prefill_params* p, hipStream_t stream) {
  if (int rc = validate(p, false)) return rc;
  if (p->seqs == 0 || p->max_rows == 0) return GK_OK;
  PrefillArgs a = common_args(p);
  a.seq_request = p->seq_request;
  a.seq_first_row = p->seq_first_row;
  a.seq_rows = p->seq_rows;
  a.seq_prefix = p->seq_prefix;
  a.seqs = p->seqs;
  a.tiles = (p->max_rows + a.rows_per_tile - 1) / a.rows_per_tile;
  a.tiles_div = div_magic((uint32_t)a.tiles);
  a.seqs_div = div_magic((uint32_t)a.seqs);
  const int64_t items = (int64_t)a.tiles * p->kv_heads * p->seqs;
  if (items > (int64_t)1 << 30) return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill: too many rows");
  return launch_prefill(p, a, items, stream);
}

int paged_prefill_listed(const gk_prefill_params* p, const gk_prefill_list* list, void* workspace,
                         size_t workspace_bytes, hipStream_t stream) {
  if (int rc = validate(p, true)) return rc;
  if (!list || list->struct_size != sizeof(gk_prefill_list))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill_listed: struct_size does not match this library's gk_prefill_list");
  if (list->item_count < 0 || list->merge_count < 0 || list->part_slots < 0 || list->part_slots > (1 << 20) ||
      list->merge_count > (1 << 20))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill_listed: list counts out of range");
  if (list->item_count == 0) return GK_OK;
  if (!list->items || !list->row_request || (list->merge_count && !list->merges))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill_listed: null pointer");
  if (list->part_slots && (!workspace || workspace_bytes < list_workspace_bytes(p, list) ||
                           (reinterpret_cast<uintptr_t>(workspace) & 15)))
    return fail(GK_ERR_WORKSPACE, "gk_paged_prefill_listed: workspace too small or not 16-byte aligned (" +
                                      std::to_string(list_workspace_bytes(p, list)) + " bytes needed)");
  PrefillArgs a = common_args(p);
  a.items = list->items;
  a.item_count = list->item_count;
  a.row_request = list->row_request;
  int classes = kXcds;
  while (p->kv_heads % classes) classes /= 2;
  a.class_shift = log2_int(classes);
  a.class_heads = p->kv_heads / classes;
  a.class_xcds = kXcds / classes;
  a.class_heads_div = div_magic((uint32_t)a.class_heads);
  a.part_slots = list->part_slots;
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + list_output_bytes(p, list));
  const int64_t per_xcd = ((int64_t)list->item_count + a.class_xcds - 1) / a.class_xcds * a.class_heads;
  if (per_xcd * kXcds > (int64_t)1 << 30)
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_paged_prefill_listed: too many items");
  if (int rc = launch_prefill(p, a, per_xcd * kXcds, stream)) return rc;
  if (!list->merge_count) return GK_OK;
  PrefillMergeArgs m{};
  m.merges = list->merges;
  m.part_slots = list->part_slots;
  m.group = a.group;
  m.q_heads = p->q_heads;
  m.group_div = a.group_div;
  m.part_o = a.part_o;
  m.part_ml = a.part_ml;
  m.out = a.out;
  m.out_stride = a.out_stride;
  const int waves = prefill_tile_qrows(p->head_dim) / 16 * (p->head_dim / 32);
  const dim3 grid((unsigned)(list->merge_count * waves), (unsigned)p->kv_heads);
  if (p->head_dim == 64) prefill_merge_kernel<64><<<grid, 64, 0, stream>>>(m);
  else if (p->head_dim == 128) prefill_merge_kernel<128><<<grid, 64, 0, stream>>>(m);
  else prefill_merge_kernel<256><<<grid, 64, 0, stream>>>(m);
  return hip_status(hipGetLastError(), "gk_paged_prefill_listed merge launch");
}

int prefill_list_build(const int32_t* seq_first_row, const int32_t* seq_rows, const int32_t* seq_prefix, int32_t seqs,
                       int32_t q_heads, int32_t kv_heads, int32_t head_dim, int32_t sliding_window, bool cut,
                       int32_t* words, int64_t capacity, gk_prefill_list* list) {
  if (!list || list->struct_size != sizeof(gk_prefill_list))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_prefill_list_build: struct_size does not match this library's gk_prefill_list");
  if ((head_dim != 64 && head_dim != 128 && head_dim != 256) || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads ||
      q_heads / kv_heads > 128)
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_prefill_list_build: invalid head geometry");
  if (seqs < 0 || seqs > 65535 || capacity < 0 || (seqs && (!seq_first_row || !seq_rows || !seq_prefix)))
    return fail(GK_ERR_INVALID_ARGUMENT, "gk_prefill_list_build: invalid sequences");
  int64_t rows = 0;
  for (int32_t s = 0; s < seqs; ++s) {
    if (seq_rows[s] < 0 || seq_prefix[s] < 0 || seq_first_row[s] < 0 ||
        (int64_t)seq_prefix[s] + seq_rows[s] > INT32_MAX - 64)
      return fail(GK_ERR_INVALID_ARGUMENT, "gk_prefill_list_build: invalid sequences");
    rows += seq_rows[s];
  }
  if (rows > (1 << 20)) return fail(GK_ERR_INVALID_ARGUMENT, "gk_prefill_list_build: too many rows");
  try {
    std::vector<PrefillSeq> in(seqs);
    for (int32_t s = 0; s < seqs; ++s)
      in[s] = {seq_first_row[s], seq_rows[s], seq_prefix[s]};
    const int group = q_heads / kv_heads;
    const PrefillWorkList work =
        cut ? prefill_work_list(in.data(), seqs, group, kv_heads, head_dim, sliding_window, device_cus())
            : prefill_whole_list(in.data(), seqs, group, head_dim, sliding_window);
    list->item_count = (int32_t)work.items.size();
    list->merge_count = (int32_t)work.merges.size();
    list->part_slots = work.slots;
    const int64_t item_words = (int64_t)work.items.size() * kPrefillItemWords,
                  merge_words = (int64_t)work.merges.size() * kPrefillMergeWords;
    if (!words || capacity < item_words + merge_words)
      return fail(GK_ERR_WORKSPACE, "gk_prefill_list_build: the list needs " + std::to_string(item_words + merge_words) +
                                        " words");
    if (item_words) std::memcpy(words, work.items.data(), item_words * sizeof(int32_t));
    if (merge_words) std::memcpy(words + item_words, work.merges.data(), merge_words * sizeof(int32_t));
    return GK_OK;
  } catch (const std::bad_alloc&) {
    return fail(GK_ERR_OUT_OF_MEMORY, "gk_prefill_list_build: out of host memory");
  }
}

}  // namespace gk

extern "C" int gk_paged_prefill(const gk_prefill_params* params, hipStream_t stream) {
  gk::clear_error();
  return gk::paged_prefill(params, stream);
}

extern "C" int gk_prefill_list_build(const int32_t* seq_first_row, const int32_t* seq_rows, const int32_t* seq_prefix,
                                     int32_t seqs, int32_t q_heads, int32_t kv_heads, int32_t head_dim,
                                     int32_t sliding_window, int32_t* words, int64_t capacity, gk_prefill_list* list) {
  gk::clear_error();
  return gk::prefill_list_build(seq_first_row, seq_rows, seq_prefix, seqs, q_heads, kv_heads, head_dim, sliding_window,
                                true, words, capacity, list);
}

extern "C" int gk_prefill_list_build_uncut(const int32_t* seq_first_row, const int32_t* seq_rows,
                                           const int32_t* seq_prefix, int32_t seqs, int32_t q_heads, int32_t kv_heads,
                                           int32_t head_dim, int32_t sliding_window, int32_t* words, int64_t capacity,
                                           gk_prefill_list* list) {
  gk::clear_error();
  return gk::prefill_list_build(seq_first_row, seq_rows, seq_prefix, seqs, q_heads, kv_heads, head_dim, sliding_window,
                                false, words, capacity, list);
}

extern "C" size_t gk_prefill_list_workspace_bytes(const gk_prefill_params* params, const gk_prefill_list* list) {
  return params && list && params->struct_size == sizeof(gk_prefill_params) &&
                 list->struct_size == sizeof(gk_prefill_list) && params->kv_heads > 0 && list->part_slots > 0
             ? gk::list_workspace_bytes(params, list)
             : 0;
}

extern "C" int gk_paged_prefill_listed(const gk_prefill_params* params, const gk_prefill_list* list, void* workspace,
                                       size_t workspace_bytes, hipStream_t stream) {
  gk::clear_error();
  return gk::paged_prefill_listed(params, list, workspace, workspace_bytes, stream);
}
