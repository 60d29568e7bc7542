// Paged decode of short contexts for gfx950: one workgroup per work unit, one
// launch in all.
//
// A short decode step is bound by launches and memory round trips, not by
// bytes: the balanced schedule (decode_stream.hip) takes a kernel for the KV
// store, one for the attention and one for the merge, about 4 us of stream time
// and 3.5 us of host time each, for 8 us of work. In one launch 8 units of 64
// keys take 5.0 us instead of 10.5, 256 units of 512 keys 13.9 instead of 21.0
// (head_dim 128, with the store, on the stream); what then bounds it is the
// chain of round trips: arguments, the row's fields, its table and query, then
// 1.5 us for every 256 keys. Here the waves of a workgroup (eight; four or two
// for short rows of many units, so that units share a CU) share one unit (row,
// kv head, head group): wave w takes every WAVES-th of the unit's key tiles, and
// the waves' softmax states meet in LDS. Nothing is split across workgroups, so
// there is no workspace and no merge launch.
//
// The KV store of the new rows rides along: the workgroup of (row, kv head)
// writes the row's key and value into the pool, and every workgroup takes the
// new rows that its own keys include straight from the caller's tensors (a new
// row is recognised by its slot, so any row may attend any other's new key, as
// when the store ran first). What the pool holds at those slots is never used.
//
// Per-tile arithmetic is the balanced kernel's: S^T = K . Q^T on 16 x 16 MFMA
// tiles, a re-base at every new running maximum, probabilities rounded to bf16,
// P . V from a transposed LDS read, fp32 accumulation. The K and V tiles of a
// wave are 16-byte direct loads into one LDS stage; the next K tile is issued
// once this one is in registers, the next V tile after P . V, and the waves
// of a CU cover each other's waits.
#include "decode_common.hpp"

#include <algorithm>
#include <type_traits>

namespace gk {
namespace {

// In place of a slot where there is none: a new row that is not stored, a key
// that is not visible.
constexpr int32_t kNoSlot = INT32_MIN, kNoKey = -1;
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

struct UnitArgs {
  DecodeArgs d;
  int32_t units_per_row;
  DivMagic units_div, head_groups_div;  // division by units_per_row and head_groups
  // Fused KV store (null: none) of one new row per decode row.
  const uint16_t* new_key;
  const uint16_t* new_value;
  int64_t new_stride;
  const int32_t* slot_mapping;
};

// WAVES: 8, or fewer for short rows of many units (unit_waves).
template <int D, bool SOFTCAP, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 1) void decode_unit_kernel(UnitArgs ua) {
  using S = MfmaShape<D>;
  constexpr int TS = S::TS, LOADS = S::LOADS, CPR = S::CPR;
  static_assert(16 * D * 4 <= 2 * S::TILE, "a wave's partial output fits its stage");
  __shared__ __attribute__((aligned(16))) char stage[WAVES][2][S::TILE];
  constexpr int kEntries = (WAVES < 8 ? unit_short_keys(WAVES) : unit_max_keys(D)) + 1;
  __shared__ int32_t s_bt[kEntries];
  __shared__ __attribute__((aligned(16))) int32_t s_new[kUnitMaxNewRows];
  __shared__ float s_m[WAVES][16], s_l[WAVES][16];

  const DecodeArgs& a = ua.d;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c16 = lane & 15;
  const int row = (int)fast_div(blockIdx.x, ua.units_div), h = (int)blockIdx.x - row * ua.units_per_row;
  const int kvh = (int)fast_div((uint32_t)h, ua.head_groups_div), hg = h - kvh * a.head_groups;
  const int hv = min(16, a.group - hg * 16), head0 = kvh * a.group + hg * 16;
  const int qrow = a.row_map ? scalar_load(a.row_map, row) : row;
  const int request = a.row_request ? scalar_load(a.row_request, row) : row;
  const RowTiles rt = row_tiles<TS>(scalar_load(a.row_context, row), a.window);
  const int shift = a.block_shift, bmask = (1 << shift) - 1;
  uint16_t* out = a.out + (int64_t)qrow * a.out_stride + (int64_t)head0 * D;

  // The row's block-table entries of its visible keys, its query and its new
  // K/V row: one memory round trip.
  const int e0 = rt.left >> shift, ne = rt.ctx > 0 ? ((rt.ctx - 1) >> shift) - e0 + 1 : 0;
  // A row_context beyond the caller's max_context (a graph replayed on longer
  // rows) may need more entries than LDS holds: they are then read in place.
  const bool in_lds = ne <= kEntries;
  const int32_t* bt = a.block_tables + (int64_t)request * a.bt_stride + e0;
  for (int i = tid; i < min(ne, kEntries); i += WAVES * 64) s_bt[i] = bt[i];
  auto entries_at = [&](int32_t* e, const int* i, auto n) __attribute__((always_inline)) {
    if (in_lds) {
#pragma unroll
      for (int k = 0; k < n; ++k) e[k] = s_bt[i[k]];
    } else {
#pragma unroll
      for (int k = 0; k < n; ++k) e[k] = bt[i[k]];
#pragma unroll
      for (int k = 0; k < n; ++k) asm volatile("" : "+v"(e[k]));  // waited for here, not where the branches meet
    }
  };
  bf16x8_t qb[S::NC];
  {
    const uint16_t* src = a.query + (int64_t)qrow * a.q_stride + (int64_t)(head0 + c16) * D;
#pragma unroll
    for (int c = 0; c < S::NC; ++c) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (c16 < hv) v = load16(src + (4 * c + q) * 8);
      qb[c] = __builtin_bit_cast(bf16x8_t, v);
    }
  }
  // Lanes 0 .. 2 CPR - 1 (and again the lanes after them) hold the pieces of a
  // new row's key and value heads.
  const bool key_lane = (lane & (2 * CPR - 1)) < CPR;
  const int chunk = lane & (CPR - 1);
  auto new_piece = [&](int s) __attribute__((always_inline)) {
    const uint16_t* src = key_lane ? ua.new_key : ua.new_value;
    return *reinterpret_cast<const u32x4_t*>(src + (int64_t)s * ua.new_stride + (int64_t)kvh * D + chunk * 8);
  };
  u32x4_t own{0u, 0u, 0u, 0u};
  if (ua.new_key) {
    for (int s = tid; s < kUnitMaxNewRows; s += WAVES * 64) {
      const int slot = s < a.rows ? ua.slot_mapping[s] : -1;
      s_new[s] = slot >= 0 && slot < a.slots ? slot : kNoSlot;
    }
    own = new_piece(row);
  }
  __syncthreads();
  // Every load so far has landed; the compiler's wait counts do not see the
  // direct loads below.
  wait_vmem_visible();

  const uint32_t region = (uint32_t)(a.slots * D * 2);
  const uint16_t* kbase = a.pool + (int64_t)kvh * a.slots * D;
  const u32x4_t krs = buffer_words(kbase, region), vrs = buffer_words(kbase + (int64_t)a.kv_heads * a.slots * D, region);
  char* const kt = stage[wave][0];
  char* const vt = stage[wave][1];
  // Byte offsets of this lane's pieces of the tile at tb; a key outside the
  // visible ones reads the nearest visible key's row.
  struct Offsets {
    uint32_t v[LOADS];
  };
  auto offsets_of = [&](int tb) __attribute__((always_inline)) {
    Offsets of;
    int32_t e[LOADS];
    int at[LOADS];
    const auto key_of = [&](int i) { return min(max(tb + (i * 64 + lane) / CPR, rt.left), rt.ctx - 1); };
#pragma unroll
    for (int i = 0; i < LOADS; ++i) at[i] = (key_of(i) >> shift) - e0;
    entries_at(e, at, std::integral_constant<int, LOADS>{});
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int s = i * 64 + lane, tt = s / CPR, pc = s % CPR;
      const uint32_t slot = ((uint32_t)e[i] << shift) | (uint32_t)(key_of(i) & bmask);
      of.v[i] = slot * (uint32_t)(2 * D) + ((pc ^ swz(tt, D / 8)) << 4);
    }
    return of;
  };
  auto issue = [&](const Offsets& of, u32x4_t rs, char* tile) __attribute__((always_inline)) {
    const uint32_t base = lds_addr(tile);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) lds_dma16_w(base + i * 1024, rs, of.v[i]);
  };
  // The new row whose slot is that of key tb + lane % TS (-1: none): the lanes
  // of a key, 64 / TS of them, compare a share of the new slots each.
  constexpr int kShares = 64 / TS;
  const int share = ua.new_key ? (a.rows + 4 * kShares - 1) / (4 * kShares) : 0;  // in groups of four slots
  auto new_row_of = [&](int tb) __attribute__((always_inline)) {
    const int key = tb + (lane & (TS - 1));
    const bool visible = key >= rt.left && key < rt.ctx;
    const int at = (min(max(key, rt.left), rt.ctx - 1) >> shift) - e0;
    int32_t entry;
    entries_at(&entry, &at, std::integral_constant<int, 1>{});
    const int slot = visible && entry >= 0 ? (int)(((uint32_t)entry << shift) | (uint32_t)(key & bmask)) : kNoKey;
    const int g0 = (lane / TS) * share;
    int found = -1;
    for (int g = g0; g < g0 + share; ++g) {
      const i32x4_t n = *reinterpret_cast<const i32x4_t*>(s_new + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) found = n[i] == slot ? 4 * g + i : found;
    }
    return found;
  };

  f32x4_t o[S::NO];
#pragma unroll
  for (int c = 0; c < S::NO; ++c) o[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f, m_thr = -INFINITY, m_base = 0.f;
  const float inv_scale = 1.f / a.score_scale;

  const int ntiles = rt.ctx > 0 ? rt.count : 0;
  Offsets next{};
  if (wave < ntiles) {
    next = offsets_of((rt.first + wave) * TS);
    issue(next, krs, kt);
    issue(next, vrs, vt);
  }
  for (int k = wave; k < ntiles; k += WAVES) {
    const int tb = (rt.first + k) * TS;
    const bool more = k + WAVES < ntiles;
    if (more) next = offsets_of(tb + WAVES * TS);
    const int found = share ? new_row_of(tb) : -1;
    uint64_t hits = __builtin_amdgcn_ballot_w64(found >= 0);
    if (hits) {
      wait_vmem<0>();
      for (; hits; hits &= hits - 1) {
        const int l = __builtin_ctzll(hits), s = __builtin_amdgcn_readlane(found, l), tt = l & (TS - 1);
        u32x4_t v = own;
        if (s != row) v = new_piece(s);
        *reinterpret_cast<u32x4_t*>(kt + (key_lane ? 0 : S::TILE) + tt * (2 * D) + ((chunk ^ swz(tt, D / 8)) << 4)) = v;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      wait_vmem<LOADS>();
    }

    // K tile -> registers: lane (q, c16), group g holds key 16 g + c16, chunk 4 c + q.
    bf16x8_t kr[S::TG][S::NC];
#pragma unroll
    for (int g = 0; g < S::TG; ++g) {
      const int tt = 16 * g + c16;
#pragma unroll
      for (int c = 0; c < S::NC; ++c)
        kr[g][c] = *reinterpret_cast<const bf16x8_t*>(kt + tt * (2 * D) + (((4 * c + q) ^ swz(tt, D / 8)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) issue(next, krs, kt);
    f32x4_t sc[S::TG];
#pragma unroll
    for (int g = 0; g < S::TG; ++g) {
      sc[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < S::NC; ++c) sc[g] = mfma32(kr[g][c], qb[c], sc[g]);
    }
    if constexpr (!SOFTCAP) mfma_results_ready(sc);
    const bool inside = !SOFTCAP && tb >= rt.left && tb + TS <= rt.ctx;
    if (!inside) {
#pragma unroll
      for (int g = 0; g < S::TG; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float s = sc[g][r];
          if constexpr (SOFTCAP) s = soft_cap(s * a.score_scale, a.softcap_log2);
          const int key = tb + 16 * g + 4 * q + r;
          sc[g][r] = (key >= rt.left && key < rt.ctx) ? s : -INFINITY;
        }
    }
    float mx;
    {
      float v[4 * S::TG];
#pragma unroll
      for (int i = 0; i < 4 * S::TG; ++i) v[i] = sc[i >> 2][i & 3];
      mx = col4_max(tree_max(v));
    }
    if (__builtin_amdgcn_ballot_w64(mx > (SOFTCAP ? m_run + kDecodeRescaleSlack : m_thr))) {
      const float m_new = fmaxf(m_run, SOFTCAP ? mx : mx * a.score_scale);
      const float alpha = m_run == -INFINITY ? 0.f : fast_exp2(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
      m_thr = (m_new + kDecodeRescaleSlack) * inv_scale;
      m_base = m_new == -INFINITY ? 0.f : m_new;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float f = __int_as_float(__builtin_amdgcn_ds_bpermute((4 * q + r) << 2, __float_as_int(alpha)));
#pragma unroll
        for (int c = 0; c < S::NO; ++c) o[c][r] *= f;
      }
    }
#pragma unroll
    for (int g = 0; g < S::TG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = SOFTCAP ? fast_exp2(sc[g][r] - m_base) : fast_exp2(__builtin_fmaf(sc[g][r], a.score_scale, -m_base));
        sc[g][r] = p;
        l_run += p;
      }

    if (more) wait_vmem<LOADS>();
    else wait_vmem<0>();
    if (tb < rt.left || tb + TS > rt.ctx) {
      // A masked key weighs zero, but its row may hold an infinity.
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int s = i * 64 + lane, key = tb + s / CPR;
        if (key < rt.left || key >= rt.ctx) *reinterpret_cast<uint4*>(vt + s * 16) = make_uint4(0, 0, 0, 0);
      }
    }
    if constexpr (TS == 32) {
      bf16x8_t pa;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[r] = (__bf16)sc[0][r];
        pa[4 + r] = (__bf16)sc[1][r];
      }
#pragma unroll
      for (int c = 0; c < S::NO; ++c) {
        const int lc = 2 * c + ((c16 & 3) >> 1);
        const int t0 = 4 * q + (c16 >> 2), t1 = t0 + 16;
        const bf16x4_t v0 = lds_read_tr4(vt + t0 * (2 * D) + ((lc ^ swz(t0, D / 8)) << 4) + ((c16 & 1) << 3));
        const bf16x4_t v1 = lds_read_tr4(vt + t1 * (2 * D) + ((lc ^ swz(t1, D / 8)) << 4) + ((c16 & 1) << 3));
        o[c] = mfma32(pa, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7), o[c]);
      }
    } else {
      bf16x4_t pa;
#pragma unroll
      for (int r = 0; r < 4; ++r) pa[r] = (__bf16)sc[0][r];
#pragma unroll
      for (int c = 0; c < S::NO; ++c) {
        const int lc = 2 * c + ((c16 & 3) >> 1);
        const int t0 = 4 * q + (c16 >> 2);
        o[c] = mfma16(pa, lds_read_tr4(vt + t0 * (2 * D) + ((lc ^ swz(t0, D / 8)) << 4) + ((c16 & 1) << 3)), o[c]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) issue(next, vrs, vt);
  }

  // The waves' states meet in LDS: output rows in the wave's own stage.
  l_run = col4_sum(l_run);
  if (lane < 16) {
    s_m[wave][lane] = m_run;
    s_l[wave][lane] = l_run;
  }
  float* po = reinterpret_cast<float*>(stage[wave][0]);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * q + r < hv) {
#pragma unroll
      for (int c = 0; c < S::NO; ++c) po[(4 * q + r) * D + 16 * c + c16] = o[c][r];
    }
  __syncthreads();
  for (int idx = tid; idx < hv * D; idx += WAVES * 64) {
    const int hh = idx / D;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, s_m[w][hh]);
    float acc = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = s_m[w][hh] == -INFINITY ? 0.f : fast_exp2(s_m[w][hh] - mm);
      ll += s_l[w][hh] * f;
      acc += reinterpret_cast<const float*>(stage[w][0])[idx] * f;
    }
    out[idx] = (uint16_t)bf16_bits(acc * (ll > 0.f ? 1.f / ll : 0.f));
  }
  // The row's new key and value, by the last wave of the kv head's first unit.
  if (ua.new_key && hg == 0 && wave == WAVES - 1) {
    const int slot = s_new[row];
    if (slot != kNoSlot && lane < 2 * CPR) {
      uint16_t* dst = a.pool_out + ((int64_t)(key_lane ? kvh : a.kv_heads + kvh) * a.slots + slot) * D + chunk * 8;
      __builtin_nontemporal_store(own, reinterpret_cast<u32x4_t*>(dst));
    }
  }
}

}  // namespace

// Where one workgroup per unit is the faster form, and with how many waves, by
// time on the stream, both with the fused store (us; balanced schedule / unit
// kernel):
//   head_dim 128, 8 units x 64 keys 10.5 / 5.0, x 512 10.8 / 7.5, x 1024 10.8 /
//   10.6, x 1536 12.3 / 13.5, x 2048 12.6 / 16.5; 64 units x 2048 21.1 / 17.5;
//   256 x 512 21.0 / 13.9, x 2048 51.4 / 42.2, x 3072 71.2 / 72.4; 512 x 1024
//   50.6 / 44.0, x 1536 69.0 / 74.1.
//   head_dim 64, 8 x 2048 11.0 / 11.7, x 3000 11.5 / 15.5; 256 x 3000 40.0 /
//   32.6; 512 x 2048 52.4 / 42.9, x 3072 72.2 / 73.1. head_dim 256, 8 x 512
//   11.0 / 10.9, x 768 13.5 / 14.0, x 1024 14.0 / 16.6; 256 x 1024 50.8 / 43.5;
//   512 x 512 51.8 / 43.6, x 1024 90.6 / 95.9.
// So eight waves for at most 1 MiB of keys and values a unit, 256 MiB in all and
// 512 units; 3/4 MiB (2048 keys) where fewer than 32 units leave the GPU to the
// balanced schedule's many workgroups. Up to 2 us of stream time are given for
// the two launches (7 us of host time) that the unit form saves.
// More units than CUs hold of the eight-wave form (one a CU; two at head_dim 64)
// run in rounds whose start and end nothing covers; fewer waves with less LDS
// put several units on a CU, each slower (balanced / 2 / 4 / 8 waves):
//   head_dim 128, 512 units x 64 14.6 / 6.6 / 6.4 / 10.0, x 256 21.7 / 15.6 /
//   15.1 / 18.0, x 512 30.7 / - / 25.2 / 27.0; 1024 x 64 15.1 / 9.9 / 14.1 /
//   22.4, x 128 20.3 / 17.0 / 18.1 / 25.7, x 512 49.6 / - / 44.7 / 49.7; 1536 x
//   128 28.7 / 25.4 / 25.5 / 39.6, x 256 43.6 / 41.1 / 38.8 / 50.2, x 512 75.1 /
//   - / 80.1; 2048 x 64 22.8 / 22.6 / 30.2.
//   head_dim 64, 1024 x 64 13.7 / 6.1 / 6.6 / 10.7, x 512 31.2 / - / 26.4 / 26.3;
//   2048 x 64 15.2 / 11.0 / 15.7, x 512 50.2 / - / 48.4. head_dim 256, 512 x 256
//   30.3 / 24.1 / 26.2 / 26.1; 1024 x 256 53.1 / 46.4 / 50.7.
// Lengths spread from a twentieth of the longest on favour the balanced schedule:
//   head_dim 128, 1024 x up to 512 32.8 / - / 30.0, 1536 x up to 256 28.2 / 28.6 /
//   30.0; head_dim 64, 2048 x up to 512 36.3 / - / 36.6; head_dim 256, 512 x up to
//   256 23.7 / 18.9, 1024 x up to 256 35.0 / 38.3; so the line lies at 1024 eight-
//   wave workgroups, 512 at head_dim 256.
// The rule sees the longest row only. Eight waves on spread lengths (balanced /
// unit; uniform and log-uniform from a twentieth of the longest, one long row
// among rows of a twentieth):
//   head_dim 128, 32 units x up to 2048 14.1 / 16.5, 14.3 / 16.7, 13.5 / 16.5,
//   x up to 1024 12.4 / 10.8, 12.0 / 10.8, 11.9 / 10.9; 128 x up to 2048 25.1 /
//   20.9, 18.2 / 18.0, 13.9 / 17.3; 256 x up to 2048 32.4 / 26.3, 25.9 / 22.4,
//   17.4 / 18.7. head_dim 64, 32 x up to 3072 13.6 / 15.8, 13.0 / 15.7, 12.1 /
//   15.8; 256 x up to 3072 26.6 / 22.6, 23.7 / 20.8, 17.2 / 18.4. head_dim 256,
//   32 x up to 1024 14.4 / 16.9, 13.6 / 16.7, 14.6 / 17.2; 256 x up to 1024
//   37.2 / 29.9, 27.6 / 23.7, 15.7 / 18.1.
// So a few long rows among short ones lose up to 3.7 us of stream time here, more
// than equal lengths do, and the whole operator call still gains: 4 rows of which
// one has 2048 keys 16.6 us instead of 21.9 for the three launches, one of 16
// 17.2 instead of 22.3. A caller whose stream alone counts (replayed graphs) gets
// the balanced schedule with a max_context above the limit.
namespace {
// Waves of a unit's workgroup; 0: the balanced schedule.
int unit_waves(const gk_decode_params* p, int64_t units) {
  const int64_t visible = p->sliding_window > 0 ? std::min(p->max_context, p->sliding_window) : p->max_context;
  const int64_t load = p->head_dim == 64 ? (units + 1) / 2 : units;  // eight-wave workgroups in CUs
  if (load > 256) {
    if (p->head_dim == 256) {
      if (load <= 512 && visible <= unit_short_keys(2)) return 2;
    } else if (load <= 512) {
      if (visible <= unit_short_keys(4)) return 4;
    } else if (load <= 1024) {
      if (visible <= unit_short_keys(2) / 2) return 2;
      if (visible <= unit_short_keys(4)) return 4;
    }
  }
  const int64_t most = units < 32 ? std::min(2048, (3 << 16) / p->head_dim) : unit_max_keys(p->head_dim);
  return visible <= most && units <= 512 && units * visible * p->head_dim <= int64_t(1) << 26 ? 8 : 0;
}
}  // namespace

bool unit_decode_fits(const gk_decode_params* p, int64_t units) { return unit_waves(p, units) != 0; }

int launch_unit_decode(const DecodeArgs& a, bool softcap, int head_dim, const gk_decode_params* p, bool store,
                       hipStream_t stream) {
  UnitArgs ua{};
  ua.d = a;
  ua.units_per_row = a.kv_heads * a.head_groups;
  ua.units_div = div_magic((uint32_t)ua.units_per_row);
  ua.head_groups_div = div_magic((uint32_t)a.head_groups);
  if (store) {
    ua.new_key = static_cast<const uint16_t*>(p->new_key);
    ua.new_value = static_cast<const uint16_t*>(p->new_value);
    ua.new_stride = p->new_kv_row_stride;
    ua.slot_mapping = p->slot_mapping;
    ua.d.pool_out = static_cast<uint16_t*>(const_cast<void*>(p->pool));
  }
  const int64_t units = (int64_t)a.rows * ua.units_per_row;
  const dim3 grid((unsigned)units);
  const int waves = unit_waves(p, units);
  const auto launch_waves = [&](auto d, auto w) {
    constexpr int D = decltype(d)::value, W = decltype(w)::value;
    if (softcap) decode_unit_kernel<D, true, W><<<grid, W * 64, 0, stream>>>(ua);
    else decode_unit_kernel<D, false, W><<<grid, W * 64, 0, stream>>>(ua);
  };
  const auto launch = [&](auto d) {
    if (waves == 2) launch_waves(d, std::integral_constant<int, 2>{});
    else if (waves == 4) launch_waves(d, std::integral_constant<int, 4>{});
    else launch_waves(d, std::integral_constant<int, 8>{});
  };
  if (head_dim == 64) launch(std::integral_constant<int, 64>{});
  else if (head_dim == 128) launch(std::integral_constant<int, 128>{});
  else launch(std::integral_constant<int, 256>{});
  return hip_status(hipGetLastError(), "gk_paged_decode unit launch");
}

}  // namespace gk
