// Paged attention on the matrix cores for steps that bring portions of prompts, bfloat16. The
// step's (token, query head) pairs of one key/value head are cut into tiles of 16 rows: 16 / G
// consecutive tokens of one request with the G heads of the group. A workgroup of four waves takes
// up to 4 RT such tiles of consecutive tokens (RT per wave) and walks the request's keys from the
// first position any of its rows may see to the last, 32 keys at a time. Each step's keys and
// values are fetched from the pages once per workgroup, straight into LDS in the order the lanes use them, each wave
// its share of the operand registers, and all waves read the whole step back from there. Three steps are in LDS, two of them under
// way: through registers, a step ahead, every step waited for its loads (measured before and after, µs, heads of 64: 90 tokens 7.3
// and 6.4, 1,024 19.8 and 16.0, 2,048 36.1 and 32.3; 24 heads of 128: 2,048 tokens 52.5 and 45.7). With a fourth step for heads of 64
// a unit holds a workgroup fewer, which short turns behind long contexts feel: 100 tokens behind 8,000 31.8 before, 32.6 with four and
// 31.4 with three, 400 behind 16,000 125.7, 130.5 and 129.2. Beyond that the vector work of the softmax bounds it, next to LDS's reads. (Pages that are
// no multiple of 32 keys, whose steps lie in several, still go through registers.) A row masks the keys beyond its own
// position (and before its window); steps that lie wholly inside every row's range skip the masks.
// Normally nothing is split and nothing is combined: a row's sums run over the keys in ascending
// order, whatever the batch. A step of few tokens over a long context has too few tiles to fill the
// chip: then the keys are cut into chunks (num_splits > 1), a workgroup walks one chunk for its
// tile and leaves the rows' partial results (part_o, part_ml, as the decode kernel does), and the
// decode kernel's combining kernel sums the chunks in ascending order.
//
// The host lists the tiles: tiles[2 i] = index of the tile's first token in the step,
// tiles[2 i + 1] = number of its tokens (at most 4 RT (16 / G), all of one request), in ascending
// order of the number of keys a tile walks. There is one workgroup per (key/value head, tile), and
// the long tiles start first. The chip hands consecutive workgroups to its eight dies in turn, and
// each die has a cache of its own, so the kernel maps workgroups to work such that those which walk
// one head's keys sit on as few dies as possible: with eight heads (or a multiple) each die works
// on heads of its own and reads their keys from memory once.
#include <type_traits>
#include "attention_decode.h"
#include "lds_loads.h"

#define PRE_MAX_WAVES 8

// Where the steps of a walk lie (whole steps only: pages of a multiple of 32 keys): a ring of PRE_PLACES steps, refilled
// by halves, that holds for step i what its page and slot add to a lane's fixed place in the keys' pool and in the
// values'. The walk reads a step's entry instead of looking its page up and multiplying.
#define PRE_PLACES 256
template <int HD, bool WHOLE>
struct PrefillLds {
  static constexpr int STAGES = WHOLE ? 3 : 2;
  uint4 stage[STAGES][HD / 8][TS_WAVE];   // steps of operand registers, [register][lane]
  int range[4][PRE_MAX_WAVES];
  int64_t place[2][PRE_PLACES];      // [keys | values][step mod PRE_PLACES], in elements
};

// PRE_WAVES: 4, or 8 (heads of 64 or 128 dimensions): the same tokens a workgroup in tiles half as
// large a wave, so that a step's vector work is spread over twice the waves; the longest tiles of a
// short prompt, which run alone at the end, then take a shorter step (2,048 tokens at head size 64:
// 48.9 µs against 51.3; over long contexts the doubled reads of LDS cost more than that gains).
// WHOLE: a page holds a multiple of 32 keys, so that every step lies in one page.
// GENERAL: capped scores, weights in two terms (attention_mfma.h) and optionally a sink, added to a row's sum at the end.
template <int HD, int RT, int PRE_WAVES, bool WHOLE, bool GENERAL>
static __device__ __forceinline__ void
prefill_tile(PrefillLds<HD, WHOLE>& lds, int tile, int kvh, bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
             const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
             const int32_t* __restrict__ block_tables, const int32_t* __restrict__ seq_of_token,
             const int32_t* __restrict__ positions, const int32_t* __restrict__ tiles, int nh, int group, int page_size,
             int page_shift, int page_run, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks,
             float scale2, int window, float* __restrict__ part_o, float* __restrict__ part_ml, int num_splits,
             int chunk, int split, float cap_in, float cap_out, int sink, const float* __restrict__ sinks,
             const float* __restrict__ slopes, const float* __restrict__ gate, int64_t gate_stride) {
  constexpr int NC = HD / 32, NDB = HD / 16;   // operand registers of a 32-key step: 2 NC of K, NDB of V
  auto& stage = lds.stage;
  auto& wg_range = lds.range;
  const int wave = wave_index(), lane = threadIdx.x & (TS_WAVE - 1);
  const int r = lane & 15, g = lane >> 4;
  const int t0 = tiles[2 * tile], ntok = tiles[2 * tile + 1];
  const int32_t* table = block_tables + (int64_t)seq_of_token[t0] * max_blocks;
  const PageMath pm{page_size, page_shift, page_run};
  // heads of the group, tokens per row tile (16 / G), and what a row below 16 is multiplied by to be divided by G (256ths, rounded up)
  const int G = group & 255, tpt = (group >> 8) & 255, per_g = group >> 16;
  auto over_g = [&](int row) { return (row * per_g) >> 8; };

  // lane r carries row r of each of its wave's score tiles: token tk[j], head r % G of the group
  const int rt0 = over_g(r), hh = r - rt0 * G;
  // (the general variant: this row's head's penalty per position of distance, in the scores' units before scale2)
  const float slope = (GENERAL && slopes) ? slopes[kvh * G + hh] * (1.44269504088896340736f / scale2) : 0.f;
  int pos[RT], lo[RT], tk[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    tk[j] = (wave * RT + j) * tpt + rt0;
    const bool ok = rt0 < tpt && tk[j] < ntok;
    pos[j] = ok ? positions[t0 + tk[j]] : -1;               // -1: no key is visible, the row stays empty
    lo[j] = ts_first_key(pos[j], window);
    if (!ok) tk[j] = -1;
  }
  // per row tile: the smallest position and largest window start of its rows (wave-uniform)
  // (tile_vpmin: the smallest position among the rows that exist; rows that do not are never stored)
  int tile_lomax[RT], tile_pmax[RT], tile_lomin[RT], tile_vpmin[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    tile_lomax[j] = lo[j]; tile_pmax[j] = pos[j];
    tile_lomin[j] = tk[j] >= 0 ? lo[j] : 0x7fffffff;
    tile_vpmin[j] = tk[j] >= 0 ? pos[j] : 0x7fffffff;
  }
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) {                  // (the four lanes of a row hold the same)
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      tile_vpmin[j] = min(tile_vpmin[j], __shfl_xor(tile_vpmin[j], off, TS_WAVE));
      tile_pmax[j] = max(tile_pmax[j], __shfl_xor(tile_pmax[j], off, TS_WAVE));
      tile_lomax[j] = max(tile_lomax[j], __shfl_xor(tile_lomax[j], off, TS_WAVE));
      tile_lomin[j] = min(tile_lomin[j], __shfl_xor(tile_lomin[j], off, TS_WAVE));
    }
  }
  // the workgroup's key range [wlo, whi], and the range every one of its rows sees whole: [wfull_lo, wfull_hi]
  if (lane == 0) {
    int pmin = 0x7fffffff, lomax = 0, pmax = -1, lmin = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      pmin = min(pmin, tile_vpmin[j]); lomax = max(lomax, tile_lomax[j]);
      pmax = max(pmax, tile_pmax[j]); lmin = min(lmin, tile_lomin[j]);
    }
    wg_range[0][wave] = lmin; wg_range[1][wave] = pmax; wg_range[2][wave] = pmin; wg_range[3][wave] = lomax;
  }
  __syncthreads();
  int wlo = wg_range[0][0], whi = wg_range[1][0], wfull_hi = wg_range[2][0], wfull_lo = wg_range[3][0];
#pragma unroll
  for (int w = 1; w < PRE_WAVES; ++w) {
    wlo = min(wlo, wg_range[0][w]); whi = max(whi, wg_range[1][w]);
    wfull_hi = min(wfull_hi, wg_range[2][w]); wfull_lo = max(wfull_lo, wg_range[3][w]);
  }
  if (num_splits > 1) {
    // this workgroup walks one chunk of the keys only (chunks are multiples of 32 keys, so no step
    // straddles two); what the rows see of it is combined with the other chunks afterwards
    // (the last chunk has no upper end, so every position is in some chunk whatever the caller chose)
    wlo = max(wlo, split * chunk);
    wfull_lo = max(wfull_lo, split * chunk);
    if (split + 1 < num_splits) {
      whi = min(whi, split * chunk + chunk - 1);
      if (wfull_hi != 0x7fffffff) wfull_hi = min(wfull_hi, split * chunk + chunk - 1);
    }
  }
  // every lane holds the same values: say so, and loop control and page lookups become scalar
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  whi = __builtin_amdgcn_readfirstlane(whi);
  wfull_lo = __builtin_amdgcn_readfirstlane(wfull_lo);
  wfull_hi = __builtin_amdgcn_readfirstlane(wfull_hi);
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    tile_pmax[j] = __builtin_amdgcn_readfirstlane(tile_pmax[j]);
    tile_lomax[j] = __builtin_amdgcn_readfirstlane(tile_lomax[j]);
    tile_lomin[j] = __builtin_amdgcn_readfirstlane(tile_lomin[j]);
  }

  uint4 qreg[RT][NC];
  float m[RT];
  float4_t l[RT];                 // the sums of the output rows 4 g + i, made by the matrix cores
  float4_t o[RT][NDB];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    m[j] = -INFINITY; l[j] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) qreg[j][c] = make_uint4(0, 0, 0, 0);
    if (tk[j] >= 0) {
      const bf16_t* qrow = q + ((int64_t)(t0 + tk[j]) * nh + (int64_t)kvh * G + hh) * HD + 8 * g;
#pragma unroll
      for (int c = 0; c < NC; ++c) qreg[j][c] = *(const uint4*)(qrow + 32 * c);
    }
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[j][db] = (float4_t){0.f, 0.f, 0.f, 0.f};
  }

  // This wave's share of a step's operand registers, PER of the 4 NC: register q < 2 NC is piece q % NC
  // of the 16-key tile q / NC of K, register 2 NC + db is dimension block db of V.
  constexpr int PER = 4 * NC / PRE_WAVES;
  static_assert(PER >= 1 && PER * PRE_WAVES == 4 * NC, "the waves share a step's operand registers evenly");
  uint4 fetched[PER];
  const bool loads_k = wave * PER < 2 * NC;           // (a wave's registers are all of K or all of V)
  const int tau = (wave * PER) / NC, c0 = (wave * PER) % NC, db0 = wave * PER - 2 * NC;
  const int kbeg = wlo & ~31;
  const int kend = whi + 1;
  // Whole steps: a lane's pieces lie at the same places of every page, so what the lane adds to a step's
  // place is worked out once, and the steps' places come from the ring in LDS.
  const int koff = 8 * (r >> 2) + 4 * tau + (r & 3);
  const bf16_t* const lane_base = loads_k ? k_cache + ((int64_t)kvh * kh + (int64_t)koff * ks + 8 * g + 32 * c0)
                                          : v_cache + ((int64_t)kvh * vh + 8 * g + (int64_t)(db0 * 16 + r) * vd);
  const int64_t piece = loads_k ? 32 : 16 * vd;
  const int64_t* const places = lds.place[loads_k ? 0 : 1];
  // the places of the walk's steps first .. first + count - 1 go into the ring (steps beyond the last one: the
  // last one's, whose page is the request's as well)
  auto fill_places = [&](int first, int count) {
    for (int i = threadIdx.x; i < count; i += PRE_WAVES * TS_WAVE) {
      const int kb = min(kbeg + 32 * (first + i), whi & ~31);
      const int pg = pm.page(kb);
      const int64_t page = pm.pool_page(table, pg);
      const int slot = pm.slot(kb, pg);
      lds.place[0][(first + i) & (PRE_PLACES - 1)] = page * kp + (int64_t)slot * ks;
      lds.place[1][(first + i) & (PRE_PLACES - 1)] = page * vp + slot;
    }
  };
  auto place_of = [&](int kb) { return places[((kb - kbeg) >> 5) & (PRE_PLACES - 1)]; };
  // Whole steps go straight into LDS: asks for the step that lies at `place`. All its slots are memory of the request's page,
  // whoever sees them (keys out of the walk are masked, and values of theirs count as zeros: `vok` below).
  constexpr int STAGES = PrefillLds<HD, WHOLE>::STAGES;
  const uint32_t stage0 = (uint32_t)(uintptr_t)(lds_ptr_t)&stage[0][0][0] + wave * PER * 1024;
  auto bring = [&](int64_t place, int to) {
    const bf16_t* src = lane_base + place;
#pragma unroll
    for (int c = 0; c < PER; ++c) row_to_lds(src + c * piece, stage0 + (uint32_t)to * (HD / 8 * 1024) + c * 1024);
  };
  auto fetch = [&](int kb) {
#pragma unroll
    for (int c = 0; c < PER; ++c) fetched[c] = make_uint4(0, 0, 0, 0);
    if (loads_k) {
      const int key = kb + 8 * (r >> 2) + 4 * tau + (r & 3);
      if (key <= whi && key >= wlo) {
        const int pg = pm.page(key);
        const bf16_t* kr = k_cache + pm.pool_page(table, pg) * kp + (int64_t)pm.slot(key, pg) * ks + (int64_t)kvh * kh + 8 * g + 32 * c0;
#pragma unroll
        for (int c = 0; c < PER; ++c) fetched[c] = *(const uint4*)(kr + 32 * c);
      }
    } else {
      const int vkey = kb + 8 * g;
      if (vkey <= whi && vkey + 7 >= wlo) {
        const int pg = pm.page(vkey);
        const bf16_t* vr = v_cache + pm.pool_page(table, pg) * vp + pm.slot(vkey, pg) + (int64_t)kvh * vh +
                           (int64_t)(db0 * 16 + r) * vd;
#pragma unroll
        for (int c = 0; c < PER; ++c) fetched[c] = *(const uint4*)(vr + (int64_t)(16 * c) * vd);
      }
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int c = 0; c < PER; ++c) stage[buf][wave * PER + c][lane] = fetched[c];
  };

  // The walk has three stretches: steps that some row sees in part (before the last window start),
  // steps that every row of the workgroup sees whole, and the steps around the rows' own positions.
  // The middle one, nearly all of a long walk, runs without masks and without the test whether a
  // tile has anything to do; each stretch is a loop of its own so that the accumulators stay in
  // their registers from one step to the next.
  const int full_lo = min(max((wfull_lo + 31) & ~31, kbeg), kend);
  const int full_hi = min(max(wfull_hi == 0x7fffffff ? 0 : ((wfull_hi + 1) & ~31), full_lo), kend);
  int buf = 0;
  int64_t place_next = 0;                    // whole steps: the place of the next step to be asked for, read a step early
  auto walk = [&](int from, int to, auto masked) {
    constexpr bool MASKED = decltype(masked)::value;
    for (int kb = from; kb < to; kb += 32) {
      if constexpr (WHOLE) {
        // every half turn of the ring of places the half that the walk has left behind takes the places of the steps
        // a turn ahead (first read half a turn from now, many barriers later)
        const int step = (kb - kbeg) >> 5;
        if ((step & (PRE_PLACES / 2 - 1)) == 0 && step) fill_places(step + PRE_PLACES / 2, PRE_PLACES / 2);
        // this step has landed once at most STAGES - 2 others are under way; behind the barrier all waves' parts of it
        // have, and all waves have read the step before, whose stage takes the step STAGES - 1 ahead
        wait_for<(STAGES - 2) * PER, 0>();
        __builtin_amdgcn_s_barrier();
        bring(place_next, buf == 0 ? STAGES - 1 : buf - 1);
        place_next = place_of(kb + 32 * STAGES);
      }
      KVTile<HD> T;
#pragma unroll
      for (int c = 0; c < NC; ++c) { T.k[0][c] = stage[buf][c][lane]; T.k[1][c] = stage[buf][NC + c][lane]; }
#pragma unroll
      for (int db = 0; db < NDB; ++db) T.v[db] = stage[buf][2 * NC + db][lane];
      T.vok = true;                          // (what lies outside the range went into LDS as zeros)
      if constexpr (WHOLE) {
        if constexpr (MASKED) T.vok = kb + 8 * g <= whi && kb + 8 * g + 7 >= wlo;
        buf = buf == STAGES - 1 ? 0 : buf + 1;
      } else {
        buf ^= 1;
        if (kb + 32 < kend) put(buf);        // the other buffer was last read before the previous barrier
        if (kb + 64 < kend) fetch(kb + 64);
      }
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        // a step wholly beyond the tile's last position, or wholly before all its windows, has nothing for it
        if (!MASKED || (kb <= tile_pmax[j] && kb + 31 >= tile_lomin[j]))
          use_tile<HD, MASKED, float4_t, GENERAL>(T, kb, r, g, lo[j], pos[j], qreg[j], scale2, m[j], l[j], o[j], cap_in, cap_out, slope);
      }
      if constexpr (!WHOLE) __syncthreads();
    }
  };
  if (kbeg < kend) {                         // uniform over the workgroup
    if constexpr (WHOLE) {
      fill_places(0, PRE_PLACES);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < STAGES - 1; ++i) bring(place_of(kbeg + 32 * i), i);
      place_next = place_of(kbeg + 32 * (STAGES - 1));
    } else {
      fetch(kbeg);
      put(0);
      if (kbeg + 32 < kend) fetch(kbeg + 32);
      __syncthreads();
    }
    walk(kbeg, full_lo, std::true_type{});
    walk(full_lo, full_hi, std::false_type{});
    walk(full_hi, kend, std::true_type{});
    wait_for<0>();                           // (steps asked for beyond the walk land before the workgroup's LDS is another's)
  }
  // output row 4 g + i of row tile j: its token and head, and its sum
#pragma unroll
  for (int j = 0; j < RT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * g + i;
      float lj = l[j][i];
      const int at_row = over_g(row), rtk = (wave * RT + j) * tpt + at_row, rhh = row - at_row * G;
      const float mj = __shfl(m[j], row, TS_WAVE);       // the row's reference maximum (lane `row` holds it)
      // the sink's score is 0, or its head's learned one
      if (GENERAL && sink && num_splits == 1 && lj > 0.f)
        lj += fast_exp2((sinks ? sinks[kvh * G + rhh] * 1.44269504088896340736f : 0.f) - mj);
      if (num_splits > 1) {
        // the chunk's share of the row, not normalised: sums, and the reference maximum they are relative to
        if (at_row < tpt && rtk < ntok) {
          const int64_t at = (((int64_t)(t0 + rtk) * nh + (int64_t)kvh * G + rhh) * num_splits + split);
#pragma unroll
          for (int db = 0; db < NDB; ++db) part_o[at * HD + 16 * db + r] = o[j][db][i];
          if (r == 0) { part_ml[at * 2] = mj; part_ml[at * 2 + 1] = lj; }
        }
        continue;
      }
      if (at_row < tpt && rtk < ntok && lj > 0.f) {
        const float inv = 1.0f / lj;
        bf16_t* orow = out + ((int64_t)(t0 + rtk) * nh + (int64_t)kvh * G + rhh) * HD;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          float y = o[j][db][i] * inv;
          if (GENERAL) y *= ts_out_gate(gate, gate_stride, t0 + rtk, kvh * G + rhh, HD, 16 * db + r);
          orow[16 * db + r] = f2bf(y);
        }
      }
    }
}

// Workgroup `block` of `blocks`, the kernel's own or the first ones of the kernel below.
template <int HD, int RT, int PRE_WAVES, bool WHOLE, bool GENERAL>
static __device__ __forceinline__ void
prefill_block(PrefillLds<HD, WHOLE>& lds, int block, int blocks, bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                         const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_tables,
                         const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                         const int32_t* __restrict__ tiles, int num_tiles, int nh, int group, int dies_per_group,
                         int heads_per_group, int page_size, int page_shift, int page_run, int64_t kp, int64_t ks, int64_t kh,
                         int64_t vp, int64_t vh, int64_t vd, int max_blocks, float scale2, int window,
                         float* __restrict__ part_o, float* __restrict__ part_ml, int num_splits, int chunk,
                         float cap_in, float cap_out, int sink, const float* __restrict__ sinks,
                         const float* __restrict__ slopes, const float* __restrict__ gate, int64_t gate_stride) {
  // die = workgroup index mod 8. The dies form `groups` groups of `dies_per_group`, the heads as
  // many groups of `heads_per_group`; a group's (tile, head) pairs go round its dies, long tiles first.
  // A die's workgroups go round its 32 compute units. Where two of them fit a unit, those of a short prompt run all at once, and
  // every other round takes its tiles in the opposite order, so that the unit with the longest walk of one round has the
  // shortest of the next (heads of 64: 1,024 tokens 18.2 and now 16.0 µs, 2,048 33.8 and 32.3; of 128 with eight waves, one
  // workgroup a unit, 46.0 and 54.2: longest first there).
  constexpr bool PAIRS = PRE_WAVES == 4 ? RT * HD <= 256 : HD <= 64;
  const int die = block % 8, place = block / 8, round = place / 32;
  const int turn = PAIRS && round % 2 ? 32 * round + min(32 * round + 32, blocks / 8) - 1 - place : place;
  const int item = turn * dies_per_group + die % dies_per_group;
  if (item >= num_tiles * heads_per_group) return;
  const int tile = num_tiles - 1 - item / heads_per_group;
  const int kvh = (die / dies_per_group) * heads_per_group + item % heads_per_group;
  prefill_tile<HD, RT, PRE_WAVES, WHOLE, GENERAL>(lds, tile, kvh, out, q, k_cache, v_cache, block_tables, seq_of_token, positions, tiles, nh,
                       group, page_size, page_shift, page_run, kp, ks, kh, vp, vh, vd, max_blocks, scale2, window, part_o, part_ml,
                       num_splits, chunk, blockIdx.y, cap_in, cap_out, sink, sinks, slopes, gate, gate_stride);
}

template <int HD, int RT, int PRE_WAVES, bool WHOLE, bool GENERAL>
__global__ void __launch_bounds__(PRE_WAVES * TS_WAVE)
attn_prefill_mfma_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
                         const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_tables,
                         const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ positions,
                         const int32_t* __restrict__ tiles, int num_tiles, int nh, int group, int dies_per_group,
                         int heads_per_group, int page_size, int page_shift, int page_run, int64_t kp, int64_t ks, int64_t kh,
                         int64_t vp, int64_t vh, int64_t vd, int max_blocks, float scale2, int window,
                         float* __restrict__ part_o, float* __restrict__ part_ml, int num_splits, int chunk,
                         float cap_in, float cap_out, int sink, const float* __restrict__ sinks,
                         const float* __restrict__ slopes, const float* __restrict__ gate, int64_t gate_stride) {
  __shared__ __attribute__((aligned(1024))) PrefillLds<HD, WHOLE> lds;
  prefill_block<HD, RT, PRE_WAVES, WHOLE, GENERAL>(lds, blockIdx.x, gridDim.x, out, q, k_cache, v_cache, block_tables, seq_of_token, positions, tiles, num_tiles, nh,
                                                   group, dies_per_group, heads_per_group, page_size, page_shift, page_run, kp, ks, kh, vp, vh, vd, max_blocks,
                                                   scale2, window, part_o, part_ml, num_splits, chunk, cap_in, cap_out, sink, sinks, slopes, gate, gate_stride);
}

// A step of decoding tokens beside prompts in one launch: the prompts' workgroups first, then one per (decoding token, key/value head, chunk of keys), as
// attention_decode.hip has them. The ones multiply and take LDS, the others wait for memory, and side by side they take
// little more than the longer of the two, where two launches follow each other. The bits are those of the two launches. us, two launches and one (the combining kernel's
// counted with both): 24 heads of 128, 13 requests of up to 1,700 keys beside prompts of 751 and 750 tokens 48.6 and 41.8, beside 300 tokens 35.1 and 25.4; 32
// heads of 64, 8 requests of 500 beside 64 tokens 13.2 and 8.8, 32 of 1,000 beside 300 21.0 and 16.5, 64 of 2,000 beside 200 50.0 and 43.1, beside 2,000 67.2
// and 64.9; capped, 24 of 900 beside 700 29.1 and 20.2. (Both kinds of workgroup in turn: 58.8 where this order takes 38.9, 8 of 2,000 beside 2,000; two streams, which
// meet in two events: 10 to 15 us more than one launch after the other.)
template <int HD, int RT, int PRE_WAVES, bool ONE, bool GENERAL, bool ONCE>
__global__ void __launch_bounds__(PRE_WAVES * TS_WAVE)
attn_step_kernel(const DecodeArgs d, const int32_t* __restrict__ tiles, int num_tiles, int group, int dies_per_group, int heads_per_group, int prefill_blocks,
                 int decode_waves, int tokens) {
  __shared__ __attribute__((aligned(1024))) PrefillLds<HD, true> lds;
  const int block = blockIdx.x;
  if (block < prefill_blocks) {
    prefill_block<HD, RT, PRE_WAVES, true, GENERAL>(lds, block, prefill_blocks, d.out, d.q, d.k_cache, d.v_cache, d.block_tables, d.seq_of_token, d.positions, tiles,
                                                    num_tiles, d.nh, group, dies_per_group, heads_per_group, d.page_size, d.page_shift, d.page_run, d.kp, d.ks, d.kh,
                                                    d.vp, d.vh, d.vd, d.max_blocks, d.scale2, d.window, nullptr, nullptr, 1, 0, d.cap_in, d.cap_out, d.sink, d.sinks,
                                                    d.slopes, d.gate, d.gate_stride);
    return;
  }
  const int id = block - prefill_blocks, split = id % d.num_splits, rest = id / d.num_splits, heads = d.nh / d.G;
  decode_chunk<HD, ONE, GENERAL, ONCE, true>((float*)&lds, decode_waves, split, rest % heads, rest / heads, tokens, d.out, d.part_o, d.part_ml, d.q, d.k_cache,
                                              d.v_cache, d.block_tables, d.seq_of_token, d.positions, d.nh, d.G, d.page_size, d.page_shift, d.page_run, d.kp, d.ks,
                                              d.kh, d.vp, d.vh, d.vd, d.max_blocks, d.num_splits, d.chunk, d.scale2, d.window, d.cap_in, d.cap_out, d.sink, d.sinks,
                                              d.slopes, d.gate, d.gate_stride);
}

// Keys: rows dense in head_dim, strides kp/ks/kh (page, slot, head). Values: transposed pages,
// slot stride 1, strides vp/vh/vd (page, head, dimension). tile_tokens: the most tokens a listed
// tile holds, waves x RT (16 / G) for RT of 1, 2 or 4 row tiles a wave and 4 waves, or 8 waves with one or two
// (heads of 64 or 128 dimensions). num_splits > 1: chunk (a multiple of 32; the last chunk
// takes every key from its start on) and the float workspaces part_o [num_tokens, nh, num_splits, hd] and
// part_ml [num_tokens, nh, num_splits, 2]; every token from first_token on must then be in a tile (the ones
// before it keep what `out` held). An entry of block_tables names 2^page_run consecutive pages of page_size keys.
static int launch_prefill(void* out, const void* q, const void* k_cache, const void* v_cache,
                          const int32_t* block_tables, const int32_t* seq_of_token,
                          const int32_t* positions, const int32_t* tiles, int num_tiles,
                          int tile_tokens, int waves, int nh, int nkv, int hd, int page_size, int64_t kp,
                          int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks,
                          float scale, int window, int first_token, int num_tokens, int num_splits,
                          int chunk, float* part_o, float* part_ml, int page_run, bool general, float softcap, int sink,
                          const float* sinks, const float* slopes, const float* gate, int64_t gate_stride, hipStream_t stream) {
  if (num_tiles <= 0) return TS_OK;
  if (gate && (!general || (gate_stride < (int64_t)nh * hd && -gate_stride < nh))) return TS_BAD_SHAPE;
  if (general && (page_size % 32 || softcap < 0.f)) return TS_BAD_SHAPE;     // (the general variant walks whole steps only)
  const float log2e = 1.44269504088896340736f;
  const float cap_in = softcap > 0.f ? scale / softcap : 0.f, cap_out = softcap * log2e;
  const float scale2 = softcap > 0.f ? 1.0f : scale * log2e;
  if (num_splits < 1 || num_splits > 65535) return TS_BAD_SHAPE;
  if (num_splits > 1 && (chunk <= 0 || chunk % 32 || !part_o || !part_ml || first_token < 0 || num_tokens <= first_token))
    return TS_BAD_SHAPE;
  if (nkv <= 0 || nh % nkv || page_size <= 0 || page_size % 8 || max_blocks <= 0 || page_run < 0 || page_run > 16) return TS_BAD_SHAPE;
  const int G = nh / nkv;
  if (G > 16) return TS_BAD_SHAPE;
  if (waves != 4 && !(waves == 8 && (hd == 64 || hd == 128))) return TS_BAD_SHAPE;
  const int per_wave = waves * (16 / G);
  if (tile_tokens != per_wave && tile_tokens != 2 * per_wave && !(tile_tokens == 4 * per_wave && waves == 4)) return TS_BAD_SHAPE;
  const int rt = tile_tokens / per_wave, group = G | ((16 / G) << 8) | (((255 + G) / G) << 16);
  if ((kp % 8) || (ks % 8) || (kh % 8) || (vp % 8) || (vh % 8) || (vd % 8)) return TS_BAD_SHAPE;
  if ((((uintptr_t)q) | ((uintptr_t)k_cache) | ((uintptr_t)v_cache)) & 15) return TS_BAD_SHAPE;
  int page_shift = -1;
  if ((page_size & (page_size - 1)) == 0) {
    page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
  }
  int groups = 8;                                   // gcd(nkv, 8)
  while (nkv % groups) groups /= 2;
  const int dies_per_group = 8 / groups, heads_per_group = nkv / groups;
  const int64_t turns = ((int64_t)num_tiles * heads_per_group + dies_per_group - 1) / dies_per_group;
  if (turns * 8 > 0x7fffffff) return TS_BAD_SHAPE;
  dim3 grid((unsigned)(8 * turns), num_splits);
#define TS_PRE_W(HH, RR, WW)                                                                                    \
  if (general) { TS_PRE_P(HH, RR, WW, true, true); }                                                            \
  else if (page_size % 32 == 0) { TS_PRE_P(HH, RR, WW, true, false); } else { TS_PRE_P(HH, RR, WW, false, false); }
#define TS_PRE_P(HH, RR, WW, PP, GG)                                                                            \
  attn_prefill_mfma_kernel<HH, RR, WW, PP, GG><<<grid, WW * TS_WAVE, 0, stream>>>(                              \
      (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables,             \
      seq_of_token, positions, tiles, num_tiles, nh, group, dies_per_group, heads_per_group, page_size, page_shift, page_run, kp,  \
      ks, kh, vp, vh, vd, max_blocks, scale2, window, part_o, part_ml, num_splits, chunk, cap_in, cap_out, sink, sinks, slopes, \
      gate, gate_stride)
#define TS_PRE_RT(HH)                                                                                           \
  if (rt == 1) { TS_PRE_W(HH, 1, 4) } else if (rt == 2) { TS_PRE_W(HH, 2, 4) } else { TS_PRE_W(HH, 4, 4) }
#define TS_PRE_RT8(HH)                                                                                          \
  if (rt == 1) { TS_PRE_W(HH, 1, 8) } else { TS_PRE_W(HH, 2, 8) }
  if (waves == 8) {
    switch (hd) {
      case 64: TS_PRE_RT8(64); break;
      case 128: TS_PRE_RT8(128); break;
      default: return TS_BAD_SHAPE;       // (96: twelve registers a step do not go round eight waves)
    }
  } else {
    switch (hd) {
      case 32: TS_PRE_RT(32); break;
      case 64: TS_PRE_RT(64); break;
      case 96: TS_PRE_RT(96); break;
      case 128: TS_PRE_RT(128); break;
      default: return TS_BAD_SHAPE;
    }
  }
#undef TS_PRE_RT8
#undef TS_PRE_RT
#undef TS_PRE_W
#undef TS_PRE_P
  const int rc = ts_check_launch();
  if (rc || num_splits == 1) return rc;
  const int64_t skip = (int64_t)first_token * nh;     // rows of the tokens before the first listed one
  return ts_launch_attention_combine((bf16_t*)out + skip * hd, part_o + skip * num_splits * hd,
                                     part_ml + skip * num_splits * 2, positions + first_token,
                                     num_tokens - first_token, nh, hd, num_splits, chunk, window, stream, general ? sink : 0,
                                     general ? sinks : nullptr, gate ? gate + (int64_t)first_token * (gate_stride < 0 ? -gate_stride : gate_stride) : nullptr,
                                     gate_stride);
}

extern "C" int ts_paged_attention_prefill(void* out, const void* q, const void* k_cache, const void* v_cache,
                                          const int32_t* block_tables, const int32_t* seq_of_token,
                                          const int32_t* positions, const int32_t* tiles, int num_tiles,
                                          int tile_tokens, int waves, int nh, int nkv, int hd, int page_size, int64_t kp,
                                          int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks,
                                          float scale, int window, int first_token, int num_tokens, int num_splits,
                                          int chunk, float* part_o, float* part_ml, int page_run, hipStream_t stream) {
  return launch_prefill(out, q, k_cache, v_cache, block_tables, seq_of_token, positions, tiles, num_tiles, tile_tokens, waves, nh,
                        nkv, hd, page_size, kp, ks, kh, vp, vh, vd, max_blocks, scale, window, first_token, num_tokens,
                        num_splits, chunk, part_o, part_ml, page_run, false, 0.f, 0, nullptr, nullptr, nullptr, 0, stream);
}

// The same with capped scores (softcap > 0: cap * tanh(score / cap)), a sink (one more in the softmax's
// denominator; `sinks`, float [nh], if given: exp(sinks[head]) more instead), a penalty of slopes[head] (float [nh],
// if given) per position of distance taken off every score, and weights carried in two bfloat16 terms; pages of a
// multiple of 32 keys. `gate` (float [tokens, >= nh hd], rows gate_stride apart; may be null): the output leaves
// multiplied by sigmoid(gate); a stride below zero: one number per head (`ts_out_gate`).
extern "C" int ts_paged_attention_prefill_general(void* out, const void* q, const void* k_cache, const void* v_cache,
                                                  const int32_t* block_tables, const int32_t* seq_of_token,
                                                  const int32_t* positions, const int32_t* tiles, int num_tiles,
                                                  int tile_tokens, int waves, int nh, int nkv, int hd, int page_size,
                                                  int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd,
                                                  int max_blocks, float scale, int window, int first_token,
                                                  int num_tokens, int num_splits, int chunk, float* part_o,
                                                  float* part_ml, int page_run, float softcap, int sink,
                                                  const float* sinks, const float* slopes, const float* gate,
                                                  int64_t gate_stride, hipStream_t stream) {
  return launch_prefill(out, q, k_cache, v_cache, block_tables, seq_of_token, positions, tiles, num_tiles, tile_tokens, waves, nh,
                        nkv, hd, page_size, kp, ks, kh, vp, vh, vd, max_blocks, scale, window, first_token, num_tokens,
                        num_splits, chunk, part_o, part_ml, page_run, true, softcap, sink || sinks, sinks, slopes, gate, gate_stride,
                        stream);
}

// The decoding tokens 0 .. num_tokens - 1 and the tiles' tokens of a step in one launch (attn_step_kernel), then the decoding tokens' chunks combined: what
// ts_paged_attention_decode[_general] and ts_paged_attention_prefill[_general] make of these operands, for pages of whole 32-key steps, heads of 64 (plain or
// general) or 128 (plain) and prompts that are not split.
extern "C" int ts_paged_attention_step(void* out, float* part_o, float* part_ml, const void* q, const void* k_cache, const void* v_cache,
                                       const int32_t* block_tables, const int32_t* seq_of_token, const int32_t* positions, int num_tokens, int num_splits,
                                       int chunk, int decode_waves, const int32_t* tiles, int num_tiles, int tile_tokens, int waves, int nh, int nkv, int hd,
                                       int page_size, int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vh, int64_t vd, int max_blocks, float scale,
                                       int window, int page_run, int general, float softcap, int sink, const float* sinks, const float* slopes,
                                       const float* gate, int64_t gate_stride, hipStream_t stream) {
  if (num_tokens <= 0 || num_tiles <= 0 || nkv <= 0 || nh % nkv || nh / nkv > 16 || page_size <= 0 || page_size % 32 || max_blocks <= 0 || page_run < 0 || page_run > 16)
    return TS_BAD_SHAPE;
  if (!(hd == 64 || (hd == 128 && !general)) || softcap < 0.f || (!general && (softcap > 0.f || sink || sinks || slopes || gate))) return TS_BAD_SHAPE;
  if (gate && gate_stride < (int64_t)nh * hd && -gate_stride < nh) return TS_BAD_SHAPE;
  if (decode_waves < 1 || decode_waves > DEC_WAVES_FOR(hd, chunk == 32 * decode_waves) || chunk <= 0 || chunk % (32 * decode_waves) || num_splits < 1 || num_splits > 1024 || (num_splits > 1 && (!part_o || !part_ml)))
    return TS_BAD_SHAPE;
  const int G = nh / nkv;
  if ((waves != 4 && waves != 8) || decode_waves < waves) return TS_BAD_SHAPE;      // (a workgroup's waves all have chunks to walk)
  const int per_wave = waves * (16 / G), rt = tile_tokens / per_wave, group = G | ((16 / G) << 8) | (((255 + G) / G) << 16);
  if (tile_tokens != rt * per_wave || !(rt == 1 || (rt == 2 && waves == 4))) return TS_BAD_SHAPE;
  if ((size_t)decode_waves * (32 + G * hd) * sizeof(float) > (hd == 64 ? sizeof(PrefillLds<64, true>) : sizeof(PrefillLds<128, true>))) return TS_BAD_SHAPE;
  if ((kp | ks | kh | vp | vh | vd) % 8 || ((((uintptr_t)q) | ((uintptr_t)k_cache) | ((uintptr_t)v_cache)) & 15)) return TS_BAD_SHAPE;
  int groups = 8;                                   // gcd(nkv, 8)
  while (nkv % groups) groups /= 2;
  const int dies_per_group = 8 / groups, heads_per_group = nkv / groups;
  const int64_t turns = ((int64_t)num_tiles * heads_per_group + dies_per_group - 1) / dies_per_group, all = 8 * turns + (int64_t)num_tokens * nkv * num_splits;
  if (all > 0x7fffffff) return TS_BAD_SHAPE;
  int page_shift = -1;
  if ((page_size & (page_size - 1)) == 0) page_shift = __builtin_ctz(page_size);
  const float log2e = 1.44269504088896340736f;
  const bool capped = softcap > 0.f;
  const DecodeArgs d = {(bf16_t*)out, part_o, part_ml, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, seq_of_token, positions, nh, G,
                        page_size, page_shift, page_run, kp, ks, kh, vp, vh, vd, max_blocks, num_splits, chunk, capped ? 1.0f : scale * log2e, window,
                        capped ? scale / softcap : 0.f, softcap * log2e, sink || sinks, sinks, slopes, gate, gate_stride};
  const int64_t reach = (int64_t)num_splits * chunk, within = window < 0 ? -(int64_t)window : window, keys = within && within < reach ? within : reach;
  const bool once = (int64_t)num_tokens * nkv * hd * 4 * keys >= DEC_ONCE_BYTES;
#define TS_STEP(HH, RR, WW, ON, GG, NC) \
  attn_step_kernel<HH, RR, WW, ON, GG, NC><<<(unsigned)all, WW * TS_WAVE, 0, stream>>>(d, tiles, num_tiles, group, dies_per_group, heads_per_group, (int)(8 * turns), decode_waves, num_tokens)
#define TS_STEP_N(HH, RR, WW, ON, GG) if (once) { TS_STEP(HH, RR, WW, ON, GG, true); } else { TS_STEP(HH, RR, WW, ON, GG, false); }
#define TS_STEP_O(HH, RR, WW, GG) if (chunk == 32 * decode_waves) { TS_STEP_N(HH, RR, WW, true, GG) } else { TS_STEP_N(HH, RR, WW, false, GG) }
#define TS_STEP_1(HH, RR, WW, GG) TS_STEP_N(HH, RR, WW, true, GG)
#define TS_STEP_W(HH, GG, EIGHT) \
  if (rt == 2) { TS_STEP_O(HH, 2, 4, GG) } else if (waves == 4) { TS_STEP_O(HH, 1, 4, GG) } else { EIGHT(HH, 1, 8, GG) }
  // (eight waves of wide heads have a single step each: DEC_WAVES_FOR)
  if (hd == 128) { TS_STEP_W(128, false, TS_STEP_1) } else if (general) { TS_STEP_W(64, true, TS_STEP_O) } else { TS_STEP_W(64, false, TS_STEP_O) }
#undef TS_STEP_W
#undef TS_STEP_1
#undef TS_STEP_O
#undef TS_STEP_N
#undef TS_STEP
  const int rc = ts_check_launch();
  if (rc || num_splits == 1) return rc;
  return ts_launch_attention_combine(out, part_o, part_ml, positions, num_tokens, nh, hd, num_splits, chunk, window, stream, general ? (sink || sinks) : 0,
                                     general ? sinks : nullptr, gate, gate_stride);
}
