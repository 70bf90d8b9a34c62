// y[M, N] = x[M, K] · W[N, K]^T in bfloat16 for many rows of x, a workgroup adding up the whole reduction of a tile
// (tile_product.h) and taking it to its place itself: as 32-bit or bfloat16 numbers, or, for the q|k|v projection of an
// attention layer, through the rotation into q and the cache.
//
// What bounds it: from some 800 rows on the matrix cores, at the 1.6 to 1.9 GHz that their power leaves them; at fewer rows the chain of a tile's steps, of
// which each waits for LDS (0.3 µs a step of 64 x 128, whose products take 0.11). Measured with W coming from memory: q|k|v of 32 heads of 64 beside 8 + 8,
// K 2,048, 192 rows 13.8 µs, 513 rows 14.2, 1,024 rows 22.8, 2,048 rows 30.0; the library's product and `rope_store` took 20.9, 20.9, 26.6
// and 37.0. The rotation's kernel read and wrote what the product had just written, and was a launch of its own.
#include "tile_product.h"

#define GW_PRODUCTS 8           // products of one launch
// A product's sums are one chain of its whole reduction, or GW_CHAINS of it, whose sums a tile adds up in memory: as near to 64 bits as the library's for
// small results, which it splits (600 x 64 over 2,048: 1.3e-7, one chain 2.7e-7). A tile of so many chains begins as many times, and the launch begins with
// these: 3,072, 2,048 four times, 64 and 32 columns over 2,048, the last two in chains, 320 rows 26.6 µs, with the two by the library 41.2, all in one chain each 25.3.
#define GW_CHAINS 4

struct WholeProduct {
  const bf16_t *x, *w;
  void* y;                      // [M, N], 32-bit or bfloat16
  int N, first;                 // columns, and its first tile of columns among those of all products
  int chains;                   // that its reduction is cut into, one after the other, each added to y (32-bit)
};
struct WholeArgs {
  WholeProduct p[GW_PRODUCTS];
  int products, M, steps, row_tiles, items, per_die;
  int64_t ldx, ldw;
};

template <int BM, int BN, int WM, int WN, int XN, bool WIDE>
__global__ __launch_bounds__(WM * WN * TS_WAVE, 2) void gemm_whole_kernel(const WholeArgs a) {
  using Tile = TileProduct<BM, BN, WM, WN, XN>;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[Tile::LDS];
  // consecutive workgroups go to different dies: a die takes a run of tiles, those of one slice of W's rows side by side
  const int item = blockIdx.x % 8 * a.per_die + blockIdx.x / 8;
  if (item >= a.items) return;
  const int m0 = item % a.row_tiles * BM, column = item / a.row_tiles;
  int which = 0;
  while (which + 1 < a.products && column >= a.p[which + 1].first) ++which;
  const WholeProduct p = a.p[which];
  const int c0 = (column - p.first) * BN;
  uint32_t xoff[Tile::NX], woff[Tile::NW];
#pragma unroll
  for (int q = 0; q < Tile::NX; ++q) {
    const int at = Tile::x_row(q);
    xoff[q] = (uint32_t)(min(at, a.M - 1 - m0) * a.ldx * 2) + Tile::piece(at);      // (rows past the end: the last one again)
  }
#pragma unroll
  for (int q = 0; q < Tile::NW; ++q) {
    const int at = Tile::w_row(q);
    woff[q] = (uint32_t)(min(at, p.N - 1 - c0) * a.ldw * 2) + Tile::piece(at);
  }
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16, wm = wave_index() % WM, wn = wave_index() / WM;
  float4_t acc[Tile::TN][Tile::TM];
  if constexpr (WIDE) {
    const int base = a.steps / p.chains, longer = a.steps % p.chains;      // (the first chains take a step more where they are uneven)
    int64_t k0 = 0;
#pragma unroll 1
    for (int q = 0; q < p.chains; ++q) {
      const int steps = base + (q < longer ? 1 : 0);
      if (q) __syncthreads();      // every wave has read the chain before's last operands
      Tile::run(lds, load_base(p.x + (int64_t)m0 * a.ldx + k0), load_base(p.w + (int64_t)c0 * a.ldw + k0), xoff, woff, steps, acc);
      k0 += 64 * (int64_t)steps;
#pragma unroll
      for (int i = 0; i < Tile::TM; ++i) {
        const int m = m0 + (wm * Tile::TM + i) * 16 + r;
        const int64_t row = (int64_t)m * p.N;
#pragma unroll
        for (int j = 0; j < Tile::TN; ++j) {
          const int c = c0 + (wn * Tile::TN + j) * 16 + 4 * g;
          if (m < a.M && c < p.N) {
            float4_t* const at = (float4_t*)((float*)p.y + row + c);
            if (q) acc[j][i] += *at;
            *at = acc[j][i];
          }
        }
      }
    }
  } else {
    Tile::run(lds, load_base(p.x + (int64_t)m0 * a.ldx), load_base(p.w + (int64_t)c0 * a.ldw), xoff, woff, a.steps, acc);
#pragma unroll
    for (int i = 0; i < Tile::TM; ++i) {
      const int m = m0 + (wm * Tile::TM + i) * 16 + r;
      const int64_t row = (int64_t)m * p.N;
      // lane (r, g) holds columns 16 j + 4 g .. + 3 of row r: lanes g and g ^ 1 exchange so that each has eight in a row
#pragma unroll
      for (int j = 0; j < Tile::TN; j += 2) {
        const auto lo = __builtin_amdgcn_permlane16_swap(pack_bf16(acc[j][i][0], acc[j][i][1]), pack_bf16(acc[j + 1][i][0], acc[j + 1][i][1]), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(pack_bf16(acc[j][i][2], acc[j][i][3]), pack_bf16(acc[j + 1][i][2], acc[j + 1][i][3]), false, false);
        const int c = c0 + (wn * Tile::TN + j + (g & 1)) * 16 + (g >> 1) * 8;
        if (m < a.M && c < p.N) *(u32x4_t*)((bf16_t*)p.y + row + c) = (u32x4_t){lo[0], hi[0], lo[1], hi[1]};
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int XN>
static int launch_whole(WholeArgs a, bool wide, hipStream_t stream) {
  a.row_tiles = (a.M + BM - 1) / BM;
  int64_t columns = 0;
  for (int i = 0; i < a.products; ++i) {
    a.p[i].first = (int)columns;
    columns += (a.p[i].N + BN - 1) / BN;
  }
  if (columns * a.row_tiles > (1 << 24)) return TS_TOO_LARGE;
  a.items = (int)columns * a.row_tiles, a.per_die = (a.items + 7) / 8;
  if (wide) gemm_whole_kernel<BM, BN, WM, WN, XN, true><<<8 * a.per_die, WM * WN * TS_WAVE, 0, stream>>>(a);
  else gemm_whole_kernel<BM, BN, WM, WN, XN, false><<<8 * a.per_die, WM * WN * TS_WAVE, 0, stream>>>(a);
  return ts_check_launch();
}

static bool narrow(const WholeArgs& a, int bm) {
  int64_t wide = 0, narrow = 0;
  for (int i = 0; i < a.products; ++i) wide += (a.p[i].N + 255) / 256, narrow += (a.p[i].N + 191) / 192;
  const int64_t rows = (a.M + bm - 1) / bm;
  return tiles_go_narrow(rows * wide, rows * narrow, bm);
}

static bool whole_operands_ok(const void* x, const void* w, int K, int64_t ldx, int64_t ldw) {
  return x && w && !(((uintptr_t)x | (uintptr_t)w) & 15) && K > 0 && K % 64 == 0 && K / 64 >= TileProduct<64, 128, 1, 4, 3>::MIN_STEPS && ldx >= K && ldw >= K &&
         ldx % 8 == 0 && ldw % 8 == 0;
}

// `products` of them in one launch (1 to 8), all of M rows and the reduction K: x[i] [M, K] and w[i] [N[i], K] bfloat16, 16-byte aligned, rows
// ldx and ldw elements apart (multiples of 8), y[i] [M, N[i]] contiguous, 16-byte aligned, 32-bit or bfloat16; K a multiple of 64 of at least 3, N[i] of
// 8. tile (rows of x by rows of W of a workgroup): 0 128 x 128, 1 128 x 256, 2 192 x 256, 3 256 x 256, 4 64 x 128; 192 columns for 256 by `tiles_go_narrow`. chained: a bit for each product whose
// reduction is cut into GW_CHAINS chains (32-bit, K of 64 times 3 a chain).
extern "C" int ts_gemm_whole_bf16(int products, void* const* y, const void* const* x, const void* const* w, const int* N, int M, int K, int64_t ldx,
                                  int64_t ldw, int tile, int chained, int out_f32, hipStream_t stream) {
  if (M <= 0) return TS_OK;
  if (products < 1 || products > GW_PRODUCTS || !y || !x || !w || !N || tile < 0 || tile > 4 || chained < 0 || chained >> products) return TS_BAD_SHAPE;
  if (chained && (!out_f32 || K / 64 / GW_CHAINS < TileProduct<64, 128, 1, 4, 3>::MIN_STEPS)) return TS_BAD_SHAPE;
  WholeArgs a = {};
  a.products = products, a.M = M, a.steps = K / 64, a.ldx = ldx, a.ldw = ldw;
  int at[2] = {0, __builtin_popcount(chained)};      // the next place of those in chains, which come first, and of the others
  for (int i = 0; i < products; ++i) {
    if (N[i] <= 0 || N[i] % 8 || !y[i] || ((uintptr_t)y[i] & 15) || !whole_operands_ok(x[i], w[i], K, ldx, ldw)) return TS_BAD_SHAPE;
    const int in_chains = chained >> i & 1;
    a.p[at[!in_chains]++] = {(const bf16_t*)x[i], (const bf16_t*)w[i], y[i], N[i], 0, in_chains ? GW_CHAINS : 1};
  }
  if (256 * ldx * 2 >= (1ll << 31) || 256 * ldw * 2 >= (1ll << 31)) return TS_TOO_LARGE;      // (byte offsets from a tile's start)
  switch (tile) {
    case 0: return launch_whole<128, 128, 2, 2, 2>(a, out_f32, stream);
    case 1: return narrow(a, 128) ? launch_whole<128, 192, 4, 2, 2>(a, out_f32, stream) : launch_whole<128, 256, 2, 4, 2>(a, out_f32, stream);
    case 2: return narrow(a, 192) ? launch_whole<192, 192, 4, 2, 2>(a, out_f32, stream) : launch_whole<192, 256, 2, 4, 2>(a, out_f32, stream);
    case 3: return narrow(a, 256) ? launch_whole<256, 192, 4, 2, 2>(a, out_f32, stream) : launch_whole<256, 256, 2, 4, 2>(a, out_f32, stream);
    default: return launch_whole<64, 128, 1, 4, 3>(a, out_f32, stream);
  }
}

// ---- the q|k|v projection through the rotation into q and the cache ----

struct WholeRopeArgs {
  const bf16_t *x, *w;
  int M, N, steps, row_tiles, items, per_die;
  int64_t ldx, ldw;
  const float* cos_sin;         // [positions, hd], [cos | sin] halves; null: nothing turns
  const int32_t *positions, *slots;
  bf16_t *q_out, *k_cache, *v_cache;      // k_cache null: only q is made
  int nh, nkv, hd, page_size, page_shift;
  int runs;                     // values lie eight slots to a 16-byte piece: page sizes and strides of whole pieces, slots side by side
  int64_t kp, ks, kh, vp, vs, vh, vd;
};

// A wave's columns of the tile are units of 16 HT dimensions of a head's first half and those that turn with them, hd / 2 further on (W's rows are
// fetched in that order), so that a pair meets in a lane; with values, whose pages are transposed, the lanes exchange through LDS, which
// is free by then. The product is rounded as it would be stored, turned and stored as `rope_store` does it.
template <int BM, int BN, int WM, int WN, int XN, int HT>
__global__ __launch_bounds__(WM * WN * TS_WAVE, 2) void gemm_whole_rope_kernel(const WholeRopeArgs a) {
  using Tile = TileProduct<BM, BN, WM, WN, XN>;
  constexpr int PASSES = (Tile::TM + 3) / 4, TP = Tile::TM / PASSES, TOKENS = TP * 16;      // a wave's values go at most 64 tokens at a time
  constexpr int SPAN = TOKENS + 8;                              // numbers between two dimensions of the values in LDS
  constexpr int UNIT = 32 * HT, UNITS = Tile::TN / (2 * HT);    // columns of a unit, and units of a wave
  static_assert(Tile::TN % (2 * HT) == 0 && Tile::TM % PASSES == 0, "a wave has whole units, and passes of as many tokens each");
  static_assert(WM * WN * UNIT * SPAN * 2 <= Tile::LDS, "the values' way through LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[Tile::LDS];
  const int item = blockIdx.x % 8 * a.per_die + blockIdx.x / 8;
  if (item >= a.items) return;
  const int m0 = item % a.row_tiles * BM, u0 = item / a.row_tiles * (BN / UNIT);      // first row, and first unit
  const int units = a.N / UNIT, per_head = a.hd / UNIT, half = a.hd / 2;
  uint32_t xoff[Tile::NX], woff[Tile::NW];
#pragma unroll
  for (int q = 0; q < Tile::NX; ++q) {
    const int at = Tile::x_row(q);
    xoff[q] = (uint32_t)(min(at, a.M - 1 - m0) * a.ldx * 2) + Tile::piece(at);      // (rows past the end: the last one again)
  }
#pragma unroll
  for (int q = 0; q < Tile::NW; ++q) {
    const int at = Tile::w_row(q), u = min(u0 + at / UNIT, units - 1), in = at % UNIT;
    const int row = u / per_head * a.hd + u % per_head * (UNIT / 2) + in % (UNIT / 2) + (in >= UNIT / 2 ? half : 0);
    woff[q] = (uint32_t)(row * a.ldw * 2) + Tile::piece(at);
  }
  const int lane = threadIdx.x % TS_WAVE, r = lane % 16, g = lane / 16, wave = wave_index(), wm = wave % WM, wn = wave / WM;
  const int first = m0 + wm * Tile::TM * 16;
  int position[Tile::TM], slot[Tile::TM];
#pragma unroll
  for (int i = 0; i < Tile::TM; ++i) {
    const int m = min(first + 16 * i + r, a.M - 1);
    position[i] = a.cos_sin ? a.positions[m] : 0;
    slot[i] = a.k_cache ? a.slots[m] : -1;
  }
  float4_t acc[Tile::TN][Tile::TM];
  Tile::run(lds, load_base(a.x + (int64_t)m0 * a.ldx), load_base(a.w), xoff, woff, a.steps, acc);
  const int values = (a.nh + a.nkv) * per_head;      // the first unit of the values
  if (a.k_cache && u0 + BN / UNIT > values) __syncthreads();      // every wave has read its last operands: LDS is free
  auto page_of = [&](int s) { return a.page_shift >= 0 ? s >> a.page_shift : s / a.page_size; };
  bf16_t* turn = (bf16_t*)lds + wave * (UNIT * SPAN);
#pragma unroll
  for (int w = 0; w < UNITS; ++w) {
    const int u = u0 + wn * UNITS + w, head = u / per_head, d0 = u % per_head * (UNIT / 2);      // the unit's head, and the first of its dimensions in the first half
    if (u >= units || (head >= a.nh && !a.k_cache)) return;
    if (u < values) {
#pragma unroll
      for (int i = 0; i < Tile::TM; ++i) {
        const int m = first + 16 * i + r;
        uint32_t p[2][HT][2];      // [half][tile of the half][pair]
#pragma unroll
        for (int j = 0; j < HT; ++j) {
          float y[2][4];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const float4_t& at = acc[(2 * w + h) * HT + j][i];
              const uint32_t both = pack_bf16(at[2 * e], at[2 * e + 1]);      // as the product would be stored
              y[h][2 * e] = __uint_as_float(both << 16), y[h][2 * e + 1] = __uint_as_float(both & 0xffff0000u);
            }
          if (a.cos_sin) {
            const float* at = a.cos_sin + (int64_t)position[i] * a.hd + d0 + 16 * j + 4 * g;
            const float4 c = *(const float4*)at, s = *(const float4*)(at + half);
            const float cs[4] = {c.x, c.y, c.z, c.w}, sn[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float y1 = fmaf(y[0][e], cs[e], -(y[1][e] * sn[e])), y2 = fmaf(y[1][e], cs[e], y[0][e] * sn[e]);      // (as rope_store's are compiled)
              y[0][e] = y1, y[1][e] = y2;
            }
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) p[h][j][0] = pack_bf16(y[h][0], y[h][1]), p[h][j][1] = pack_bf16(y[h][2], y[h][3]);
        }
        bf16_t* dst = nullptr;
        if (m < a.M) {
          if (head < a.nh) {
            dst = a.q_out + ((int64_t)m * a.nh + head) * a.hd;
          } else if (slot[i] >= 0) {
            const int page = page_of(slot[i]);
            dst = a.k_cache + (int64_t)page * a.kp + (int64_t)(slot[i] - page * a.page_size) * a.ks + (int64_t)(head - a.nh) * a.kh;
          }
        }
        // lane (r, g) holds four dimensions of each of two tiles (of one half; of both, where a half is one tile): lanes g and g ^ 1 exchange
        // so that each has eight in a row
#pragma unroll
        for (int h = 0; h < HT; ++h) {
          const uint32_t(&one)[2] = HT == 2 ? p[h][0] : p[0][0], (&other)[2] = HT == 2 ? p[h][HT - 1] : p[1][0];
          const auto lo = __builtin_amdgcn_permlane16_swap(one[0], other[0], false, false);
          const auto hi = __builtin_amdgcn_permlane16_swap(one[1], other[1], false, false);
          const int at = HT == 2 ? h * half + (g & 1) * 16 : (g & 1) * half;
          if (dst) *(u32x4_t*)(dst + at + d0 + (g >> 1) * 8) = (u32x4_t){lo[0], hi[0], lo[1], hi[1]};
        }
      }
      continue;
    }
    // ---- values: [dimension of the unit][token] in LDS, then eight slots a store wherever eight tokens of this wave have slots in a row
    // that begin at a multiple of eight, a store a token for the others
    bf16_t* const base = a.v_cache + (int64_t)(head - a.nh - a.nkv) * a.vh;
    auto dimension = [&](int d) { return d0 + d % (UNIT / 2) + (d >= UNIT / 2 ? half : 0); };
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      const int begin0 = first + pass * TOKENS;
      if (w || pass) wave_sync();      // the unit or pass before has been read
#pragma unroll
      for (int i = 0; i < TP; ++i)
#pragma unroll
        for (int j = 0; j < 2 * HT; ++j)
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            const float4_t& at = acc[2 * HT * w + j][pass * TP + i];
            const uint32_t both = pack_bf16(at[e], at[e + 1]);
            turn[(16 * j + 4 * g + e) * SPAN + 16 * i + r] = (bf16_t)both;
            turn[(16 * j + 4 * g + e + 1) * SPAN + 16 * i + r] = (bf16_t)(both >> 16);
          }
      wave_sync();
      const int mine = lane < TOKENS && begin0 + lane < a.M ? a.slots[begin0 + lane] : -1, in_run = mine & 7, begin = lane - in_run;
      bool whole = a.runs && mine >= 0 && begin >= 0 && begin + 7 < TOKENS;
#pragma unroll
      for (int k = 0; k < 8; ++k) whole = (__shfl(mine, (begin + k) & (TS_WAVE - 1), TS_WAVE) == mine - in_run + k) & whole;
      const uint64_t runs = __ballot(whole && in_run == 0), singles = __ballot(mine >= 0 && !whole);
      if (runs) {
        // eight lanes take the runs, eight dimensions at a time (so that a dimension's runs leave together)
        uint64_t left = runs;
        for (int k = 0; k < lane % 8; ++k) left &= left - 1;
        const int t = left ? __builtin_ctzll(left) : -1, s0 = __shfl(mine, t & (TS_WAVE - 1), TS_WAVE), page = page_of(s0);
        bf16_t* const to = base + (int64_t)page * a.vp + (s0 - page * a.page_size);
        const bool in_pieces = !(runs & ~0x0101010101010101ull);
        if (t >= 0) {
#pragma unroll
          for (int q = 0; q < UNIT / 8; ++q) {
            const int d = lane / 8 + 8 * q;
            const bf16_t* from = turn + d * SPAN + t;
            u32x4_t v;
            if (in_pieces) {
              v = *(const u32x4_t*)from;
            } else {
#pragma unroll
              for (int k = 0; k < 4; ++k) v[k] = (uint32_t)from[2 * k] | ((uint32_t)from[2 * k + 1] << 16);
            }
            *(u32x4_t*)(to + (int64_t)dimension(d) * a.vd) = v;
          }
        }
      }
      for (uint64_t left = singles; left; left &= left - 1) {
        const int t = __builtin_ctzll(left), s = __builtin_amdgcn_readlane(mine, t), page = page_of(s);
        if (UNIT == TS_WAVE || lane < UNIT)
          base[(int64_t)page * a.vp + (int64_t)(s - page * a.page_size) * a.vs + (int64_t)dimension(lane) * a.vd] = turn[lane * SPAN + t];
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int XN, int HT = 2>
static int launch_whole_rope(WholeRopeArgs a, hipStream_t stream) {
  a.row_tiles = (a.M + BM - 1) / BM;
  const int64_t items = (int64_t)a.row_tiles * ((a.N + BN - 1) / BN);
  if (items > (1 << 24)) return TS_TOO_LARGE;
  a.items = (int)items, a.per_die = (a.items + 7) / 8;
  gemm_whole_rope_kernel<BM, BN, WM, WN, XN, HT><<<8 * a.per_die, WM * WN * TS_WAVE, 0, stream>>>(a);
  return ts_check_launch();
}

// `ts_rope_store` of x [M, K] · w [(nh + 2 nkv) hd, K]^T (operands as for ts_gemm_whole_bf16) rounded to bfloat16, whole heads turned by the
// table or, with cos_sin null, none; hd a multiple of 64, the table, q_out, the key cache and its strides in whole 16-byte pieces. tile (rows of x
// by rows of W of a workgroup): 0 128 x 128, 1 128 x 256, or x 192 where that is no more than a workgroup a compute unit either (the same bits: 3,072 columns
// over 2,048, 2,048 rows 192 workgroups of 32.7 us and 256 of 30.0, 1,400 rows 32.1 and 28.4; 5,120 over 3,072, 1,024 rows 46.9 and 41.5, 1,280 rows,
// 270 of them (left) 47.3 and 70.1; of two rounds either way, 1,700 rows (left) 78.1 and 78.3), 2 192 x 256, 3 64 x 128.
extern "C" int ts_gemm_whole_rope_bf16(void* q_out, const void* x, const void* w, int M, int K, int64_t ldx, int64_t ldw, const float* cos_sin,
                                       const int32_t* positions, const int32_t* slots, void* k_cache, void* v_cache, int nh, int nkv, int hd, int page_size,
                                       int64_t kp, int64_t ks, int64_t kh, int64_t vp, int64_t vs, int64_t vh, int64_t vd, int tile, hipStream_t stream) {
  if (M <= 0) return TS_OK;
  if (nh <= 0 || nkv < 0 || hd <= 0 || hd % 64 || page_size <= 0 || tile < 0 || tile > 3 || !whole_operands_ok(x, w, K, ldx, ldw)) return TS_BAD_SHAPE;
  const int64_t N = ((int64_t)nh + 2 * (int64_t)nkv) * hd;
  if (!q_out || ((uintptr_t)q_out & 15) || (cos_sin && (!positions || ((uintptr_t)cos_sin & 15)))) return TS_BAD_SHAPE;
  if (k_cache && (!v_cache || !slots || kp % 8 || ks % 8 || kh % 8 || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 1))) return TS_BAD_SHAPE;
  if (256 * ldx * 2 >= (1ll << 31) || N * ldw * 2 >= (1ll << 31)) return TS_TOO_LARGE;      // (byte offsets from a tile's start, and from W's)
  WholeRopeArgs a = {(const bf16_t*)x, (const bf16_t*)w, M, (int)N, K / 64, 0, 0, 0, ldx, ldw, cos_sin, positions, slots, (bf16_t*)q_out, (bf16_t*)k_cache,
                     (bf16_t*)v_cache, nh, nkv, hd, page_size, (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1, 0, kp, ks, kh, vp, vs, vh, vd};
  a.runs = vs == 1 && page_size % 8 == 0 && vp % 8 == 0 && vh % 8 == 0 && vd % 8 == 0 && !((uintptr_t)v_cache & 15);
  switch (tile) {
    case 0: return launch_whole_rope<128, 128, 2, 2, 2>(a, stream);
    case 1:
      if ((int64_t)((M + 127) / 128) * ((N + 191) / 192) <= COMPUTE_UNITS) return launch_whole_rope<128, 192, 4, 2, 2, 1>(a, stream);
      return launch_whole_rope<128, 256, 2, 4, 2>(a, stream);
    case 2: return launch_whole_rope<192, 256, 2, 4, 2>(a, stream);
    default: return launch_whole_rope<64, 128, 2, 2, 3>(a, stream);
  }
}
