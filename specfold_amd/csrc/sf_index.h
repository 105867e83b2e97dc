// Integer index maps of the kernels, shared with their CPU checker.
//
// Plain integer functions: the stream-K schedule of the weight-streaming GEMMs
// and their output-column / packed-weight addressing, and the prefix attention's
// work decomposition, key-slot permutation, V^T swizzle and page-group
// addressing.  Under hipcc they are host+device functions used by the kernels
// and the launchers; under a plain C++ compiler they build on their own, so the
// CPU test tests/cpp/index_check.cpp walks them over the shapes the entry points
// accept and checks that every access lands inside its buffer, every unit of
// work is done exactly once and the kernels that pass work to each other agree
// on its layout.
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define SF_IDX __host__ __device__ __forceinline__
#else
#define SF_IDX inline
#endif

SF_IDX int sf_imin(int a, int b) { return a < b ? a : b; }
SF_IDX int sf_imax(int a, int b) { return a > b ? a : b; }

// ---------------------------------------------------------------------------
// Weight-streaming GEMM (sf_gemm_core.h)
// ---------------------------------------------------------------------------
namespace sfg {

// Packed ("fragment-major") weights: for each 16-row tile of W [N, K] and each
// 32-wide K chunk, the 64 lanes' MFMA B fragments (lane l holds
// W[16t + l%16][32c + 8(l/16) .. +8]) are one contiguous 1 KB block, and the
// chunks of a tile follow each other.
constexpr int kKsStride = 512;     // elements between 32-wide chunks of a tile
constexpr int kKC = 64;            // K per stage: two 32-wide MFMA chunks
constexpr int kLdsBudget = 152 * 1024;  // LDS of a stage ring
#ifndef SFG_RING_MAX
#define SFG_RING_MAX 6
#endif

// Lane `lane`'s first fragment of 16-row tile `tile16`, from base W (a pointer to
// the packed weights in the kernels; an integer 0 gives the element offset).
template <typename P>
SF_IDX P weight_lane_ptr(P W, int tile16, int K, int lane) {
  return W + (size_t)tile16 * (K / 32) * 512 + lane * 8;
}

// A stage of the GEMM core is 64 K, two 32-wide MFMA chunks; chunk c of stage sc:
SF_IDX int weight_chunk(int sc, int c) { return 2 * sc + c; }

// A operand in LDS: per m tile 16 rows x 128 bytes (a stage's 64 K), brought by two
// direct copies of 8 rows each, so that every copy takes whole 128-byte cache lines.
// (Two copies that share a line stall the vector cache: the second hits a line whose
// data is still on its way.)  Copy j of wave wv is a_copy(wv, j, NMT) of the 2·NMT (waves
// with fewer real copies repeat the last one).  Word r*8 + (u ^ r%8) holds unit u of row
// r: lane L of a copy brings unit a2_copy_unit(L) of row L/8; the MFMA reader lane l of
// chunk k (unit 4k + l/16 of row l%16) reads word a2_read_word(l, k).
SF_IDX int a_copy(int wv, int j, int NMT) { return sf_imin(wv + 8 * j, 2 * NMT - 1); }
SF_IDX int a2_copy_unit(int L) { return (L & 7) ^ (L >> 3); }
SF_IDX int a2_read_word(int l, int k) {
  return (l & 15) * 8 + ((4 * k + (l >> 4)) ^ (l & 7));
}

// Output column held by lane `lane` of wave `wv` (its column group) in its column
// tile `tt` of 128·WN-column tile t (WN tiles of 16 per wave).  SILU: the gate and
// the up tile of one wave cover the same 16 columns of a 128-column tile.
template <int WN, bool SILU>
SF_IDX int gemm_col(int t, int wv, int tt, int lane) {
  return SILU ? t * 128 + wv * 16 + (lane & 15)
              : t * 128 * WN + wv * 16 * WN + tt * 16 + (lane & 15);
}

// Stream-K schedule.  The output columns are cut into T tiles and K into S
// stages of 64; the T*S (tile, stage) units are dealt out in tile-major order,
// U consecutive units per workgroup.
#ifndef SFG_GRID
#define SFG_GRID 256   // workgroups (MI355X: one 8-wave workgroup per CU)
#endif

struct Plan {
  int T;       // column tiles
  int S;       // K stages
  int U;       // units per workgroup
  int NU = 0;  // > 0: column-spread plan (below) over NU column units of 16
  int KS = 0;  // > 0: split plan (below), KS workgroups per tile
};

// Balanced plan over SFG_GRID workgroups.
inline Plan make_plan(int T, int S) {
  const long long units = (long long)T * S;
  const int U = (int)((units + SFG_GRID - 1) / SFG_GRID);
  return Plan{T, S, U < 1 ? 1 : U};
}
// One workgroup per whole tile: every tile has a single contributor.
inline Plan make_plan_whole(int T, int S) { return Plan{T, S, S}; }
// Column-spread plan (gate/up: kSilu only): the NU 16-column units of the output
// are dealt out over T workgroups, workgroup t taking units [spread_begin(t),
// spread_begin(t + 1)) -- between 1 and 8, one per wave -- over all S stages of K.
// Every tile (a workgroup's columns) is whole, so there are no partial slots, and
// every CU streams NU/T units instead of the 8 of a 128-column tile.
inline Plan make_plan_spread(int NU, int S, int T) { return Plan{T, S, S, NU}; }
SF_IDX int spread_begin(int t, const Plan& p) { return (int)((long long)t * p.NU / p.T); }
// Workgroups of a column-spread plan over nu units: the fewest that give none more
// than ceil(nu / grid) units, so all but a few carry the same count (a full grid
// of 4 and 5 units leaves the CUs with 4 idle through the last fifth of the
// stream, when the others no longer fill HBM).
SF_IDX int spread_workgroups(int nu, int grid) {
  const int k = (nu + grid - 1) / grid;
  return (nu + k - 1) / k;
}
// Split plan: each of the T tiles is cut into KS ranges of whole K stages (range
// j: [split_begin(j), split_begin(j + 1))), one workgroup each, so T·KS workgroups
// each hold a single piece -- no range crosses a tile, so no workgroup pays a
// second ring fill and epilogue (the stream-K ranges that straddle two tiles
// finish last) -- and range j of a tile goes to partial slot j.  KS is the most
// that keeps T·KS within the grid and min_stages stages in a range.
inline Plan make_plan_split(int T, int S, int min_stages = 1) {
  int ks = SFG_GRID / T;
  ks = sf_imax(1, sf_imin(ks, S / min_stages));
  return Plan{T, S, (S + ks - 1) / ks, 0, ks};
}
SF_IDX int split_begin(int j, const Plan& p) { return (int)((long long)j * p.S / p.KS); }

SF_IDX int plan_grid(const Plan& p) {
  if (p.KS) return p.T * p.KS;
  return (int)(((long long)p.T * p.S + p.U - 1) / p.U);
}
// Upper bound of contributors (slots) per tile.
inline int plan_slots(const Plan& p) {
  if (p.KS) return p.KS;
  return p.U >= p.S ? 2 : (p.S + p.U - 1) / p.U + 1;
}

// First and last workgroup holding units of tile t; a piece of tile t computed by
// workgroup g goes to partial slot g - tile_first(t).
SF_IDX int tile_first(int t, const Plan& p) {
  if (p.KS) return t * p.KS;
  return (int)((long long)t * p.S / p.U);
}
SF_IDX int tile_last(int t, const Plan& p) {
  if (p.KS) return t * p.KS + p.KS - 1;
  return (int)(((long long)(t + 1) * p.S - 1) / p.U);
}

// Workgroup g's units are [plan_range_begin(g), plan_range_end(g)) in tile-major
// unit order (unit t·S + s): [g·U, min((g + 1)·U, T·S)) for stream-K and the
// spread plan, range g % KS of tile g / KS for a split plan.
SF_IDX int plan_range_begin(int g, const Plan& p) {
  if (p.KS) return (g / p.KS) * p.S + split_begin(g % p.KS, p);
  return g * p.U;
}
SF_IDX int plan_range_end(int g, const Plan& p) {
  if (p.KS) return (g / p.KS) * p.S + split_begin(g % p.KS + 1, p);
  const int total = p.T * p.S;
  return sf_imin((g + 1) * p.U, total);
}

// The piece of a workgroup's range that starts at unit u: tile t, stages [sa, sb).
struct Piece {
  int t, sa, sb;
};
SF_IDX Piece plan_piece(int u, int u_end, const Plan& p) {
  const int t = u / p.S;
  const int sa = u - t * p.S;
  return Piece{t, sa, sf_imin(p.S, sa + (u_end - u))};
}

// Partial slots of a plan: [plan_slots][mcap][N] fp32.
inline size_t part_bytes(const Plan& p, int mcap, int N) {
  return (size_t)plan_slots(p) * mcap * N * sizeof(float);
}

// ---------------------------------------------------------------------------
// All-rows GEMM (sf_gemm_rows.h): every row of A, up to 128·RG, in one pass over
// the weights.  The 8 waves are RG row groups (128 rows each) x CG = 8 / RG
// column groups (WN tiles of 16 columns each), so a workgroup tile is 16·WN·CG
// columns by all rows.  K (S stages of 64) is cut into KS ranges of whole stages;
// workgroup g computes range s of tile t, (s, t) = item rows_item(g) in split-major
// order.  KS > 1 leaves KS fp32 partial sums per output for the consumer to add
// in range order.
struct RowsPlan {
  int T;   // column tiles
  int KS;  // K ranges
  int S;   // K stages
};
// KS fills SFG_GRID workgroups without exceeding ks_max (1 where the caller has
// no partial buffer) or an eighth of the stages (a range of at least 8 stages
// keeps the partial traffic below the weight stream's).
inline RowsPlan make_rows_plan(int T, int S, int ks_max) {
  int ks = SFG_GRID / T;
  ks = sf_imin(ks, (S + 7) / 8);
  ks = sf_imin(ks, ks_max);
  return RowsPlan{T, ks < 1 ? 1 : ks, S};
}
SF_IDX int rows_grid(const RowsPlan& p) { return p.T * p.KS; }
// Workgroup g runs on XCD g % 8; the G items are numbered so that one XCD's
// workgroups take consecutive items (split-major: they share their K range of A,
// which stays in that XCD's L2).  A bijection of [0, G).
SF_IDX int rows_item(int g, int G) {
  const int x = g & 7;
  return x * (G >> 3) + sf_imin(x, G & 7) + (g >> 3);
}
SF_IDX int rows_split_begin(int s, const RowsPlan& p) {
  return (int)((long long)p.S * s / p.KS);
}
// Stage layout of a workgroup of RG row groups and WN 16-column tiles per wave,
// CPS 32-wide K chunks per stage.  The copies of a stage are dealt over the 8 waves
// (copy q = wv + 8j); a wave with fewer real copies repeats the last one (the same
// bytes to the same place), so every wave issues the same number per stage.
#ifndef SFG_ROWS_CPS
#define SFG_ROWS_CPS 2
#endif
template <int RG, int WN, int CPS = SFG_ROWS_CPS>
struct RowsStage {
  static constexpr int kMB = 128 * RG;       // rows per pass
  static constexpr int kMT = kMB / 16;       // m tiles
  static constexpr int kCG = 8 / RG;         // column groups
  static constexpr int kTW = kCG * WN;       // 16-column tiles of a workgroup tile
  static constexpr int kCPS = CPS;           // K chunks per stage
  static constexpr int kKS = 32 * CPS;       // K per stage
  static constexpr int kNA = CPS * kMT;      // A tile copies per stage
  static constexpr int kNW = CPS * kTW;      // weight block copies per stage
  static constexpr int kA = kNA * 64;        // 16-byte words of A per stage
  static constexpr int kW = kNW * 64;        // words of weights per stage
  static constexpr int kWords = kA + kW;
  static constexpr int kDA = (kNA + 7) / 8;  // A copies per wave per stage
  static constexpr int kDW = (kNW + 7) / 8;  // weight copies per wave per stage
  static constexpr int kRing =
      kLdsBudget / (kWords * 16) < SFG_RING_MAX ? kLdsBudget / (kWords * 16) : SFG_RING_MAX;
};
// A pass of at most 128 rows uses one row group (RG = 1, 8 column groups) with
// half the tiles per wave (at least one), a pass of up to 256 rows two; WN is
// the two-group configuration's.
inline int rows_rg(int mb) { return mb <= 128 ? 1 : 2; }
template <int WN>
constexpr int rows_wn(int rg) { return rg == 2 ? WN : (WN > 1 ? WN / 2 : 1); }
template <int WN>
inline int rows_tiles(int N, int rg) { return N / (16 * rows_wn<WN>(rg) * (8 / rg)); }
// K stages of an all-rows GEMM (32·CPS each).
inline int rows_stages(int K) { return K / (32 * SFG_ROWS_CPS); }
// K ranges of an all-rows GEMM over M rows: those of a pass of up to 256, whatever
// computes more rows (the consumer adds the same number of partial slots for each).
template <int WN>
inline int rows_splits(int M, int N, int K, int ks_max) {
  const int rg = rows_rg(sf_imin(256, M));
  return make_rows_plan(rows_tiles<WN>(N, rg), rows_stages(K), ks_max).KS;
}
// Copy q of a stage (clamped to the last real copy): rows 8q .. +8 of A; weight block
// (tile q / CPS, chunk q % CPS).
SF_IDX int rows_a_copy(int q, int NA) { return sf_imin(q, NA - 1); }
SF_IDX int rows_w_copy(int q, int NW) { return sf_imin(q, NW - 1); }
SF_IDX int rows_w_tile(int q, int CPS) { return q / CPS; }
SF_IDX int rows_w_chunk(int q, int CPS) { return q % CPS; }
// fp32 partials of a plan for M rows and N columns: [KS][M][N].
inline size_t rows_part_bytes(const RowsPlan& p, int M, int N) {
  return p.KS > 1 ? (size_t)p.KS * M * N * sizeof(float) : 0;
}

// ---------------------------------------------------------------------------
// Tile GEMM (sf_gemm_tile.h): more than kTileRows rows.  M rows are cut into
// tile_blocks(M) blocks of at most 256, all of 64·tile_nmt(M) rows (the last one
// shorter); a workgroup tile is one block by 32·NT columns, K cut into ks ranges.
constexpr int kTileRows = 128;       // rows one pass of the streaming core holds
constexpr int kTileMaxBlocks = 4;    // <= 1024 rows
SF_IDX int tile_blocks(int M) { return (M + 255) / 256; }
SF_IDX int tile_nmt(int M) {
  const int nb = tile_blocks(M);
  return (M + nb - 1) / nb <= 192 ? 3 : 4;
}
// The ring of a workgroup tile of 64·NMT rows x 32·NT columns.
template <int NMT, int NT>
struct TileShape {
  static constexpr int kRB = 64 * NMT;            // rows of a block
  static constexpr int kAW = 8 * NMT * 64;        // 16-byte words of A per stage (64 K)
  static constexpr int kNW = 2 * NT;              // weight copies (1 KB) per chunk (32 K)
  static constexpr int kWW = kNW * 64;            // words of weights per chunk
  // A stages: 3 (copied two stages ahead) where four weight chunks fit beside them
  static constexpr int kRA = (kLdsBudget / 16 - 3 * kAW) / kWW >= 4 ? 3 : 2;
  static constexpr int kRWmax = (kLdsBudget / 16 - kRA * kAW) / kWW;
  static constexpr int kRW = kRWmax < 6 ? kRWmax : 6;   // weight chunks
  static constexpr int kWords = kRA * kAW + kRW * kWW;
  static constexpr int kCW = (kNW + 7) / 8;       // weight copies per wave (the last: waves
  static constexpr int kRem = kNW % 8;            // below kRem, if it is not 0)
  static_assert(kRW >= 3 && kRW >= 2 * kRA - 2, "ring depths");
  // Copies go out in windows, window c from chunk c's barrier to chunk c + 1's: the A
  // rows of stage (c - 1)/2 + kRA when c is odd, then the weights of chunk c - 1 + kRW.
  // Copies of a wave (w weight copies per chunk) in windows [a, b).
  static constexpr int window_copies(int a, int b, int w) {
    int n = 0;
    for (int v = a; v < b; ++v) n += (v - 1 + kRW >= 0 ? w : 0) + ((v & 1) ? NMT : 0);
    return n;
  }
  // Younger copies than those chunk c + 1 needs, at chunk c's barrier (c = 2 + k stands
  // for every c of its parity once the windows are regular): its weights went out in
  // window c + 2 - kRW, and when c is odd the A rows of its stage in c + 2 - 2 kRA.
  static constexpr int in_flight(int k, int w) {
    const int c = 2 * kRA + 2 * kRW + k;
    const int nw = window_copies(c + 3 - kRW, c, w);
    const int na = w + window_copies(c + 3 - 2 * kRA, c, w);
    return k == 1 && na < nw ? na : nw;
  }
  // ... than those chunk 0 needs, after the prologue (windows below 0)
  static constexpr int in_flight_first(int w) {
    const int nw = window_copies(2 - kRW, 0, w);
    const int na = (2 - 2 * kRA - 1 + kRW > 0 ? w : 0) + window_copies(2 - 2 * kRA, 0, w);
    return na < nw ? na : nw;
  }
  // chunks before the end at which the windows stop being regular
  static constexpr int kTail = 2 * kRA > kRW - 1 ? 2 * kRA : kRW - 1;
};

// The order of a wave's LDS reads and how many of them may be in flight at each use.
// The MFMAs of a chunk go in NT steps, step t those of weight tile t with the NMT A
// tiles; D steps ahead of it the step's fragments are read: step t reads weight
// fragment t + D of its chunk while t < NT - D, and from step NT - D on, fragment
// j = t - (NT - D) of the NEXT chunk, the first NA0 of its A fragments in front of
// j = 0 and the others in front of j = 1 (D = 1: all in front of j = 0).
template <int NMT, int NT>
struct TileSteps {
  static constexpr int kD = NT >= 4 ? 3 : NT - 1;
  static constexpr int kNA0 = kD == 1 ? NMT : (NMT + 1) / 2;
  static constexpr int a_reads(int j) { return j == 0 ? kNA0 : j == 1 ? NMT - kNA0 : 0; }
  static constexpr int reads(int t) { return t < NT - kD ? 1 : 1 + a_reads(t - (NT - kD)); }
  // reads issued after the ones step t uses, its own step's reads included
  static constexpr int later(int t) {
    int n = 0;
    for (int i = 1; i <= kD; ++i) n += reads((t - kD + i + NT) % NT);
    // step 0 also takes the A fragments, the last of them in front of j = 1's weight
    // fragment: of the reads after j = 0's, those A reads must have landed too
    if (t == 0 && kD > 1) n -= a_reads(1);
    return n;
  }
};

struct TilePlans {
  int ks = 1;        // K ranges
  unsigned nt = 0;   // byte tile_blocks(M) - 1: NT, or 0: such rows stay on the streaming core
};
SF_IDX int tile_nt(int M, const TilePlans& p) { return (p.nt >> (8 * (tile_blocks(M) - 1))) & 255; }
// A table of `rows` rows of K that the tile GEMM's 32-bit row offsets reach (64-bit ones
// take its copies a few cycles more: a prefill of 2048 tokens 6812 -> 6867 us).
inline bool tile_reach(long long rows, int K) { return rows * K * 2 <= 1ll << 32; }
// Whether the tile GEMM computes M rows.
SF_IDX bool tile_takes(int M, const TilePlans& p) { return M > kTileRows && tile_nt(M, p) != 0; }
// Cycles of a workgroup per 32-wide K chunk: the LDS operand reads of 8 waves
// (128 B a cycle) with the copies' writes, or two waves' MFMAs per SIMD.
inline long long tile_chunk_cycles(int nmt, int nt) {
  const long long lds = (nmt + nt) * 64 + (4 * nmt + 2 * nt) * 8;
  const long long mfma = nmt * nt * 32;
  return lds > mfma ? lds : mfma;
}
// NT of the tile GEMM of `units` 16-column units (silu: gate units; the up units are
// as many again) over K in ks ranges, for every row-block count: the lowest estimate
// of whole rounds of the grid (never below the weight stream, ~2000 bytes a cycle)
// and a fixed cost per item.  The K ranges are those of the streaming core's plan
// (a whole K, or its split plan), so a row's sums are the same for every row count.
// Short ranges are all ring fill and partial sums, and the streaming core's narrower
// pieces overlap those of several passes: with K cut up, the tile GEMM takes rows from
// 3 / 2 / 2 / 1 stages in a range on, on average, for 1 / 2 / 3 / 4 row blocks.  Measured,
// streaming -> tile, us, ranges of 1.0 to 1.4 / 2 / 2.75 / 3.3 to 3.6 stages:
//   256 rows: down 1024 x 1408 18.8 -> 21.9 / QKV 2048 x 1536 22.2 -> 25.4 / down
//     2048 x 2816 22.5 -> 25.9 / down 768 x 8960 31.2 -> 24.3, 1536 x 4864 29.6 -> 24.5
//   257-320: down 2048 x 1408 23.0 -> 26.0 / QKV 29.4 -> 29.5 (512: 38.0 -> 34.2) / 28.8 ->
//     27.3 / 37.1 -> 29.1, 35.1 -> 28.6
//   640: down 1024 x 1408 35.6 -> 37.3 / QKV 46.0 -> 45.9 / 48.3 -> 47.7 / 63.3 -> 51.1
//   1024: down 1024 x 1408 53.1 -> 45.5 / QKV 72.8 -> 57.8 / 74.5 -> 60.0 / 99.0 -> 62.0
inline TilePlans make_tile_plans(int units, int K, bool silu, int ks) {
  TilePlans p;
  p.ks = ks;
  for (int b = 1; b <= kTileMaxBlocks; ++b) {
    long long best = -1;
    unsigned best_nt = 0;
    for (int nt = 2; nt <= 8; ++nt) {
      if (silu ? nt == 2 : (nt != 2 && nt != 4 && nt != 8)) continue;
      const int per = silu ? nt : 2 * nt;
      const int T = (units + per - 1) / per;
      const long long rounds = ((long long)T * b * ks + SFG_GRID - 1) / SFG_GRID;
      long long cost = rounds * ((K / 32 + ks - 1) / ks) * tile_chunk_cycles(4, nt);
      const long long stream = (long long)units * (silu ? 2 : 1) * K * 32 / 2000;
      if (cost < stream) cost = stream;
      cost += rounds * 6000;
      if (best < 0 || cost < best) {
        best = cost;
        best_nt = (unsigned)nt;
      }
    }
    const int least = b == 1 ? 3 : (b <= 3 ? 2 : 1);
    if (ks > 1 && K / 64 < least * ks) best_nt = 0;
    p.nt |= best_nt << (8 * (b - 1));
  }
  return p;
}

}  // namespace sfg

// ---------------------------------------------------------------------------
// Prefix attention (sf_attn.hip)
// ---------------------------------------------------------------------------
namespace sfa {

constexpr int kHD = 128;
constexpr int kQT = 128;       // queries per work item: 4 query groups of 32
constexpr int kChunk = 64;     // prefix keys per chunk (one LDS ring stage)
constexpr int kMaxChunks = 512;   // prefix <= 32768 keys
constexpr int kMaxRanges = 64;    // prefix partials per query at most
#ifndef SFA_ITEMS_TARGET
#define SFA_ITEMS_TARGET 256
#endif
constexpr int kItemsTarget = SFA_ITEMS_TARGET;

// LDS layout of a staged chunk: key rows of 256 bytes (16 units of 16 bytes =
// 8 dims each), K rows then V rows.  Unit u of key row r sits at unit
//  k_unit(r, u) = u ^ (r & 15)      in K: the 16 consecutive rows one MFMA
//                                   operand read takes at one unit hit 16
//                                   distinct units;
//  v_unit(r, u) = u ^ 2 * (r & 7)   in V: a transposing read takes 16
//                                   consecutive rows x one aligned unit pair;
//                                   rows 0-7 land on 8 distinct pairs, rows 8-15
//                                   on the same 8 (the read's second pass).
// Both are involutions, so the copy that fills physical unit p of row r reads
// logical unit k_unit(r, p) / v_unit(r, p).
SF_IDX int k_unit(int r, int u) { return u ^ (r & 15); }
SF_IDX int v_unit(int r, int u) { return u ^ (2 * (r & 7)); }
constexpr int kRowBytes = kHD * 2;               // one key row in LDS
constexpr int kHalfBytes = kChunk * kRowBytes;   // the K (or V) rows of a chunk

// Operand reads of a staged chunk, byte offsets from the chunk's K rows:
// * K fragment of MFMA A = K (16 keys of tile 0 x 32 dims ds*32..): lane l reads
//   key row l%16, logical unit ds*4 + l/16 (16 bytes); tile t adds 16 rows.
SF_IDX int k_frag_off(int lane, int ds) {
  const int row = lane & 15;
  return row * kRowBytes + k_unit(row, ds * 4 + (lane >> 4)) * 16;
}
// * V^T fragment of MFMA A = V^T (16 dims dt*16.. x 32 keys) by two transposing
//   reads (keys 4g..4g+3 of tiles 0 and 1, g = l/16): lane L of group g points at
//   row 4g + L/4, dims dt*16 + 4(L%4) .. +4 (8 bytes); tile 1 adds 16 rows.
SF_IDX int v_tr_off(int lane, int dt) {
  const int L = lane & 15;
  const int row = 4 * (lane >> 4) + (L >> 2);
  const int col = dt * 16 + 4 * (L & 3);  // first dim
  return kHalfBytes + row * kRowBytes + v_unit(row, col >> 3) * 16 + (col & 7) * 2;
}

// Chunks per work item: enough that the items fill about one round of the
// resident grid (longer ranges write fewer partials) and no query has more
// than kMaxRanges partials.  A pure function of device-side sizes, evaluated
// identically by the prefix and merge kernels.
SF_IDX int prefix_cpi(int nch, int n_qt, int Hkv) {
  const long long work = (long long)nch * n_qt * Hkv;
  int c = (int)((work + kItemsTarget - 1) / kItemsTarget);
  c = sf_imax(c, (nch + kMaxRanges - 1) / kMaxRanges);
  return sf_imax(1, sf_imin(c, nch));
}

// 16-key group j (0..3) of chunk ci starts at key chunk_group_g0 (groups past
// the prefix end are clamped to the last group holding keys, last_group_g0(P));
// row kr of the group holds key g0 + group_key(kr, g0, P) (keys past the end
// clamped to the last key).  With a page size that is a multiple of 16 a group
// never straddles pages.
SF_IDX int last_group_g0(int P) { return (P - 1) & ~15; }
SF_IDX int chunk_group_g0(int ci, int j, int last_g0) {
  return sf_imin(ci * kChunk + 16 * j, last_g0);
}
SF_IDX int group_key(int kr, int g0, int P) { return sf_imin(kr, P - 1 - g0); }

// Persistent prefix grid (a multiple of 8 workgroups; workgroup b runs on XCD
// b % 8): XCD x walks items [xcd_begin(items, x), xcd_begin(items, x + 1)).
SF_IDX int xcd_begin(int items, int xcd) { return (int)(((long long)items * xcd) >> 3); }

// Item it of the prefix pass: query tile qt, chunk range r, kv head h (the
// query tiles of one (range, head) are consecutive: one XCD, one L2).
struct AttnItem {
  int qt, r, h;
};
SF_IDX AttnItem attn_item(int it, int n_qt, int nr) {
  const int qt = it % n_qt;
  const int rest = it / n_qt;
  return AttnItem{qt, rest % nr, rest / nr};
}

// The prefix pass's decomposition for nq active queries per kv head and a prefix
// of P keys: n_qt query tiles, nch chunks, cpi chunks per range, nr ranges
// (= partials per query); items = n_qt · nr · Hkv ...
struct PrefixGrid {
  int n_qt, nch, cpi, nr;
};
SF_IDX PrefixGrid prefix_grid(int P, int nq, int Hkv) {
  const int n_qt = (nq + kQT - 1) / kQT;
  const int nch = (P + kChunk - 1) / kChunk;
  const int cpi = prefix_cpi(nch, n_qt, Hkv);
  return PrefixGrid{n_qt, nch, cpi, (nch + cpi - 1) / cpi};
}
// ... and the partials per query as the merge kernel derives them from its
// query count nq = rows · G.
SF_IDX int merge_ranges(int P, int nq, int Hkv) {
  return P > 0 ? prefix_grid(P, nq, Hkv).nr : 0;
}

inline int nchunks_for(int P) { return (P + kChunk - 1) / kChunk; }
// Range slots the workspace holds per (kv head, query) for a prefix capacity P.
inline int ranges_cap(int P) { return nchunks_for(P) < kMaxRanges ? nchunks_for(P) : kMaxRanges; }

// Partial slot of query qi of range r, kv head h: the workspace holds
// [Hkv][nr_cap][qmax] slots of kHD fp32 (acc), then the same count of (m, l).
SF_IDX size_t attn_slot(int h, int r, int qi, int nr_cap, int qmax) {
  return ((size_t)h * nr_cap + r) * qmax + qi;
}

// Persistent prefix grid for a capacity of qmax queries per kv head and a prefix
// capacity of nch chunks: enough workgroups for every item, at most one per CU
// (256 CUs), a multiple of 8.
inline int prefix_launch_grid(int qmax, int nch, int Hkv) {
  const int nr = nch < kMaxRanges ? nch : kMaxRanges;
  const long long items_cap = (long long)((qmax + kQT - 1) / kQT) * nr * Hkv;
  const long long g = ((items_cap + 7) / 8) * 8;
  return g < 256 ? (int)g : 256;
}

}  // namespace sfa

// ---------------------------------------------------------------------------
// Greedy statistics (sf_logits.hip): the slices of a logits row
// ---------------------------------------------------------------------------
namespace sfl {

constexpr int kMaxSlices = 32;          // slices per row: one wave merges their lists
constexpr int kMaxSliceVectors = 8191;  // 8-token vectors per slice: <= 65528 tokens,
                                        // so a slice's 16-bit counts and places fit
constexpr int kMaxVocab = kMaxSlices * kMaxSliceVectors * 8;   // 2,096,896 tokens

// Slices per row of V tokens (V % 8 == 0) for M rows: about 256 workgroups in
// all, at most kMaxSlices, and enough that no slice holds more than
// kMaxSliceVectors vectors (V <= kMaxVocab).
inline int slices_for(int M, int V) {
  const int nvec = V / 8;
  const int need = (nvec + kMaxSliceVectors - 1) / kMaxSliceVectors;
  return sf_imax(need, sf_imax(1, sf_imin(kMaxSlices, 256 / M)));
}
// Slice s of S holds the vectors [slice_begin(s), slice_begin(s + 1)) of nvec.
SF_IDX int slice_begin(int s, int nvec, int S) { return (int)((long long)nvec * s / S); }

}  // namespace sfl
