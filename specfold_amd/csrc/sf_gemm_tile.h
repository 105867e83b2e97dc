// Tile GEMM: the same products as the weight-streaming core (sf_gemm_core.h) for
// MORE rows than one of its passes holds.  Included by sf_gemm_core.h (after
// sf_common.h and sf_index.h).
//
// What bounds it: from ~130 rows on, a weight byte feeds enough rows that the
// matrix cores, the LDS operand reads and the weight stream cost about the same,
// so all rows have to share one pass over the weights (the streaming core would
// stream them once per 128 rows).  A workgroup of 8 waves computes 64·NMT rows x
// 32·NT columns: 4 row groups of NMT 16-row tiles x 2 column halves of NT 16-column
// tiles, so an operand byte read from LDS feeds NMT or NT MFMAs (at NMT = 4, NT = 8
// per 32-wide K chunk: 96 KB of LDS reads, 32 KB of copies and 32 MFMAs per wave,
// ~1024 cycles each).  Operands go to two LDS rings by direct copies: the A rows 64 K
// at a time, so that a copy takes whole cache lines (see a2_copy_unit), the weights a
// 32-K chunk at a time.  One barrier per chunk; fragments are read a few MFMAs ahead
// of their use, across the chunk boundary too, and the copies are spread between the
// MFMAs.  NT, the K ranges and the row blocks are chosen per shape by TilePlans
// (sf_index.h).  Measured: see the entry points that dispatch to it.
#pragma once

#include <type_traits>

namespace sfg {

// At most N of this wave's vector-memory loads in flight, then the workgroup barrier.
// Its LDS reads stay in flight (sf_wait_vm_barrier would wait for them).
template <int N>
SF_DEV void tile_barrier() {
#if defined(__HIPCC__)
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
#else
  sf_wait_vm_barrier<N>();
#endif
}
// Fragments [I, E) of f, STEP bytes apart from LDS byte address a (that of fragment
// 0), without waiting.
template <int STEP, int I, int E, int N>
SF_DEV void tile_reads(sf_u32x4 (&f)[N], sf_lds_off a) {
  if constexpr (I < E) {
    f[I] = sf_lds_read16<I * STEP>(a);
    tile_reads<STEP, I + 1, E>(f, a);
  }
}
// A fragment becomes usable: at most LATER younger LDS reads in flight.
template <int LATER>
SF_DEV void tile_use(sf_u32x4& f) {
  sf_u32x4(&one)[1] = reinterpret_cast<sf_u32x4(&)[1]>(f);
  sf_lds_reads_done_but<LATER>(one);
}
// f(integral_constant I) .. f(E - 1)
template <int I, int E, class F>
SF_DEV void tile_for(const F& f) {
  if constexpr (I < E) {
    f(std::integral_constant<int, I>{});
    tile_for<I + 1, E>(f);
  }
}

// The items of one launch, walked by every workgroup: nb row blocks x T column
// tiles x ks K ranges, row blocks fastest (they share the weight tile), and a
// contiguous eighth of the list per XCD (workgroup g runs on XCD g % 8), so what
// neighbours share is in that XCD's L2.  SILU: a tile is NT gate and the same NT
// up units of 16 columns (W0, W1; column half 0 and 1).
// in_row(r): input row of output row r < M; store(m, s, unit, cg, acc, rgrp...) is
// called per item with the accumulators.
struct TileGemm {
  const uint16_t* A;
  int lda;
  const uint16_t* W0;
  const uint16_t* W1;
  int K;
  int units;   // 16-column units of the output (SILU: of the gate)
};

template <bool SILU, int NMT, int NT, class In, class Store>
SF_DEV void tile_items(const TileGemm& g, int M, int n_ranges, sf_u32x4* ring, const In& in_row,
                       const Store& store) {
  const int ks = SILU ? 1 : n_ranges;
  using Sh = TileShape<NMT, NT>;
  using St = TileSteps<NMT, NT>;
  constexpr int RA = Sh::kRA, RW = Sh::kRW, CW = Sh::kCW;
  constexpr int D = St::kD;
  constexpr int kPer = SILU ? NT : 2 * NT;   // units per tile
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int rgrp = wv & 3;
  const int cg = wv >> 2;
  const int nb = (M + Sh::kRB - 1) / Sh::kRB;
  const int T = (g.units + kPer - 1) / kPer;
  const int items = nb * T * ks;
  const int stages = g.K / 64;
  const int G = gridDim.x;
  const int nx = (G & 7) ? 1 : 8;
  const int xcd = (int)blockIdx.x % nx;
  const int it_end = (int)((long long)items * (xcd + 1) / nx);
  const bool full = Sh::kRem == 0 || wv < Sh::kRem;   // this wave has all CW weight copies
  for (int it = (int)((long long)items * xcd / nx) + (int)blockIdx.x / nx; it < it_end;
       it += G / nx) {
    const int mb = it % nb;
    const int q = it / nb;
    const int t = q % T;
    const int s = q / T;
    const int m0 = mb * Sh::kRB;
    const int mrows = sf_imin(Sh::kRB, M - m0);
    const int sa = (int)((long long)stages * s / ks);
    const int nst = (int)((long long)stages * (s + 1) / ks) - sa;
    const int nch = 2 * nst;
    const int u0 = t * kPer;

    // this wave's copies.  A block b = wv + 8j of a stage: rows 8b .. +8 (rows past the
    // end repeat the last); weight block w = wv + 8j of a chunk: tile w.  A uniform
    // base advancing per stage / chunk plus this lane's 32-bit offset (tile_reach).
    const char* abase = reinterpret_cast<const char*>(g.A) + (size_t)sa * 128;
    uint32_t aoff[NMT];
#pragma unroll
    for (int j = 0; j < NMT; ++j) {
      const int r = in_row(m0 + sf_imin((wv + 8 * j) * 8 + (lane >> 3), mrows - 1));
      aoff[j] = (uint32_t)r * (uint32_t)g.lda * 2u + (uint32_t)a2_copy_unit(lane) * 16u;
    }
    const char* wbase[CW];
#pragma unroll
    for (int j = 0; j < CW; ++j) {
      const int w = sf_imin(wv + 8 * j, Sh::kNW - 1);
      const bool second = SILU && w >= NT;
      const int unit = sf_imin(u0 + (second ? w - NT : w), g.units - 1);
      wbase[j] = reinterpret_cast<const char*>(second ? g.W1 : g.W0) +
                 ((size_t)unit * stages + sa) * 2048;
    }
    const uint32_t woff = (uint32_t)lane * 16u;
    sf_u32x4* const aring = ring + wv * 64;
    sf_u32x4* const wring = ring + RA * Sh::kAW + wv * 64;
    auto copy_a = [&](int slot, int j) {
      sf_lds_dma16(abase + aoff[j], aring + slot * Sh::kAW + j * 512);
      if (j == NMT - 1) abase += 128;
    };
    auto copy_w = [&](int slot, int j) {
      if (j < CW - 1 || full) {   // wave-uniform
        sf_lds_dma16(wbase[j] + woff, wring + slot * Sh::kWW + j * 512);
        wbase[j] += 1024;
      }
    };
    // the prologue: the copies of the windows below 0, in window order
    constexpr int kFirst = 1 - 2 * RA < 1 - RW ? 1 - 2 * RA : 1 - RW;
    tile_for<0, -kFirst>([&](auto vc) {
      constexpr int v = decltype(vc)::value + kFirst;
      constexpr int q = (v - 1) / 2 + RA;   // (v odd: exact)
      if constexpr ((v & 1) != 0 && q >= 0) {
        if (q < nst) tile_for<0, NMT>([&](auto j) { copy_a(q, j); });
      }
      if constexpr (v - 1 + RW >= 0) {
        if (v - 1 + RW < nch) tile_for<0, CW>([&](auto j) { copy_w(v - 1 + RW, j); });
      }
    });

    sf_f32x4 acc[NMT][NT];
#pragma unroll
    for (int i = 0; i < NMT; ++i)
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[i][tt] = sf_f32x4{0.f, 0.f, 0.f, 0.f};

    // this lane's fragments: A tile rgrp*NMT + i (chunk k of its stage), weight tile
    // cg*NT + tt
    const sf_lds_off lds = sf_lds_addr(ring);
    sf_lds_off a_off[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      a_off[k] = lds + (sf_lds_off)(rgrp * NMT * 128 + a2_read_word(lane, k)) * 16;
    const sf_lds_off w_off =
        lds + (sf_lds_off)(RA * Sh::kAW + cg * NT * 64 + lane) * 16;
    sf_u32x4 fa[2][NMT], fw[NT];
    // the reads that open a chunk (A fragments at ao, weights at wo): weight fragment j
    // and the A fragments in front of it
    auto open_reads = [&](auto jc, sf_lds_off ao, sf_lds_off wo, sf_u32x4 (&fn)[NMT]) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j == 0) tile_reads<2048, 0, St::kNA0>(fn, ao);
      if constexpr (j == 1) tile_reads<2048, St::kNA0, NMT>(fn, ao);
      tile_reads<1024, j, j + 1>(fw, wo);
    };
    if (nch >= Sh::kTail) {
      if (full)
        tile_barrier<Sh::in_flight_first(CW)>();
      else
        tile_barrier<Sh::in_flight_first(CW - 1)>();
    } else {
      tile_barrier<0>();
    }
    tile_for<0, D>([&](auto j) { open_reads(j, a_off[0], w_off, fa[0]); });
    int as = 0, ws = 0;              // slots of the stage and the chunk computed
    int fill_a = 0, fill_w = 0;      // slots the current window's copies go to,
    bool fa_on = false, fw_on = false;   // if it has any
    // chunk c = 2p + k of the item
    auto chunk = [&](int c, auto kc) {
      constexpr int k = decltype(kc)::value;
      const sf_lds_off wo = w_off + (sf_lds_off)(ws * Sh::kWW) * 16;
      const int wn = ws + 1 == RW ? 0 : ws + 1;
      const sf_lds_off wno = w_off + (sf_lds_off)(wn * Sh::kWW) * 16;
      const int an = k == 0 ? as : (as + 1 == RA ? 0 : as + 1);
      const sf_lds_off ano = a_off[1 - k] + (sf_lds_off)(an * Sh::kAW) * 16;
      tile_for<0, NT>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        if constexpr (t < NT - D) {
          tile_reads<1024, t + D, t + D + 1>(fw, wo);
        } else {
          if constexpr (t == NT - D) {
            // chunk c + 1 has landed in every wave's share, and every wave is past its
            // last use of chunk c - 1's weights (and, k = 1, has read the last of this
            // stage's A): their slots are refilled
            if (c + Sh::kTail <= nch) {
              if (full)
                tile_barrier<Sh::in_flight(k, CW)>();
              else
                tile_barrier<Sh::in_flight(k, CW - 1)>();
            } else {
              tile_barrier<0>();
            }
            fill_w = ws == 0 ? RW - 1 : ws - 1;
            fw_on = c - 1 + RW < nch;
            if constexpr (k == 1) {
              fill_a = as;
              fa_on = (c - 1) / 2 + RA < nst;
            }
          }
          // (past the last chunk: stale bytes, read and dropped)
          open_reads(std::integral_constant<int, t - (NT - D)>{}, ano, wno, fa[1 - k]);
        }
        tile_use<St::later(t)>(fw[t]);
        if constexpr (t == 0) {
#pragma unroll
          for (int i = 0; i < NMT; ++i) tile_use<St::later(t)>(fa[k][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NMT; ++i)
          acc[i][t] = sf_mfma16x16x32(sf_as_bf16x8(fw[t]), sf_as_bf16x8(fa[k][i]), acc[i][t]);
        __builtin_amdgcn_sched_barrier(0);
        // the window's copies a few at a time between the MFMAs (A first)
        constexpr bool odd = t >= NT - D ? k == 1 : k == 0;   // the window's parity
        constexpr int n = CW + (odd ? NMT : 0);
        tile_for<0, n>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if constexpr ((NT - D + i * NT / n) % NT == t) {
            if constexpr (odd && i < NMT) {
              if (fa_on) copy_a(fill_a, i);
            } else {
              if (fw_on) copy_w(fill_w, i - (odd ? NMT : 0));
            }
          }
        });
      });
      ws = wn;
      as = an;
    };
#pragma unroll 1
    for (int c = 0; c < nch; c += 2) {
      chunk(c, std::integral_constant<int, 0>{});
      chunk(c + 1, std::integral_constant<int, 1>{});
    }
    // the reads past the last chunk land before their registers are reused, and every
    // wave is done with the ring before the epilogue or the next item writes it
    sf_lds_reads_done(fa[0]);
    sf_lds_reads_done(fa[1]);
    sf_lds_reads_done(fw);
    sf_wait_vm_barrier<0>();

    // lane: row m0 + (rgrp*NMT + i)*16 + lane%16, columns 16*unit + 4*(lane/16) .. +4 of
    // unit u0 + cg*NT + tt (SILU: u0 + tt, the gate's in half 0 and the up's in half 1)
    store(m0, mrows, s, u0, rgrp, cg, acc);
    sf_wait_vm_barrier<0>();
  }
}

// The stores below are plain, not the hand-off stores of the few-row kernels: a store
// instruction covers 64 (fp32) or 32 bytes (bf16) of a row, which the non-temporal hint
// sends on as they are, part of a line each, while plain ones meet in L2 and leave as
// whole lines.  From 129 rows on that outweighs the dirty lines the next kernel's
// weight stream finds (non-temporal -> plain, us: QKV + o_proj of 144 of 640 rows
// at 4096 78.5 -> 76.8; MLP of 256 rows at 5120 x 17408 187.5 -> 185.0; with the head's,
// prefill of 2048 tokens, 4 layers at 7B widths 7408 -> 6867).

// fp32 sums of K range s to part[(s * mcap + m) * N + c]
struct TilePartStore {
  float* part;
  int mcap, N;
  template <int NMT, int NT>
  SF_DEV void operator()(int m0, int mrows, int s, int u0, int rgrp, int cg,
                         const sf_f32x4 (&acc)[NMT][NT]) const {
    int lane = threadIdx.x & 63;
    sf_pin(lane);   // nothing of the epilogue is hoisted over the item's main loop
#pragma unroll
    for (int i = 0; i < NMT; ++i) {
      const int m = (rgrp * NMT + i) * 16 + (lane & 15);
      if (m < mrows) {
        float* p = part + ((size_t)s * mcap + m0 + m) * N + (lane >> 4) * 4;
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
          const int unit = u0 + cg * NT + tt;
          if (unit * 16 < N)
            *reinterpret_cast<sf_f32x4*>(p + unit * 16) = acc[i][tt];
        }
      }
    }
  }
};

// act = bf16(bf16(silu(bf16 gate)) * bf16 up): the waves of a row group hold the gate
// (half 0) and the up sums (half 1) of the same outputs; each takes half of the m
// tiles and gets the other operand through LDS (the ring's memory).
struct TileSiluStore {
  sf_u32x4* ring;
  uint16_t* out;
  int ldo, units;
  template <int NMT, int NT>
  SF_DEV void operator()(int m0, int mrows, int, int u0, int rgrp, int cg,
                         const sf_f32x4 (&acc)[NMT][NT]) const {
    int lane = threadIdx.x & 63;
    sf_pin(lane);   // nothing of the epilogue is hoisted over the item's main loop
    constexpr int NH = (NMT + 1) / 2;   // m tiles of half 0
    static_assert(8 * NH * NT * 64 <= TileShape<NMT, NT>::kWords,
                  "the exchange fits the ring");
    sf_f32x4* xch = reinterpret_cast<sf_f32x4*>(ring) + lane;
    sf_f32x4* mine = xch + (rgrp * 2 + cg) * NH * NT * 64;
    const sf_f32x4* theirs = xch + (rgrp * 2 + 1 - cg) * NH * NT * 64;
#pragma unroll
    for (int i = 0; i < NMT; ++i)
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        if (i < NH) {
          if (cg == 1) mine[(i * NT + tt) * 64] = acc[i][tt];
        } else {
          if (cg == 0) mine[((i - NH) * NT + tt) * 64] = acc[i][tt];
        }
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NMT; ++i) {
      if ((i < NH) != (cg == 0)) continue;   // wave-uniform
      const int m = (rgrp * NMT + i) * 16 + (lane & 15);
      if (m >= mrows) continue;
      uint16_t* p = out + (size_t)(m0 + m) * ldo + (lane >> 4) * 4;
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        if (u0 + tt >= units) continue;
        const sf_f32x4 o = theirs[((i < NH ? i : i - NH) * NT + tt) * 64];
        float r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float gt = sf_rbf(i < NH ? acc[i][tt][k] : o[k]);
          r[k] = sf_rbf(gt / (1.0f + expf(-gt))) * sf_rbf(i < NH ? o[k] : acc[i][tt][k]);
        }
        sf_u32x2 v;
        v[0] = sf_pack2(r[0], r[1]);
        v[1] = sf_pack2(r[2], r[3]);
        *reinterpret_cast<sf_u32x2*>(p + (u0 + tt) * 16) = v;
      }
    }
  }
};

// tile_items at the plan's shape for M rows.
template <bool SILU, int NMT, class In, class Store>
SF_DEV void tile_gemm_nt(const TileGemm& g, int M, int nt, int ks, sf_u32x4* ring, const In& in,
                         const Store& st) {
  if constexpr (SILU) {
    if (nt == 3) return tile_items<SILU, NMT, 3>(g, M, ks, ring, in, st);
    if (nt == 5) return tile_items<SILU, NMT, 5>(g, M, ks, ring, in, st);
    if (nt == 6) return tile_items<SILU, NMT, 6>(g, M, ks, ring, in, st);
    if (nt == 7) return tile_items<SILU, NMT, 7>(g, M, ks, ring, in, st);
  } else {
    if (nt == 2) return tile_items<SILU, NMT, 2>(g, M, ks, ring, in, st);
  }
  if (nt == 4) return tile_items<SILU, NMT, 4>(g, M, ks, ring, in, st);
  return tile_items<SILU, NMT, 8>(g, M, ks, ring, in, st);
}
template <bool SILU, class In, class Store>
SF_DEV void tile_gemm(const TileGemm& g, int M, const TilePlans& tp, sf_u32x4* ring, const In& in,
                      const Store& st) {
  const int nt = tile_nt(M, tp), ks = tp.ks;
  if (tile_nmt(M) == 3)
    tile_gemm_nt<SILU, 3>(g, M, nt, ks, ring, in, st);
  else
    tile_gemm_nt<SILU, 4>(g, M, nt, ks, ring, in, st);
}

}  // namespace sfg
