// Reaction rates of 64 cells per block, with the mechanism walked by whole wavefronts (and the row sums
// that setTemperature uses too).
//
// A block of 64 G threads (G wavefronts) owns 64 cells and sees them in two layouts:
//  * rows: a cell belongs to G neighbouring lanes of one wavefront (64 / G cells per wavefront),
//    lane j holding component rows 2 j and 2 j + 1 of every 2 G-row block. The canonical pairwise
//    sum (bdf_kernel.h, gpsum) then starts with an add inside the lane and goes on with DPP adds
//    inside the quad: no LDS and no barrier for any sum, norm or maximum over a cell's components;
//  * cells: lane = cell, every wavefront evaluating its share of the reactions (then of the
//    species) for all 64 cells. The reaction is the same for all lanes, so its record comes
//    through scalar loads, its kind and stoichiometry are scalar branches (no lane of a falloff
//    or third-body reaction waits for another kind), every lane does useful work, and the
//    concentrations are read at one stride (conflict-free) from LDS.
// What bounds it is the latency of each reaction's chain at the three wavefronts per SIMD that 53 KB of LDS
// per block leave (drm19, 138 VGPRs; one block per CU at 53 species): on 64^3 drm19 cells the SIMDs issue
// VALU instructions in 52 % of the cycles, 55 % of them FP64 arithmetic. Measured on reactionRateRhoY
// (rates_block_kernel) against the group kernel's reaction-per-lane form (a record read per lane
// from LDS, drm19's 84 reactions in three passes of 32 lanes with mixed kinds): 64^3 drm19 cells 471
// -> 222 us per call, 22533 dodecane_lu cells 186 -> 126 us, the same bits.
//
// Sums run in the same order as everywhere else: a species' incidence list in blocks of
// PR_GATHER_BLOCK entries, block sums added in list order. Rates pass through LDS in chunks of
// consecutive mechanism reactions, a block split by a chunk border keeping its partial sum in
// registers, so chunking does not show in the results.
#ifndef PR_BLOCK_RATES_H
#define PR_BLOCK_RATES_H
#include "react_kernel.h"

namespace prk {

// Constant address space: loads at wavefront-uniform addresses become scalar loads whatever
// stores the kernel does (the tables are never written while a kernel runs).
#define PR_CONST_AS __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ const PR_CONST_AS T* const_as(const T* p) {
  return (const PR_CONST_AS T*)p;
}

// One piece of a species' incidence list: up to PR_GATHER_BLOCK entries of one gather block inside
// one chunk. first / last: the piece opens / closes its gather block; lead: the block is the
// species' first.
struct GatherPiece {
  double nu[PR_GATHER_BLOCK];
  int32_t qoff[PR_GATHER_BLOCK];  // double offset of the entry's rate row inside the chunk (slot * 64)
  int32_t ne, first, last, lead;
};

// Host-built tables of the cells layout (device pointers into one allocation).
struct BlockTabs {
  const RxRec* rx;          // records in evaluation order: chunk by chunk, wavefront by wavefront
  const int32_t* rx_range;  // [nchunk * waves + 1] first record of each (chunk, wavefront)
  const GatherPiece* piece;
  const int32_t* piece_range;  // [nchunk * N + 1] first piece of each (chunk, species)
};

// Sizes of the two layouts for a mechanism.
template <int N, int R, int G>
struct BlockCell {
  static constexpr int n = N + 1;
  static constexpr int CELLS = 64;
  static constexpr int B = 2 * G;                // rows per block of rows
  static constexpr int NB = (n + B - 1) / B;
  static constexpr int RPL = 2 * NB;             // rows per lane
  static constexpr int NP = NB * B;              // rows, padded
  static constexpr int SPW = (N + G - 1) / G;    // species per wavefront in the gather
  // Rates per chunk: all of them when they fit beside the concentrations in the LDS two blocks
  // share (n <= 16) or in half of it (n <= 32), a third of them above
  static constexpr int NCHUNK = n <= 16 ? 1 : (n <= 32 ? 2 : 3);
  static constexpr int QROWS = (R + NCHUNK - 1) / NCHUNK;
  static __device__ __forceinline__ int row(int lane, int s) { return B * (s >> 1) + 2 * lane + (s & 1); }
};

// Canonical pairwise sum over components 0 .. CNT - 1 held in the rows layout: every lane of the
// cell's group gets it. The same tree as gpsum: pairs, then lane ^ 1, lane ^ 2 (and lane ^ 4) by
// DPP form a block of 2 G rows; the blocks' sums are combined pairwise up to 64 slots.
template <int N, int R, int G, int CNT>
__device__ __forceinline__ double rsum(int lane, const double (&a)[BlockCell<N, R, G>::RPL]) {
  using C = BlockCell<N, R, G>;
  static_assert(G == 4 || G == 8, "groups of 4 or 8 lanes");
  constexpr int T = 64 / C::B;
  double t[T];
#pragma unroll
  for (int b = 0; b < T; ++b) {
    if (b >= C::NB || C::B * b >= CNT) {  // an all-zero block sums to +0.0
      t[b] = 0.0;
      continue;
    }
    double a0 = a[2 * b], a1 = a[2 * b + 1];
    if (C::B * (b + 1) > CNT) {
      a0 = C::row(lane, 2 * b) < CNT ? a0 : 0.0;
      a1 = C::row(lane, 2 * b + 1) < CNT ? a1 : 0.0;
    }
    double v = a0 + a1;
    v = v + dpp_d<0xB1>(v);
    v = v + dpp_d<0x4E>(v);
    if (G == 8) v = v + dpp_d<0x141>(v);  // quad-uniform values: the mirrored quad is lane ^ 4
    t[b] = v;
  }
#pragma unroll
  for (int w = 1; w < T; w <<= 1)
#pragma unroll
    for (int j = 0; j < T; j += 2 * w) t[j] = t[j] + t[j + w];
  return t[0];
}

// LDS of the rates: concentrations and g / RT as [species][64 cells] (the gathered production
// rates later take the concentrations' place), one chunk of rates as [reaction][64], and per-cell
// T, ln T, 1 / T, ln(R T / P_atm), sum C.
template <int N, int R, int G>
struct RateLds {
  using C = BlockCell<N, R, G>;
  static constexpr int cg_doubles = 2 * N * C::CELLS;
  static constexpr int q_doubles = C::QROWS * C::CELLS;
  static constexpr int sc_doubles = 5 * C::CELLS;
  double* cg;
  double* q;
  double* sc;
  const SpRec* sp;
};

// Temperature of each cell's group from (h, Y), as hy2t; and its species thermodynamics.
template <int N, int R, int G>
__device__ __forceinline__ double rows_hy2t(const SpRec* sp, int lane, const double (&Y)[BlockCell<N, R, G>::RPL],
                                            double h, double T) {
  using C = BlockCell<N, R, G>;
  for (int it = 0; it < 20; ++it) {
    const double invT = 1.0 / T;
    double ph[C::RPL], pc[C::RPL];
#pragma unroll
    for (int s = 0; s < C::RPL; ++s) {
      const int i = C::row(lane, s);
      ph[s] = 0.0;
      pc[s] = 0.0;
      if (i < N) {
        double cpR, hRT;
        nasa_hcp(sp[i], T, invT, cpR, hRT);
        const double RW = sp[i].RW;
        ph[s] = ((Y[s] * hRT) * RW) * T;
        pc[s] = (Y[s] * cpR) * RW;
      }
    }
    const double hm = rsum<N, R, G, N>(lane, ph), cpm = rsum<N, R, G, N>(lane, pc);
    const double dT = (h - hm) / cpm;
    T = T + dT;
    if (fabs(dT) <= 1e-10 * T) break;
  }
  return T;
}

// The first half of net_rates in the rows layout: what the cells layout reads goes to LDS (cell: the
// cell's column).
template <int N, int R, int G>
__device__ __forceinline__ void rows_thermo(const RateLds<N, R, G>& L, int lane, int cell, double T,
                                            const double (&cc)[BlockCell<N, R, G>::RPL]) {
  using C = BlockCell<N, R, G>;
  const double lnT = pr_log(T), invT = 1.0 / T, lnRTP = pr_log((PR_RU * T) / PR_PATM);
#pragma unroll
  for (int s = 0; s < C::RPL; ++s) {
    const int i = C::row(lane, s);
    if (i < N) {
      double cpR, hRT, gRT, dcp;
      nasa_full(L.sp[i], T, invT, lnT, cpR, hRT, gRT, dcp);
      L.cg[i * C::CELLS + cell] = cc[s];
      L.cg[(N + i) * C::CELLS + cell] = gRT;
    }
  }
  const double Ctot = rsum<N, R, G, N>(lane, cc);
  if (lane == 0) {
    L.sc[cell] = T;
    L.sc[C::CELLS + cell] = lnT;
    L.sc[2 * C::CELLS + cell] = invT;
    L.sc[3 * C::CELLS + cell] = lnRTP;
    L.sc[4 * C::CELLS + cell] = Ctot;
  }
}

// A reaction's record in scalar registers: everything but the falloff parameters.
struct RxHead {
  double lnA, beta, Ta, effd;
  int info, reac, prod, eff, qoff;
  template <class Rx>
  __device__ __forceinline__ void load(const Rx& rx) {
    lnA = rx.lnA;
    beta = rx.beta;
    Ta = rx.Ta;
    effd = rx.effd;
    info = rx.info;
    reac = rx.reac;
    prod = rx.prod;
    eff = rx.eff;
    qoff = rx.qoff;
  }
};

// Rate of progress of one reaction, the same for every lane, at each lane's cell: rx_eval<false>'s
// fwd - rev with its operations in its order. h is the reaction's record, rx the falloff part of it
// (read only by falloff reactions); sC, sG: the cell's columns of LDS.
template <class Rx, class EffSp, class EffVal>
__device__ __forceinline__ double cell_rate(const ExpK& K, const RxHead& h, const Rx& rx, const double* sC,
                                            const double* sG, double Ctot, double T, double lnT, double invT,
                                            double lnRTP, const EffSp* effsp, const EffVal* effval) {
  const int type = h.info & 15, rev = (h.info >> 4) & 15, nre = (h.info >> 8) & 15, npr = (h.info >> 12) & 15;
  const int r0 = (h.reac & 0xFF) * 64, r1 = ((h.reac >> 8) & 0xFF) * 64, r2 = ((h.reac >> 16) & 0xFF) * 64;
  const int p0 = (h.prod & 0xFF) * 64, p1 = ((h.prod >> 8) & 0xFF) * 64, p2 = ((h.prod >> 16) & 0xFF) * 64;
  // two slots on each side are read unconditionally (an absent one holds species 0, not used)
  const double cr0 = sC[r0], cr1 = sC[r1], gr0 = sG[r0], gr1 = sG[r1];
  const double cp0 = sC[p0], cp1 = sC[p1], gp0 = sG[p0], gp1 = sG[p1];
  double M = 0.0;
  if (type != PR_RX_ELEM) {
    M = h.effd * Ctot;
    const int ee = (h.eff >> 16) & 0xFFFF;
#pragma unroll 1
    for (int e = h.eff & 0xFFFF; e < ee; e += 4) {  // in list order, four table reads issued together
      const int e1 = e + 1 < ee ? e + 1 : e, e2 = e + 2 < ee ? e + 2 : e, e3 = e + 3 < ee ? e + 3 : e;
      const double c0 = sC[effsp[e] * 64], c1 = sC[effsp[e1] * 64], c2 = sC[effsp[e2] * 64], c3 = sC[effsp[e3] * 64];
      const double v0 = effval[e], v1 = effval[e1], v2 = effval[e2], v3 = effval[e3];
      M = fma(v0, c0, M);
      if (e + 1 < ee) M = fma(v1, c1, M);
      if (e + 2 < ee) M = fma(v2, c2, M);
      if (e + 3 < ee) M = fma(v3, c3, M);
    }
  }
  double pr = cr0;
  if (nre > 1) pr *= cr1;
  if (nre > 2) pr *= sC[r2];
  const double ka = fma(-h.Ta, invT, fma(h.beta, lnT, h.lnA));
  double kinf, invKc = 0.0, pp = 0.0;
  if (rev) {
    double dG = gp0;
    if (npr > 1) dG += gp1;
    if (npr > 2) dG += sG[p2];
    dG -= gr0;
    if (nre > 1) dG -= gr1;
    if (nre > 2) dG -= sG[r2];
    pp = cp0;
    if (npr > 1) pp *= cp1;
    if (npr > 2) pp *= sC[p2];
    const double x[2] = {ka, fma((double)(npr - nre), lnRTP, dG)};
    double e[2];
    exp_n<2>(K, x, e);
    kinf = e[0];
    invKc = e[1];
  } else {
    // invKc = 0: the reverse rate is kf * 0 * pp, formed below as rx_eval forms it
    pp = cp0;
    if (npr > 1) pp *= cp1;
    if (npr > 2) pp *= sC[p2];
    const double x[1] = {ka};
    double e[1];
    exp_n<1>(K, x, e);
    kinf = e[0];
  }
  if (type <= PR_RX_THIRDBODY) {
    const double kr0 = kinf * invKc;
    const double fwd0 = kinf * pr, rev0 = kr0 * pp;
    return type == PR_RX_ELEM ? fwd0 - rev0 : M * fwd0 - M * rev0;
  }
  const double ta1 = rx.troe[1], ta2 = rx.troe[2], ta3 = rx.troe[3];
  const double k0a = fma(-rx.Ta0, invT, fma(rx.beta0, lnT, rx.lnA0));
  double k0, F = 1.0;
  if (type == PR_RX_TROE) {
    const double tr0 = rx.troe[0];
    double Fc;
    const int ntroe = (h.info >> 16) & 15;
    if (ntroe == 4) {
      const double x[4] = {k0a, -T / ta1, -T / ta2, -ta3 * invT};
      double e[4];
      exp_n<4>(K, x, e);
      k0 = e[0];
      Fc = (1.0 - tr0) * e[1] + tr0 * e[2];
      Fc += e[3];
    } else {
      const double x[3] = {k0a, -T / ta1, -T / ta2};
      double e[3];
      exp_n<3>(K, x, e);
      k0 = e[0];
      Fc = (1.0 - tr0) * e[1] + tr0 * e[2];
    }
    double Pr = (k0 * M) / kinf;
    if (Pr < 1e-300) Pr = 1e-300;
    if (Fc < 1e-300) Fc = 1e-300;
    const double logFc = pr_log10(Fc);
    const double x = pr_log10(Pr);
    const double c = -0.4 - 0.67 * logFc, nn = 0.75 - 1.27 * logFc;
    const double xc = x + c, D = nn - 0.14 * xc, f1 = xc / D;
    const double den = 1.0 + f1 * f1;
    const double xf[1] = {(logFc / den) * PRK_LN10};
    double ef[1];
    exp_n<1>(K, xf, ef);
    F = ef[0];
    const double kf = ((kinf * Pr) / (1.0 + Pr)) * F;
    return kf * pr - (kf * invKc) * pp;
  }
  {
    const double x[1] = {k0a};
    double e[1];
    exp_n<1>(K, x, e);
    k0 = e[0];
  }
  double Pr = (k0 * M) / kinf;
  if (Pr < 1e-300) Pr = 1e-300;
  const double kf = ((kinf * Pr) / (1.0 + Pr)) * F;
  return kf * pr - (kf * invKc) * pp;
}

// The cells layout: rates of progress chunk by chunk and the species' gathered sums, left as
// [species][64] in L.cg. Called by every thread of the block after rows_thermo; ends behind a
// barrier.
template <int N, int R, int G>
__device__ __forceinline__ void cells_rates(const RateLds<N, R, G>& L, const BlockTabs& tab, const int* effsp,
                                            const double* effval) {
  using C = BlockCell<N, R, G>;
  const int cell = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const auto* rxs = const_as(tab.rx);
  const auto* rng = const_as(tab.rx_range);
  const auto* pcs = const_as(tab.piece);
  const auto* prng = const_as(tab.piece_range);
  double p[C::SPW], a[C::SPW];
#pragma unroll
  for (int s = 0; s < C::SPW; ++s) p[s] = a[s] = 0.0;
  __syncthreads();
#pragma unroll 1
  for (int c = 0; c < C::NCHUNK; ++c) {
    int m = rng[c * G + wave];
    const int m1 = rng[c * G + wave + 1];
    if (m < m1) {
      const ExpK K = exp_constants();
      const double T = L.sc[cell], lnT = L.sc[C::CELLS + cell], invT = L.sc[2 * C::CELLS + cell],
                   lnRTP = L.sc[3 * C::CELLS + cell], Ctot = L.sc[4 * C::CELLS + cell];
      RxHead h;
      h.load(rxs[m]);
#pragma unroll 1
      for (; m < m1; ++m) {
        RxHead nx;  // the next record's scalar loads are in flight during this reaction
        nx.load(rxs[m + 1 < m1 ? m + 1 : m]);
        L.q[h.qoff + cell] = cell_rate(K, h, rxs[m], L.cg + cell, L.cg + N * C::CELLS + cell, Ctot, T, lnT, invT,
                                       lnRTP, const_as(effsp), const_as(effval));
        h = nx;
      }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < C::SPW; ++s) {
      const int k = wave + G * s;
      if (k < N) {
        const int e1 = prng[c * N + k + 1];
#pragma unroll 1
        for (int e = prng[c * N + k]; e < e1; ++e) {
          const auto& pc = pcs[e];
          double qv[PR_GATHER_BLOCK];
#pragma unroll
          for (int j = 0; j < PR_GATHER_BLOCK; ++j) qv[j] = L.q[pc.qoff[j] + cell];
          double v = pc.first ? 0.0 : p[s];
          const int ne = pc.ne;
#pragma unroll
          for (int j = 0; j < PR_GATHER_BLOCK; ++j)
            if (j < ne) v += pc.nu[j] * qv[j];
          p[s] = v;
          if (pc.last) a[s] = pc.lead ? v : a[s] + v;
        }
        if (c == C::NCHUNK - 1) L.cg[k * C::CELLS + cell] = a[s];
      }
    }
    __syncthreads();
  }
}

// The next (up to) 64 uncovered cells of a block's rounds in a box with a mask, their covered cells'
// rates set to zero on the way: the index of the group's cell, -1 past the last one. rd, cur, left: the
// round to look at next, the last one looked at and its cells still to do, the same in every
// wavefront (each looks at the 64 cells of a round). list: 64 ints of LDS, free again after the block's
// next barrier. Called by every thread, behind a barrier; ends behind one. more: whether any cell is left.
template <int N, int R, int G>
__device__ __forceinline__ long next_uncovered(const RateParams& P, long rounds, long& rd, long& cur,
                                               unsigned long long& left, int* list, bool& more) {
  constexpr int CELLS = BlockCell<N, R, G>::CELLS;
  const int wave = threadIdx.x / 64, l = threadIdx.x % 64, cell = threadIdx.x / G;
  int have = 0;
  while (have < CELLS) {
    if (left == 0) {
      if (rd >= rounds) break;
      cur = rd;
      rd += gridDim.x;
      const long c = cur * CELLS + l;
      const unsigned u = (unsigned)c;
      const int i = P.lo0 + (int)(u % (unsigned)P.nx);
      const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
      const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
      const bool covered = c < P.ncells && P.mask.p[(long)(i - P.mask.bx) + (long)(j - P.mask.by) * P.mask.js +
                                                    (long)(k - P.mask.bz) * P.mask.ks] == -1;
      if (covered) {
        const long offO = aoff(P.out, i, j, k);
        for (int ii = wave; ii < N; ii += G) P.out.p[offO + (long)ii * P.out.ns] = 0.0;
      }
      left = __ballot(c < P.ncells && !covered);
    }
    const int at = have + __popcll(left & ((1ull << l) - 1));
    const bool mine = (left >> l) & 1;
    if (mine && at < CELLS && wave == 0) list[at] = (int)(cur * CELLS + l);
    have += __popcll(left);
    left = __ballot(mine && at >= CELLS);
  }
  __syncthreads();
  more = have > 0;
  return cell < have ? list[cell] : -1;
}

// reactionRateRhoY over a box (see rate_kernel): 64 cells per block and pass, consecutive ones, or with
// MASKED the next uncovered ones, so that a mostly covered box costs what is left of it. Measured (us
// per call, 0 / 50 / 90 / 100 % of the cells in a covered slab), 64^3 drm19 cells: a group of lanes per
// cell 447 / 251 / 97 / 63, rates formed for covered cells too 221 / 205 / 196 / 192, now 223 / 135 / 65 /
// 34; 40^3 dodecane_lu 428 / 248 / 108 / 73, 212 / 198 / 191 / 183, 223 / 127 / 80 / 30. A kernel of its own:
// the list costs a box with nothing covered up to 10 % (48^3 LiDryer cells 50 -> 55 us).
template <int N, int R, int G, bool MASKED>
__global__ void __launch_bounds__(64 * G) rates_block_kernel(RateParams P, BlockTabs tab) {
  using C = BlockCell<N, R, G>;
  extern __shared__ __align__(16) unsigned char smem[];
  RateLds<N, R, G> L;
  L.cg = reinterpret_cast<double*>(smem);
  L.q = L.cg + RateLds<N, R, G>::cg_doubles;
  L.sc = L.q + RateLds<N, R, G>::q_doubles;
  L.sp = reinterpret_cast<const SpRec*>(L.sc + RateLds<N, R, G>::sc_doubles);
  const BlobLayout BL = blob_layout(N, R, P.neff, P.ninc);
  {
    const uint4* srcb = reinterpret_cast<const uint4*>(P.blob + BL.off_sp);
    uint4* dst = reinterpret_cast<uint4*>(L.sc + RateLds<N, R, G>::sc_doubles);
    for (int b = threadIdx.x; b < (int)(N * sizeof(SpRec)) / 16; b += blockDim.x) dst[b] = srcb[b];
  }
  __syncthreads();
  const int lane = threadIdx.x % G;
  const int cell = threadIdx.x / G;
  const long rounds = (P.ncells + C::CELLS - 1) / C::CELLS;
  long rd = blockIdx.x, cur = 0;
  unsigned long long left = 0;
  for (;;) {
    long c;
    if constexpr (MASKED) {
      bool more;
      c = next_uncovered<N, R, G>(P, rounds, rd, cur, left, reinterpret_cast<int*>(L.q), more);
      if (!more) break;
    } else {
      if (rd >= rounds) break;
      c = rd * C::CELLS + cell;
      rd += gridDim.x;
    }
    const bool active = MASKED ? c >= 0 : c < P.ncells;
    const unsigned u = (unsigned)(active ? c : P.ncells - 1);
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    if (active) {
      const long offY = aoff(P.rY, i, j, k);
      double ry[C::RPL], Y[C::RPL], cc[C::RPL];
#pragma unroll
      for (int s = 0; s < C::RPL; ++s) {
        const int ii = C::row(lane, s);
        ry[s] = ii < N ? P.rY.p[offY + (long)ii * P.rY.ns] : 0.0;
      }
      const double rH = P.rH.p[aoff(P.rH, i, j, k)], T0 = P.T.p[aoff(P.T, i, j, k)];
      const double rho = rsum<N, R, G, N>(lane, ry);
      const double rhoinv = 1.0 / rho;
#pragma unroll
      for (int s = 0; s < C::RPL; ++s) Y[s] = C::row(lane, s) < N ? ry[s] * rhoinv : 0.0;
      const double T = rows_hy2t<N, R, G>(L.sp, lane, Y, (rH * rhoinv) * 1.0e4, T0);
      const double rho_cgs = rho * 0.001;
#pragma unroll
      for (int s = 0; s < C::RPL; ++s) {
        const int ii = C::row(lane, s);
        cc[s] = ii < N ? (rho_cgs * Y[s]) * L.sp[ii].invW : 0.0;
      }
      rows_thermo<N, R, G>(L, lane, cell, T, cc);
    }
    cells_rates<N, R, G>(L, tab, reinterpret_cast<const int*>(P.blob + BL.off_effsp),
                         reinterpret_cast<const double*>(P.blob + BL.off_effval));
    if (active) {
      const long offO = aoff(P.out, i, j, k);
#pragma unroll
      for (int s = 0; s < C::RPL; ++s) {
        const int ii = C::row(lane, s);
        if (ii < N)
          P.out.p[offO + (long)ii * P.out.ns] = (L.cg[ii * C::CELLS + cell] * L.sp[ii].W) * 1000.0;
      }
    }
    __syncthreads();
  }
}

}  // namespace prk
#endif
