// Equation-of-state box kernels around the chemistry advance, MKS Array4 views (cells fastest, so
// every species row of the box is read and written coalesced; the species records are staged in
// LDS), one thread per cell except setTemperature (a quad or eight lanes per cell):
//  * setTemperature  (Source/PeleLMeX_Eos.cpp:218-240 -> getTfromHY, Source/PeleLMeX_K.H:700-723):
//    rhoinv = 1 / rho, Y = rhoY * rhoinv, h = rhoH * rhoinv * 1e4, T = HY2T(h, Y) from the stored
//    T - the reactor's own iteration and sums (hy2t), so the temperature is the one its
//    right-hand side computes;
//  * floorSpecies    (Source/PeleLMeX_Utils.cpp:649-690, fabMinMax Source/PeleLMeX_K.H:894-907):
//    rhoY_k = max(0, min(DBL_MAX, rhoY_k)) with std::min / std::max semantics, rho = sum_k rhoY_k
//    and h = TY2H(T, Y) = sum_k Y_k h_k(T) in species order, rhoH = h * 1e-4 * rho;
//  * getHeatRelease  (Source/PeleLMeX_Reactions.cpp:477-506, getHGivenT Source/PeleLMeX_K.H:598-615):
//    HR = 0 - sum_k (h_k(T) * 1e-4) * I_R,k in species order.
// h_k(T) = (h_k / RT) (R / W_k) T in erg / g, the reactor's species enthalpy. HBM-bound: a cell
// moves (N + 4), (2 N + 3) and (N + 2) doubles.
#pragma once

#include <cfloat>

#include "block_rates.h"

namespace prk {

enum { EOS_SET_T = 0, EOS_FLOOR = 1, EOS_HEAT_RELEASE = 2 };

struct EosParams {
  int lo0, lo1, lo2, nx, ny;
  long ncells;
  Arr rY, rho, rH, T, IR, HR;
  const unsigned char* blob;
  int blob_bytes, neff, ninc;
};

template <int N, int R, int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) eos_cell_kernel(EosParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  {
    // the species records only: the blob's first section
    const BlobLayout BL = blob_layout(N, R, P.neff, P.ninc);
    const uint4* srcb = reinterpret_cast<const uint4*>(P.blob + BL.off_sp);
    uint4* dst = reinterpret_cast<uint4*>(smem);
    for (int b = threadIdx.x; b < (int)(N * sizeof(SpRec)) / 16; b += blockDim.x) dst[b] = srcb[b];
  }
  __syncthreads();
  const SpRec* sp = reinterpret_cast<const SpRec*>(smem);
  const long stride = (long)gridDim.x * blockDim.x;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < P.ncells; c += stride) {
    const unsigned u = (unsigned)c;
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    if constexpr (MODE == EOS_FLOOR) {
      const long offY = aoff(P.rY, i, j, k);
      double rho = 0.0;
#pragma unroll 4
      for (int s = 0; s < N; ++s) {
        double x = P.rY.p[offY + (long)s * P.rY.ns];
        x = (x < DBL_MAX) ? x : DBL_MAX;  // min(DBL_MAX, x): NaN becomes DBL_MAX
        x = (0.0 < x) ? x : 0.0;          // max(0, x): negatives and -0 become +0
        P.rY.p[offY + (long)s * P.rY.ns] = x;
        rho += x;
      }
      const double rhoinv = 1.0 / rho;
      const double T = P.T.p[aoff(P.T, i, j, k)];
      const double invT = 1.0 / T;
      double h = 0.0;
#pragma unroll 4
      for (int s = 0; s < N; ++s) {  // the floored values just written, re-read from the row
        double cpR, hRT;
        nasa_hcp(sp[s], T, invT, cpR, hRT);
        h += ((P.rY.p[offY + (long)s * P.rY.ns] * rhoinv * hRT) * sp[s].RW) * T;
      }
      P.rho.p[aoff(P.rho, i, j, k)] = rho;
      P.rH.p[aoff(P.rH, i, j, k)] = (h * 1.0e-4) * rho;
    } else {
      const double T = P.T.p[aoff(P.T, i, j, k)];
      const double invT = 1.0 / T;
      const long offR = aoff(P.IR, i, j, k);
      double hr = 0.0;
#pragma unroll 4
      for (int s = 0; s < N; ++s) {
        double cpR, hRT;
        nasa_hcp(sp[s], T, invT, cpR, hRT);
        hr -= (((hRT * sp[s].RW) * T) * 0.0001) * P.IR.p[offR + (long)s * P.IR.ns];
      }
      P.HR.p[aoff(P.HR, i, j, k)] = hr;
    }
  }
}

// setTemperature with G lanes per cell in the rows layout (block_rates.h): the pairwise sums start
// inside a lane and end in DPP adds. What bounds it is the latency of the iteration (a reciprocal,
// two fourth-order polynomials per species, a division) for a box of tens of thousands of cells and
// FP64 issue above. One thread per cell, the sums over a tree of pending partial sums, was slower at
// every size (us per call, thread / rows): drm19 512 cells 66 / 26, 64000 71 / 32, 262144 97 / 59,
// 884736 223 / 131; dodecane_lu 64000 91 / 50, 884736 378 / 351; LiDryer 262144 80 / 42.
template <int N, int R, int G>
__global__ void __launch_bounds__(256) set_temp_rows_kernel(EosParams P) {
  using C = BlockCell<N, R, G>;
  extern __shared__ __align__(16) unsigned char smem[];
  {
    const BlobLayout BL = blob_layout(N, R, P.neff, P.ninc);
    const uint4* srcb = reinterpret_cast<const uint4*>(P.blob + BL.off_sp);
    uint4* dst = reinterpret_cast<uint4*>(smem);
    for (int b = threadIdx.x; b < (int)(N * sizeof(SpRec)) / 16; b += blockDim.x) dst[b] = srcb[b];
  }
  __syncthreads();
  const SpRec* sp = reinterpret_cast<const SpRec*>(smem);
  const int lane = threadIdx.x % G;
  const long stride = (long)gridDim.x * (blockDim.x / G);
  for (long c = (long)blockIdx.x * (blockDim.x / G) + threadIdx.x / G; c < P.ncells; c += stride) {
    const unsigned u = (unsigned)c;
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    const double rhoinv = 1.0 / P.rho.p[aoff(P.rho, i, j, k)];
    const long offY = aoff(P.rY, i, j, k), oT = aoff(P.T, i, j, k);
    double Y[C::RPL];
#pragma unroll
    for (int s = 0; s < C::RPL; ++s) {
      const int ii = C::row(lane, s);
      Y[s] = ii < N ? P.rY.p[offY + (long)ii * P.rY.ns] * rhoinv : 0.0;
    }
    const double T = rows_hy2t<N, R, G>(sp, lane, Y, (P.rH.p[aoff(P.rH, i, j, k)] * rhoinv) * 1.0e4, P.T.p[oT]);
    if (lane == 0) P.T.p[oT] = T;
  }
}

// I_R formation after the advance (Source/PeleLMeX_Reactions.cpp:141-160, and :342-347 on the
// chemistry BoxArray): I_R_k = -(rhoY_old_k - rhoY_new_k) * dt_inv - F_rhoY_k with
// dt_inv = 1 / dt formed on the host, as the reference forms it before its ParallelFor. One
// thread per (cell, species), cells fastest so that the Array4 reads coalesce; HBM-bound (three
// reads and one write of 8 bytes per entry).
struct IrParams {
  int lo0, lo1, lo2, nx, ny;
  long ncells;
  int N;
  Arr rYo, rYn, F, IR;
  double dt_inv;
};

__global__ void __launch_bounds__(256) ir_kernel(IrParams P) {
  const long total = P.ncells * (long)P.N;
  const long stride = (long)gridDim.x * blockDim.x;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride) {
    const long c = e % P.ncells;
    const long n = e / P.ncells;
    const unsigned u = (unsigned)c;
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    const double o = P.rYo.p[aoff(P.rYo, i, j, k) + n * P.rYo.ns];
    const double w = P.rYn.p[aoff(P.rYn, i, j, k) + n * P.rYn.ns];
    const double f = P.F.p[aoff(P.F, i, j, k) + n * P.F.ns];
    P.IR.p[aoff(P.IR, i, j, k) + n * P.IR.ns] = -(o - w) * P.dt_inv - f;
  }
}

// The unit conversions around react in advanceChemistry (Source/PeleLMeX_Reactions.cpp:68-79
// before, :110-120 after), one thread per cell, MKS views:
//  before: rhoY_new = rhoY_old * 1e-3, F_rhoY *= 1e-3, T_new = T_old, rhoH_new = rhoH_old * 10,
//          F_rhoH *= 10 (the forcing is scaled in place, as the reference scales it);
//  after:  rhoY_new *= 1e3, F_rhoY *= 1e3, rhoH_new *= 0.1, F_rhoH *= 0.1, then
//          I_R = -(rhoY_old - rhoY_new) * dt_inv - F_rhoY (:141-160) from the restored forcing.
struct ChemBoxParams {
  int lo0, lo1, lo2, nx, ny;
  long ncells;
  int N;
  Arr rYo, rHo, To, rYn, rHn, Tn, FY, FH, IR;
  double dt_inv;
};

template <bool AFTER>
__global__ void __launch_bounds__(256) chem_units_kernel(ChemBoxParams P) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < P.ncells; c += stride) {
    const unsigned u = (unsigned)c;
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    const long oYo = aoff(P.rYo, i, j, k), oYn = aoff(P.rYn, i, j, k), oF = aoff(P.FY, i, j, k);
    if (!AFTER) {
      for (int n = 0; n < P.N; ++n) {
        P.rYn.p[oYn + n * P.rYn.ns] = P.rYo.p[oYo + n * P.rYo.ns] * 1.0e-3;
        P.FY.p[oF + n * P.FY.ns] *= 1.0e-3;
      }
      P.Tn.p[aoff(P.Tn, i, j, k)] = P.To.p[aoff(P.To, i, j, k)];
      P.rHn.p[aoff(P.rHn, i, j, k)] = P.rHo.p[aoff(P.rHo, i, j, k)] * 10.0;
      P.FH.p[aoff(P.FH, i, j, k)] *= 10.0;
    } else {
      const long oI = aoff(P.IR, i, j, k);
      for (int n = 0; n < P.N; ++n) {
        const double w = P.rYn.p[oYn + n * P.rYn.ns] * 1.0e3;
        const double f = P.FY.p[oF + n * P.FY.ns] * 1.0e3;
        P.rYn.p[oYn + n * P.rYn.ns] = w;
        P.FY.p[oF + n * P.FY.ns] = f;
        if (P.IR.p) P.IR.p[oI + n * P.IR.ns] = -(P.rYo.p[oYo + n * P.rYo.ns] - w) * P.dt_inv - f;
      }
      P.rHn.p[aoff(P.rHn, i, j, k)] *= 0.1;
      P.FH.p[aoff(P.FH, i, j, k)] *= 0.1;
    }
  }
}

// advanceChemistryBAChem's unit conversions on the chemistry BoxArray's copy, in place
// (Source/PeleLMeX_Reactions.cpp:228-238 and :284-291): before the react, rhoY and its forcing
// times 1e-3, rho h and its forcing times 10 (P.rYn, P.rHn, P.FY, P.FH); after it, the state only
// (rhoY times 1e3, rho h times 0.1: the forcing copy stays in CGS). ZERO_FC additionally writes
// FC = 0 (a covered box, which skips the react).
template <int MODE>   // 0 before, 1 after, 2 after with FC = 0
__global__ void __launch_bounds__(256) chem_units_inplace_kernel(ChemBoxParams P, Arr FC) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < P.ncells; c += stride) {
    const unsigned u = (unsigned)c;
    const int i = P.lo0 + (int)(u % (unsigned)P.nx);
    const int j = P.lo1 + (int)((u / (unsigned)P.nx) % (unsigned)P.ny);
    const int k = P.lo2 + (int)(u / ((unsigned)P.nx * (unsigned)P.ny));
    const long oY = aoff(P.rYn, i, j, k);
    if (MODE == 0) {
      const long oF = aoff(P.FY, i, j, k);
      for (int n = 0; n < P.N; ++n) {
        P.rYn.p[oY + n * P.rYn.ns] *= 1.0e-3;
        P.FY.p[oF + n * P.FY.ns] *= 1.0e-3;
      }
      P.rHn.p[aoff(P.rHn, i, j, k)] *= 10.0;
      P.FH.p[aoff(P.FH, i, j, k)] *= 10.0;
    } else {
      for (int n = 0; n < P.N; ++n) P.rYn.p[oY + n * P.rYn.ns] *= 1.0e3;
      P.rHn.p[aoff(P.rHn, i, j, k)] *= 0.1;
      if (MODE == 2) FC.p[aoff(FC, i, j, k)] = 0.0;
    }
  }
}

}  // namespace prk
