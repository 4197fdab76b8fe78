// fused64.hpp -- FP64 faces and flux divergence of 3D blocks in one kernel.
//
// One lane per face (k_flux_x1, k_flux_h) reconstructs every cell twice per
// direction and passes the face fluxes through HBM to k_divergence.  Here a
// workgroup owns a tile of columns and marches up a segment of levels, as
// the FP32-flux form's tile kernel does: the level's plane with its halo in
// LDS, one reconstruction per cell and direction, the x2 and x3 Riemann
// fluxes of the tile's faces as one item list (velocities rotated so that the
// normal one comes first, which is the order hllc and lmars read them in), x1
// faces marched in registers.  Each value comes from the same operations in
// the same order as in the per-face kernels, so du is equal bit for bit.
//
// Bound by FP64 VALU (two WENO5 per cell and variable, three Riemann
// fluxes).  The fluxes take the plane's place in LDS once the states are
// formed (a fourth barrier per level): 69 KB for 32 x 8 columns and five
// variables, so two workgroups and their eight wavefronts share a compute
// unit and cover each other's barriers.
#pragma once

#include "flux32.hpp"

namespace cg {

template <int NM, int TJ, int TK>
struct Fused64Lds {
  static constexpr int H = 3, PJ = TJ + 2 * H, PK = TK + 2 * H, N = 5 + NM, NP = PJ * PK;
  static constexpr int C2 = TJ + 2, C3 = TK + 2;  // cells with face states
  static constexpr int NQ2 = TK * C2, NQ = NQ2 + C3 * TJ;
  static constexpr int NF2 = TK * (TJ + 1), NF = NF2 + (TK + 1) * TJ;
  static constexpr int SHARED = NP > NF ? NP : NF;
  double pf[N * SHARED];       // plane (N, PK, PJ), then face fluxes (N, NF)
  double qm[N * NQ], qp[N * NQ];  // face states, velocities rotated
};

template <int NM, int OH, int OV, int TJ, int TK>
__device__ __forceinline__ void fused64_tile(const KGrid& g, const KThermo& th,
                                             const KSource& src, int rsolver, int j0, int k0,
                                             int c0, int c1, const double* __restrict__ w,
                                             const double* __restrict__ psf,
                                             const double* __restrict__ psv,
                                             double* __restrict__ du,
                                             Fused64Lds<NM, TJ, TK>& L) {
  using S = Fused64Lds<NM, TJ, TK>;
  constexpr int NT = TJ * TK, H = S::H, PJ = S::PJ, NP = S::NP, N = S::N;
  constexpr int IPR = 4 + NM, IVX = 1 + NM;
  constexpr int LO = (OV == 5) ? 0 : 1, HI = (OV == 5) ? 5 : 4;
  constexpr int C2 = S::C2, NQ2 = S::NQ2, NQ = S::NQ, NF2 = S::NF2, NF = S::NF;
  const bool decomp = g.grav != 0.0;
  const int t = threadIdx.x;
  const int tj = t % TJ, tk = t / TJ;
  const int j = j0 + tj, k = k0 + tk;
  const bool own = (j <= g.je) && (k <= g.ke);
  const int jc = min(j, g.je), kc = min(k, g.ke);  // lanes past the block
  const long long pc = g.pcol(kc, jc) * g.ps_c;
  const long long colb = (long long)kc * g.c.k + (long long)jc * g.c.j;
  constexpr int NPL = (NP + NT - 1) / NT;
  long long pbase[NPL];
#pragma unroll
  for (int m = 0; m < NPL; ++m) {
    const int e = min(t + m * NT, NP - 1);
    const int gj = min(max(j0 - H + e % PJ, 0), g.nc2 - 1);
    const int gk = min(max(k0 - H + e / PJ, 0), g.nc3 - 1);
    pbase[m] = (long long)gk * g.c.k + (long long)gj * g.c.j;
  }
  // x1 window of the own column: cells f - 3 + m of face f
  double q[N][6];
  double rdv[6];
  auto window = [&](int m, int i, double* wc, double pv) {
    if (decomp) {
      rdv[m] = decomp_r<NM>(th, wc);
      const int ib = decomp_cell(g, i);
      double pb = wc[IPR], db = wc[0], rb = rdv[m];
      if (ib != i) {  // outflow ghost: the boundary cell's T, p'
        double wb[N];
#pragma unroll
        for (int n = 0; n < N; ++n) wb[n] = w[colb + n * g.c.n + (long long)ib * g.c.i];
        pb = wb[IPR];
        db = wb[0];
        rb = decomp_r<NM>(th, wb);
        pv = psv[pc + ib * g.ps_i];
      }
      wc[0] = pb / (db * rb);
      wc[IPR] = pb - pv;
    }
#pragma unroll
    for (int n = 0; n < N; ++n) q[n][m] = wc[n];
  };
  auto face1 = [&](double* fx, double ps) {
    double wl[N], wr[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      double qm, qp;
      if (OV == 5) {
        weno5_cell<double>(q[n][0], q[n][1], q[n][2], q[n][3], q[n][4], &qm, &qp);
        wl[n] = qp;
        weno5_cell<double>(q[n][1], q[n][2], q[n][3], q[n][4], q[n][5], &qm, &qp);
        wr[n] = qm;
      } else {
        plm_cell<double>(q[n][1], q[n][2], q[n][3], &qm, &qp);
        wl[n] = qp;
        plm_cell<double>(q[n][2], q[n][3], q[n][4], &qm, &qp);
        wr[n] = qm;
      }
    }
    if (decomp) {
      wr[IPR] += ps;
      if (wr[IPR] < 0.) wr[IPR] = ps;
      const double gamma = sqrt(rdv[3] * rdv[2]);
      wr[0] = wr[IPR] / (wr[0] * gamma);
      wl[IPR] += ps;
      if (wl[IPR] < 0.) wl[IPR] = ps;
      wl[0] = wl[IPR] / (wl[0] * gamma);
    }
    face_check<NM, double>(g.status, wl, wr, 0.0);
    riemann<NM, 0, double>(th, rsolver, wl, wr, fx);
  };
#pragma unroll
  for (int m = LO; m <= HI; ++m) {
    const int i = c0 - 3 + m;
    double wc[N];
#pragma unroll
    for (int n = 0; n < N; ++n) wc[n] = w[colb + n * g.c.n + (long long)i * g.c.i];
    window(m, i, wc, decomp ? psv[pc + i * g.ps_i] : 0.0);
  }
  double fm[N];
  face1(fm, decomp ? psf[pc + c0 * g.ps_i] : 0.0);
  // the next level's plane cells and window cell, requested a level ahead
  double pl[NPL][N], wn[N], psvn = 0.0, psfn = 0.0;
  auto fetch = [&](int i) {
#pragma unroll
    for (int m = 0; m < NPL; ++m)
#pragma unroll
      for (int n = 0; n < N; ++n)
        pl[m][n] = w[pbase[m] + n * g.c.n + (long long)i * g.c.i];
    const int in = i + 1 - 3 + HI;
#pragma unroll
    for (int n = 0; n < N; ++n) wn[n] = w[colb + n * g.c.n + (long long)in * g.c.i];
    if (decomp) {
      psvn = psv[pc + in * g.ps_i];
      psfn = psf[pc + (i + 1) * g.ps_i];
    }
  };
  auto land = [&]() {
#pragma unroll
    for (int n = 0; n < N; ++n) {
#pragma unroll
      for (int m = 0; m < NPL; ++m) landed(pl[m][n]);
      landed(wn[n]);
    }
    landed(psvn);
    landed(psfn);
  };
  fetch(c0);
  land();
  const double A1 = g.dx2 * g.dx3, A2 = g.dx1 * g.dx3, A3 = g.dx1 * g.dx2;
  const double vol = g.dx1 * g.dx2 * g.dx3;
  const double wght = src.weight();
  for (int i = c0; i < c1; ++i) {
    // (1) the level's plane with its halo
#pragma unroll
    for (int m = 0; m < NPL; ++m) {
      const int e = t + m * NT;
      if (e < NP) {
#pragma unroll
        for (int n = 0; n < N; ++n) L.pf[n * NP + e] = pl[m][n];
      }
    }
    double wx[N];
#pragma unroll
    for (int n = 0; n < N; ++n) wx[n] = wn[n];
    const double psvx = psvn, psfx = psfn;
    if (i + 1 < c1) fetch(i + 1);
    __syncthreads();
    // (2) face states: x2 for the cells j0-1 .. j0+TJ of the tile's rows, x3
    //     for k0-1 .. k0+TK of its columns (started a wavefront further on,
    //     which evens out the remainders)
    auto states = [&](auto dirc, int e, int pj, int pk) {
      constexpr int D = decltype(dirc)::value;
      constexpr int st = (D == 1) ? 1 : PJ;
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int sv = (n >= IVX && n < IVX + 3) ? IVX + (n - IVX + D) % 3 : n;
        const double* pv = &L.pf[sv * NP + pk * PJ + pj];
        double qm, qp;
        if (OH == 5)
          weno5_cell<double>(pv[-2 * st], pv[-st], pv[0], pv[st], pv[2 * st], &qm, &qp);
        else
          plm_cell<double>(pv[-st], pv[0], pv[st], &qm, &qp);
        L.qm[n * NQ + e] = qm;
        L.qp[n * NQ + e] = qp;
      }
    };
    for (int e = t; e < NQ2; e += NT)
      states(std::integral_constant<int, 1>(), e, (e % C2) + H - 1, (e / C2) + H);
    {
      constexpr int R2 = ((NQ2 % NT) + 63) / 64 * 64;
      for (int e3 = (t + NT - R2) % NT; e3 < NQ - NQ2; e3 += NT)
        states(std::integral_constant<int, 2>(), NQ2 + e3, (e3 % TJ) + H, (e3 / TJ) + H - 1);
    }
    __syncthreads();
    // (3) x2 and x3 fluxes of the tile's faces into the plane's place; faces
    //     past the block's end are not checked (their cells are not its own)
    for (int e = t; e < NF; e += NT) {
      const bool x2 = e < NF2;
      const int e3 = e - NF2;
      const int lq = x2 ? (e / (TJ + 1)) * C2 + e % (TJ + 1) : NQ2 + e3;
      const int rq = lq + (x2 ? 1 : TJ);
      double wl[N], wr[N], fx[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        wl[n] = L.qp[n * NQ + lq];
        wr[n] = L.qm[n * NQ + rq];
      }
      const int fj = j0 + (x2 ? e % (TJ + 1) : e3 % TJ), fk = k0 + (x2 ? e / (TJ + 1) : e3 / TJ);
      if (fj <= g.je + (x2 ? 1 : 0) && fk <= g.ke + (x2 ? 0 : 1))
        face_check<NM, double>(g.status, wl, wr, 0.0);
      riemann<NM, 0, double>(th, rsolver, wl, wr, fx);
#pragma unroll
      for (int n = 0; n < N; ++n) L.pf[n * NF + e] = fx[n];
    }
    // (4) x1 face i + 1, then the cell's divergence and sources
#pragma unroll
    for (int m = LO; m < HI; ++m) {
#pragma unroll
      for (int n = 0; n < N; ++n) q[n][m] = q[n][m + 1];
      rdv[m] = rdv[m + 1];
    }
    window(HI, i + 1 - 3 + HI, wx, psvx);
    double fp[N];
    face1(fp, psfx);
    land();
    __syncthreads();
    if (own) {
      double d[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        // slot of component n among the rotated momenta of x2 / x3 faces
        const int s2 = (n >= IVX && n < IVX + 3) ? IVX + (n - IVX + 2) % 3 : n;
        const int s3 = (n >= IVX && n < IVX + 3) ? IVX + (n - IVX + 1) % 3 : n;
        const int f2 = s2 * NF + tk * (TJ + 1) + tj, f3 = s3 * NF + NF2 + tk * TJ + tj;
        double dflx = A1 * fp[n] - A1 * fm[n];
        dflx += A2 * L.pf[f2 + 1] - A2 * L.pf[f2];
        dflx += A3 * L.pf[f3 + TJ] - A3 * L.pf[f3];
        d[n] = 0.0 - wght * dflx / vol;
      }
      add_sources_cell<NM>(g, th, src, w, decomp ? psv : nullptr, k, j, i, d);
#pragma unroll
      for (int n = 0; n < N; ++n)
        __builtin_nontemporal_store(d[n], &du[colb + n * g.c.n + (long long)i * g.c.i]);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) fm[n] = fp[n];
    __syncthreads();  // the fluxes are read before the next plane is staged
  }
}

// The tiles of every 3D block of a run in one launch.
template <int NM, int OH, int OV, int TJ, int TK>
__global__ void __launch_bounds__(TJ * TK)
    k_fused64_batch(const KBlockPtr* __restrict__ bp, const KTile* __restrict__ tiles,
                    KThermo th, KSource src, int rsolver) {
  __shared__ Fused64Lds<NM, TJ, TK> L;
  const KTile tt = tiles[blockIdx.x];
  const int b = __builtin_amdgcn_readfirstlane(tt.b);
  if (b < 0) return;  // padding of the table
  const KBlockPtr& p = bp[b];
  fused64_tile<NM, OH, OV, TJ, TK>(
      p.g, th, src, rsolver, __builtin_amdgcn_readfirstlane(tt.j0),
      __builtin_amdgcn_readfirstlane(tt.k0), __builtin_amdgcn_readfirstlane(tt.c0),
      __builtin_amdgcn_readfirstlane(tt.c1), gptr(p.w), gptr(p.psf), gptr(p.psv), gptr(p.du), L);
}

}  // namespace cg
