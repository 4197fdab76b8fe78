// rows.hpp -- implicit lines with eight lanes per line.
//
// The one-lane-per-line sweeps (fwd_column / bwd_update_column, lines.hpp)
// issue the whole algebra of a level, about 3,800 instructions, from one
// wavefront, so a launch with fewer than 65,536 lines leaves SIMDs idle and
// takes as long as one with 65,536.  Here a wavefront holds eight lines, one
// per octet of lanes, and the work of a level is spread over its octet:
//
//   assembly    eight levels of each line at once, one (line, level) per
//               lane: Roe averages, |A|, Jacobians, the blocks a, b, c and
//               the right-hand side go to LDS
//   elimination level by level: lane q < B of the octet holds column q of M
//               and of c, lane B the right-hand side; the pivot column is
//               broadcast to the octet by DPP, each lane updates its columns
//   way back    level by level with lane r holding row r, then eight levels
//               at once, one (line, level) per lane: write-back, stage
//               update, ConservedToPrimitive, ghosts, hydrostatic pressures
//
// Every number is computed by the same operations in the same order as in
// the one-lane sweeps (and as in the CPU evaluation), so results are equal
// bit for bit; only which lane computes what differs.  A wavefront needs 40
// KB of LDS for B = 5 (80 doubles per lane), so four wavefronts fill a
// compute unit's 160 KB, one per SIMD.
#pragma once

#include "lines.hpp"

namespace cg {

constexpr int OCT = 8;              // lanes per line, levels per chunk
constexpr int RLINES = 64 / OCT;    // lines per wavefront
constexpr int RWAVES = 4;           // wavefronts per workgroup

// LDS doubles of a (line, level) record: the columns of [M | c | rhs] row by
// row, then b.  Both strides are odd, which keeps the one-record-per-lane
// writes and the one-column-per-lane reads free of bank conflicts.
template <int B>
struct RowRec {
  static constexpr int NC = 2 * B + 1;
  static constexpr int COLS = B * NC, BM = B * B;
  static constexpr int WAVE = 64 * (COLS + BM);  // doubles per wavefront
};

// DPP moves of a double; all 64 lanes must be active.  Lane CC of each octet
// to all of the octet (a DPP row holds two: both halves from the lower one,
// then banks 2 and 3 from the upper one), and the value of the lane below in
// the row.
template <int CC>
__device__ __forceinline__ double oct_bcast(double v) {
  const double lo = __builtin_amdgcn_mov_dpp(v, 0x150 + CC, 0xf, 0xf, true);
  return __builtin_amdgcn_update_dpp(lo, v, 0x150 + OCT + CC, 0xf, 0xc, false);
}
__device__ __forceinline__ double row_below1(double v) {
  return __builtin_amdgcn_mov_dpp(v, 0x111, 0xf, 0xf, true);
}

// LDS exchange between lanes of one wavefront: its LDS operations complete
// in order; the fence keeps the compiler from moving them across.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void oct_swap(bool sw, double& a, double& b) {
  const double x = a, y = b;
  a = sw ? y : x;
  b = sw ? x : y;
}

// Step CC of the Gauss-Jordan elimination with partial pivoting (first row of
// largest |pivot|): this lane's columns m and c against the broadcast pivot
// column (column CC of M, lane CC's m).  FMA: the fused update of the walled
// recurrences; else the separate product and difference of minv.  The full
// search runs only when some line of the wavefront needs it.
template <int B, bool FMA, int CC>
__device__ __forceinline__ void gj_oct_step(double* m, double* c, bool& ok) {
  double f[B];
#pragma unroll
  for (int r = 0; r < B; ++r) f[r] = oct_bcast<CC>(m[r]);
  // rows CC and B - 1 decide the first pivot nearly always (the energy row
  // has the largest entry unless the step is small), the diagonal the others
  bool other = false, sw = false;
  if constexpr (CC == 0) {
    sw = fabs(f[B - 1]) > fabs(f[0]);
    const double top = sw ? f[B - 1] : f[0];
#pragma unroll
    for (int r = 1; r < B - 1; ++r) other = other || (fabs(f[r]) >= fabs(top));
  } else {
#pragma unroll
    for (int r = CC + 1; r < B; ++r) other = other || (fabs(f[r]) > fabs(f[CC]));
  }
  if (__any(other)) {
    int p = CC;
    double best = fabs(f[CC]);
#pragma unroll
    for (int r = CC + 1; r < B; ++r) {
      const bool up = fabs(f[r]) > best;
      best = up ? fabs(f[r]) : best;
      p = up ? r : p;
    }
#pragma unroll
    for (int r = CC + 1; r < B; ++r) {
      oct_swap(p == r, f[CC], f[r]);
      oct_swap(p == r, m[CC], m[r]);
      oct_swap(p == r, c[CC], c[r]);
    }
  } else if constexpr (CC == 0) {
    oct_swap(sw, f[0], f[B - 1]);
    oct_swap(sw, m[0], m[B - 1]);
    oct_swap(sw, c[0], c[B - 1]);
  }
  if (f[CC] == 0.0) ok = false;
  const double inv = 1.0 / f[CC];
  m[CC] = m[CC] * inv;
  c[CC] = c[CC] * inv;
#pragma unroll
  for (int r = 0; r < B; ++r) {
    if (r == CC) continue;
    m[r] = FMA ? fma(-f[r], m[CC], m[r]) : m[r] - f[r] * m[CC];
    c[r] = FMA ? fma(-f[r], c[CC], c[r]) : c[r] - f[r] * c[CC];
  }
}

template <int B, bool FMA>
__device__ __forceinline__ void gj_oct(double* m, double* c, bool& ok) {
  gj_oct_step<B, FMA, 0>(m, c, ok);
  gj_oct_step<B, FMA, 1>(m, c, ok);
  gj_oct_step<B, FMA, 2>(m, c, ok);
  if constexpr (B == 5) {
    gj_oct_step<B, FMA, 3>(m, c, ok);
    gj_oct_step<B, FMA, 4>(m, c, ok);
  }
}

// Assembly of eight levels of the octet's line (LineAsm / fwd_column with one
// level per lane).  |A| of the face below a lane's cell is the one the lane
// below computed; the first lane takes `below`, the last face of the chunk
// before (of the line's lower end at the start).
template <int NM, int B, int DIR>
struct RowAsm {
  static constexpr int N = 5 + NM, IVX = 1 + NM, IEN = 4 + NM;
  const KLines& L;
  const KThermo& th;
  const double* __restrict__ w;
  const double* __restrict__ du;
  long long o;             // offset of the line's cell 0, variable 0
  // hydrostatic cell pressures of the column (runs with gravity and an
  // outflow x1 side, else null) and their stride: ghosts beyond an outflow
  // side enter as CalculateFluxes left them (outflow_ghost_w)
  const double* __restrict__ psv;
  long long ps;
  bool out_lo, out_hi;
  double gm1, gm, idt;
  int hi;
  Mt<B> below;
  double wm[N], wc[N], wp[N], dv[N];  // the chunk's cells, loaded ahead

  __device__ __forceinline__ void load(double* dst, int i) const {
#pragma unroll
    for (int n = 0; n < N; ++n) dst[n] = w[o + n * L.sn + (long long)i * L.sl];
  }
  __device__ __forceinline__ void jac(const double* wv, Mt<B>& out) const {
    double f[N];
    to_frame<NM, DIR>(wv, f);
    flux_jac<NM, B>(gm1, f, out);
  }
  __device__ __forceinline__ void abs_a(const double* wl, const double* wr, Mt<B>& out) const {
    double prim[N], pf[N];
    roe_average<NM>(prim, gm, wl, wr);
    to_frame<NM, DIR>(prim, pf);
    abs_roe_fma<NM, B>(th, pf, gm, out);
  }
  __device__ RowAsm(const KLines& L_, const KThermo& th_, const double* w_, const double* du_,
                    long long o_, double dt, const double* psv_, long long ps_, bool olo,
                    bool ohi)
      : L(L_), th(th_), w(w_), du(du_), o(o_), psv(psv_), ps(ps_), out_lo(olo), out_hi(ohi) {
    gm1 = th.gammad - 1.;
    gm = 0.5 * (gm1 + gm1);
    idt = 1. / dt;
    hi = L.lo + L.n - 1;
  }
  // |A| of the line's lowest face; with um1 the corner block c of the cell
  // below the line (periodic lines)
  __device__ __forceinline__ void start(Mt<B>* um1) {
    double a[N], c[N];
    load(a, L.lo - 1);
    load(c, L.lo);
    if (out_lo)
      outflow_ghost_w<NM>(th, c, psv[L.lo * ps], psv[(L.lo - 1) * ps], a);
    abs_a(a, c, below);
    if (um1) {
      Mt<B> d;
      jac(c, d);
#pragma unroll
      for (int r = 0; r < B; ++r)
#pragma unroll
        for (int q = 0; q < B; ++q) um1->a[r][q] = -(below.a[r][q] - d.a[r][q]) * L.sra;
    }
  }
  // cells of the lane's level i (past the end: the last level again)
  __device__ __forceinline__ void fetch(int i) {
    i = min(i, hi);
    load(wm, i - 1);
    load(wc, i);
    load(wp, i + 1);
#pragma unroll
    for (int n = 0; n < N; ++n) dv[n] = du[o + n * L.sn + (long long)i * L.sl];
  }
  __device__ __forceinline__ void land() {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      landed(wm[n]);
      landed(wc[n]);
      landed(wp[n]);
      landed(dv[n]);
    }
  }
  // records of the fetched chunk; fold_lo, fold_hi: reflecting walls at the
  // line's ends; seven: the next chunk starts at the eighth lane's level
  __device__ __forceinline__ void store(int i, bool fold_lo, bool fold_hi,
                                        double* __restrict__ cols, double* __restrict__ bm,
                                        bool seven = false) {
    constexpr int NC = RowRec<B>::NC;
    i = min(i, hi);
    if (out_lo && i == L.lo)
      outflow_ghost_w<NM>(th, wc, psv[L.lo * ps], psv[(L.lo - 1) * ps], wm);
    if (out_hi && i == hi)
      outflow_ghost_w<NM>(th, wc, psv[hi * ps], psv[(hi + 1) * ps], wp);
    const bool first = (threadIdx.x & (OCT - 1)) == 0;
    Mt<B> Ap, Am, dm, dp;
    abs_a(wc, wp, Ap);
#pragma unroll
    for (int r = 0; r < B; ++r)
#pragma unroll
      for (int q = 0; q < B; ++q) {
        const double v = row_below1(Ap.a[r][q]);
        Am.a[r][q] = first ? below.a[r][q] : v;
        below.a[r][q] = seven ? oct_bcast<OCT - 2>(Ap.a[r][q]) : oct_bcast<OCT - 1>(Ap.a[r][q]);
      }
    jac(wm, dm);
    jac(wp, dp);
    Mt<B> M, b, c;
#pragma unroll
    for (int r = 0; r < B; ++r)
#pragma unroll
      for (int q = 0; q < B; ++q) {
        double phi = 0.0;
        if ((r == 1 && q == 0) || (r == B - 1 && q == 1)) phi = L.grav;
        // the faces of a Cartesian cell are equal (sda = 0): no dc term
        double av = fma(Am.a[r][q], L.sla, Ap.a[r][q] * L.sra);
        if (r == q) av += idt;
        M.a[r][q] = av - phi;
        b.a[r][q] = -(Am.a[r][q] + dm.a[r][q]) * L.sla;
        c.a[r][q] = -(Ap.a[r][q] - dp.a[r][q]) * L.sra;
      }
    if (fold_lo && i == L.lo) {
#pragma unroll
      for (int r = 0; r < B; ++r)
#pragma unroll
        for (int q = 0; q < B; ++q) M.a[r][q] += (q == 1) ? -b.a[r][q] : b.a[r][q];
    }
    if (fold_hi && i == hi) {
#pragma unroll
      for (int r = 0; r < B; ++r)
#pragma unroll
        for (int q = 0; q < B; ++q) M.a[r][q] += (q == 1) ? -c.a[r][q] : c.a[r][q];
    }
    double r0 = dv[0];
#pragma unroll
    for (int n = 1; n < IVX; ++n) r0 += dv[n];
    double t[B];
    t[0] = r0 * idt;
    t[1] = dv[IVX + DIR] * idt;
    if (B == 5) {
      t[2] = dv[IVX + (1 + DIR) % 3] * idt;
      t[3] = dv[IVX + (2 + DIR) % 3] * idt;
    }
    t[B - 1] = dv[IEN] * idt;
#pragma unroll
    for (int r = 0; r < B; ++r) {
#pragma unroll
      for (int q = 0; q < B; ++q) {
        cols[r * NC + q] = M.a[r][q];
        cols[r * NC + B + q] = c.a[r][q];
        bm[r * B + q] = b.a[r][q];
      }
      cols[r * NC + 2 * B] = t[r];
    }
  }
};

// Archive of the wavefront's nl lines: the B (B + 1) doubles of a (line,
// level) record, rows of [a' | delta] one after the other, in pairs; a chunk
// of m levels from p0 keeps pair k of all its records together, so that a
// wavefront writes and reads it with one record per lane in whole segments.
template <int B>
struct OctArchive {
  static constexpr int AS = B * (B + 1), PAIRS = AS / 2, LS = AS + 1;  // LS: LDS stride
  double2* ar;
  int n, nl;
  __device__ __forceinline__ double2* at(int p0, int line, int l8, int& step) const {
    const int m = min(OCT, n - p0);
    step = nl * m;
    return ar + (long long)p0 * PAIRS * nl + min(line, nl - 1) * m + min(l8, m - 1);
  }
};

// ForwardSweep of the wavefront's lines.  A level's results take the place of
// its columns in LDS and go to the archive once per chunk, before the next
// chunk's cells are requested: a wait for loads also waits for the stores
// issued before them, and these have a whole chunk of elimination to
// complete.  Returns false on a zero pivot.
template <int NM, int B, int DIR>
__device__ __forceinline__ bool oct_forward(RowAsm<NM, B, DIR>& as, double* __restrict__ sh,
                                            const OctArchive<B>& ar, bool fold_lo,
                                            bool fold_hi) {
  constexpr int NC = RowRec<B>::NC, COLS = RowRec<B>::COLS, BM = RowRec<B>::BM;
  const int lane = threadIdx.x & 63, line = lane / OCT, l8 = lane & (OCT - 1);
  const int n = as.L.n, lo = as.L.lo;
  double* cols = sh;
  double* bms = sh + 64 * COLS;
  // lane q < B: m = column q of M, c = column q of c; lane B: m = the
  // right-hand side; the lanes above repeat column 0
  const int q = l8 < B ? l8 : 0;
  const bool is_t = l8 == B;
  bool ok = true;
  struct Rec {
    double m[B], c[B], b[BM];
  };
  const double* pm = cols + line * OCT * COLS + (is_t ? 2 * B : q);
  const double* pc = cols + line * OCT * COLS + B + q;
  const double* pb = bms + line * OCT * BM;
  auto get = [&](Rec& R, int l) {
#pragma unroll
    for (int r = 0; r < B; ++r) {
      R.m[r] = pm[l * COLS + r * NC];
      R.c[r] = pc[l * COLS + r * NC];
    }
#pragma unroll
    for (int e = 0; e < BM; ++e) R.b[e] = pb[l * BM + e];
  };
  double* po = cols + line * OCT * COLS + l8;
  double y[B];  // the lane's column of [a' | delta] of the level below
  auto level = [&](Rec& R, int l, bool first) {
    // M -= b a'_{p-1}, rhs -= b delta_{p-1}
    if (!first) {
#pragma unroll
      for (int r = 0; r < B; ++r)
#pragma unroll
        for (int kk = 0; kk < B; ++kk) R.m[r] = fma(-R.b[r * B + kk], y[kk], R.m[r]);
    }
    gj_oct<B, true>(R.m, R.c, ok);
#pragma unroll
    for (int r = 0; r < B; ++r) y[r] = is_t ? R.m[r] : R.c[r];
    if (l8 <= B) {
#pragma unroll
      for (int r = 0; r < B; ++r) po[l * COLS + r * NC] = y[r];
    }
  };
  as.start(nullptr);
  as.fetch(lo + l8);
  as.land();
  for (int p0 = 0; p0 < n; p0 += OCT) {
    as.store(lo + p0 + l8, fold_lo, fold_hi, cols + lane * COLS, bms + lane * BM);
    wave_sync();
    if (p0 + OCT < n) as.fetch(lo + p0 + OCT + l8);
    const int m = min(OCT, n - p0);
    // two records in turn, each read from LDS a level ahead of its use
    Rec R0, R1;
    get(R0, 0);
    for (int l = 0; l < m; l += 2) {
      get(R1, min(l + 1, m - 1));
      level(R0, l, p0 + l == 0);
      if (l + 1 >= m) break;
      get(R0, min(l + 2, m - 1));
      level(R1, l + 1, false);
    }
    as.land();
    wave_sync();
    if (l8 < m && line < ar.nl) {
      const double* src = cols + lane * COLS;
      int step;
      double2* dst = ar.at(p0, line, l8, step);
#pragma unroll
      for (int k = 0; k < OctArchive<B>::PAIRS; ++k) {
        const int e = 2 * k / (B + 1) * NC + 2 * k % (B + 1);
        dst[(long long)k * step] = double2{src[e], src[e + 1]};
      }
    }
    wave_sync();
  }
  return ok;
}

// a . x of a row a with the vector whose component k lane k of the octet
// holds, terms in order.
template <int B>
struct OctDot {
  template <int K>
  static __device__ __forceinline__ double term(const double* a, double x) {
    if constexpr (K == 0)
      return a[0] * oct_bcast<0>(x);
    else
      return term<K - 1>(a, x) + a[K] * oct_bcast<K>(x);
  }
  static __device__ __forceinline__ double dot(const double* a, double x) {
    return term<B - 1>(a, x);
  }
};

// Back substitution of a chunk of eight levels from p0, top down: the
// records pass from one per lane through LDS to one row per lane; lane r of
// the octet carries component r of the solution x (that of the level above,
// then of level p0), which also goes to LDS, B doubles per (line, level).
// The archive of the next chunk down is requested as soon as this one's is in
// LDS (deeper prefetch only fills the queue of outstanding requests).
template <int B>
struct OctBack {
  using A = OctArchive<B>;
  const A& ar;
  double x;
  double2 buf[A::PAIRS];
  __device__ __forceinline__ void fetch(int p0) {
    const int lane = threadIdx.x & 63;
    int step;
    const double2* a = ar.at(max(p0, 0), lane / OCT, lane & (OCT - 1), step);
#pragma unroll
    for (int k = 0; k < A::PAIRS; ++k) buf[k] = a[(long long)k * step];
  }
  // sa: 64 LS doubles for the records, sd: 64 B doubles for the solution
  __device__ __forceinline__ void land() {
#pragma unroll
    for (int k = 0; k < A::PAIRS; ++k) {
      landed(buf[k].x);
      landed(buf[k].y);
    }
  }
  __device__ __forceinline__ void to_lds(double* sa) const {
    const int lane = threadIdx.x & 63;
    wave_sync();
#pragma unroll
    for (int k = 0; k < A::PAIRS; ++k) {
      sa[lane * A::LS + 2 * k] = buf[k].x;
      sa[lane * A::LS + 2 * k + 1] = buf[k].y;
    }
    wave_sync();
  }
  __device__ __forceinline__ void chunk(int p0, const double* sa, double* sd) {
    const int lane = threadIdx.x & 63, l8 = lane & (OCT - 1), r = min(l8, B - 1);
    const double* pr = sa + (lane - l8) * A::LS + r * (B + 1);
    double* px = sd + (lane - l8) * B + r;
    double v[OCT][B + 1];
#pragma unroll
    for (int h = 0; h < OCT; ++h)
#pragma unroll
      for (int k = 0; k <= B; ++k) v[h][k] = pr[h * A::LS + k];
#pragma unroll
    for (int h = OCT - 1; h >= 0; --h) {
      if (p0 + h >= ar.n) continue;
      const double s = OctDot<B>::dot(v[h], x);
      x = (p0 + h == ar.n - 1) ? v[h][B] : v[h][B] - s;
      if (l8 < B) px[h * B] = x;
    }
    wave_sync();
  }
};

// The archive is read back by other lanes of the wavefront that wrote it.
__device__ __forceinline__ void archive_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

// Lines between walls of any direction on caller arrays or a run's state
// (x1 columns; x2 and x3 lines as k_line_walls).  lv: n (B B + B) doubles
// per line.
template <int NM, int B, int DIR>
__global__ void __launch_bounds__(64 * RWAVES)
    k_rows_walls(KLines L, KThermo th, double dt, const double* __restrict__ dtp,
                 bool fold_lo, bool fold_hi, const double* __restrict__ w, double* __restrict__ du,
                 double* __restrict__ lv, int* __restrict__ status) {
  __shared__ double shm[RWAVES * RowRec<B>::WAVE];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long long line0 = ((long long)blockIdx.x * RWAVES + wv) * RLINES;
  if (line0 >= L.nline) return;  // whole wavefronts; no workgroup barrier below
  double* sh = shm + wv * RowRec<B>::WAVE;
  const int lane = threadIdx.x & 63, line = lane / OCT, l8 = lane & (OCT - 1);
  const int nl = (int)min((long long)RLINES, L.nline - line0);
  const long long t = line0 + min(line, nl - 1);
  const long long o = L.org(t);
  const OctArchive<B> ar{reinterpret_cast<double2*>(lv + line0 * L.n * (B * B + B)), L.n, nl};
  if (dtp) dt = dt * dtp[0];
  RowAsm<NM, B, DIR> as(L, th, w, du, o, dt, nullptr, 0, false, false);
  const bool ok = oct_forward<NM, B, DIR>(as, sh, ar, fold_lo, fold_hi);
  if (!ok && line < nl) atomicOr(status, 1);
  archive_fence();
  double* sd = sh + 64 * OctArchive<B>::LS;
  OctBack<B> bk{ar, 0.0};
  const int ptop = (L.n - 1) / OCT * OCT;
  LineCell<NM, DIR> cell;
  auto fetch = [&](int p0) {
    bk.fetch(p0);
    cell.load(L, w, du, o, t, L.lo + min(max(p0, 0) + l8, L.n - 1), true);
  };
  fetch(ptop);
  bk.land();
  cell.land();
  for (int p0 = ptop; p0 >= 0; p0 -= OCT) {
    bk.to_lds(sh);
    const LineCell<NM, DIR> c = cell;
    fetch(p0 - OCT);
    bk.chunk(p0, sh, sd);
    Vt<B> d;
#pragma unroll
    for (int k = 0; k < B; ++k) d.v[k] = sd[lane * B + k];
    const int p = p0 + l8;
    bk.land();
    cell.land();
    if (p < L.n && line < nl)
      line_store<NM, B, DIR, false>(d, c, du, o + (long long)(L.lo + p) * L.sl, L.sn);
  }
}

// A periodic line (k_line_periodic, lines.hpp, whose recurrences and order of
// operations these are) with eight lanes: lane q < B holds column q of ainv, U
// (= c), gamma and of the products, lane B the vector zeta in gamma's place.
// Left factors pass through LDS: T = b ainv_{p-1} and beta U are written by
// columns and read whole by every lane.  A level's record is free once its
// columns are in registers; the products use its slots, and at the end of the
// level it holds what the way back needs, row r as [zeta | U | gamma] (B (2B
// + 1) doubles) and ainv (B B): 80 doubles per cell instead of the one-lane
// kernel's 105.
template <int B>
__device__ __forceinline__ void mat_col(const double* x, const double* y, double* z) {
#pragma unroll
  for (int r = 0; r < B; ++r) {
    double s = x[r * B] * y[0];
#pragma unroll
    for (int k = 1; k < B; ++k) s += x[r * B + k] * y[k];
    z[r] = s;
  }
}

template <int NM, int B, int DIR>
__global__ void __launch_bounds__(64 * RWAVES)
    k_rows_periodic(KLines L, KThermo th, double dt, const double* __restrict__ dtp,
                    const double* __restrict__ w, double* __restrict__ du,
                    double* __restrict__ lv, int* __restrict__ status) {
  constexpr int NC = RowRec<B>::NC, COLS = RowRec<B>::COLS, BM = RowRec<B>::BM;
  constexpr int PAIRS = (COLS + BM) / 2;
  static_assert(2 * PAIRS == COLS + BM, "records go out in pairs");
  __shared__ double shm[RWAVES * RowRec<B>::WAVE];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long long line0 = ((long long)blockIdx.x * RWAVES + wv) * RLINES;
  if (line0 >= L.nline) return;  // whole wavefronts; no workgroup barrier below
  double* cols = shm + wv * RowRec<B>::WAVE;
  double* bms = cols + 64 * COLS;
  const int lane = threadIdx.x & 63, line = lane / OCT, l8 = lane & (OCT - 1);
  const int nl = (int)min((long long)RLINES, L.nline - line0);
  const long long t = line0 + min(line, nl - 1);
  const long long o = L.org(t);
  const int n = L.n, lo = L.lo;
  double2* ar = reinterpret_cast<double2*>(lv + line0 * n * (COLS + BM));
  if (dtp) dt = dt * dtp[0];
  RowAsm<NM, B, DIR> as(L, th, w, du, o, dt, nullptr, 0, false, false);
  // chunks of eight levels; the first has seven where the last level would
  // otherwise start a chunk, since level n - 2 reads level n - 1's b
  const int first = ((n - 1) % OCT == 0) ? OCT - 1 : OCT;
  const int q = l8 < B ? l8 : 0;
  const bool is_z = l8 == B, is_c = l8 < B;
  bool ok = true;
  double bf[BM];              // beta_{p-1}, whole (at first the corner c_{lo-1})
  double ai[B], U[B], gm[B];  // the lane's columns of level p - 1
  double sb[B];               // sum of beta gamma (lane B: beta zeta)
  {
    Mt<B> um1;
    as.start(&um1);
#pragma unroll
    for (int r = 0; r < B; ++r) {
      sb[r] = 0.0;
      ai[r] = U[r] = gm[r] = 0.0;
#pragma unroll
      for (int k = 0; k < B; ++k) bf[r * B + k] = um1.a[r][k];
    }
  }
  as.fetch(lo + l8);
  as.land();
  auto flush = [&](int p0, int m) {
    if (l8 < m && line < nl) {
      const double* c = cols + lane * COLS;
      const double* b = bms + lane * BM;
      double2* dst = ar + (long long)p0 * PAIRS * nl + line * m + l8;
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) {
        const int e0 = 2 * k, e1 = 2 * k + 1;
        dst[(long long)k * nl * m] = double2{e0 < COLS ? c[e0] : b[e0 - COLS],
                                             e1 < COLS ? c[e1] : b[e1 - COLS]};
      }
    }
  };
  double xl = 0.0;  // component min(l8, B - 1) of the last level's solution
  for (int p0 = 0, len = first; p0 < n; p0 += len, len = OCT) {
    as.store(lo + p0 + l8, false, false, cols + lane * COLS, bms + lane * BM, len < OCT);
    wave_sync();
    if (p0 + len < n) as.fetch(lo + p0 + len + l8);
    const int m = min(len, n - p0);
    for (int l = 0; l < m; ++l) {
      const int p = p0 + l;
      double* rc = cols + (lane - l8 + l) * COLS;
      double* rb = bms + (lane - l8 + l) * BM;
      double a[B], c[B], tmp[BM];
#pragma unroll
      for (int r = 0; r < B; ++r) {
        a[r] = rc[r * NC + (is_z ? 2 * B : q)];  // lane B: the right-hand side
        c[r] = rc[r * NC + B + q];
      }
      double x[B], inv[B];
      if (p == n - 1) {
        // ainv = (a - sum beta gamma)^-1, zeta = r - sum beta zeta
#pragma unroll
        for (int r = 0; r < B; ++r) {
          a[r] = a[r] - sb[r];
          inv[r] = (r == q) ? 1.0 : 0.0;
        }
        wave_sync();
        if (is_z) {
#pragma unroll
          for (int r = 0; r < B; ++r) rc[r] = a[r];
        }
        gj_oct<B, false>(a, inv, ok);
        if (is_c) {
#pragma unroll
          for (int r = 0; r < B; ++r) rb[r * B + q] = inv[r];
        }
        wave_sync();
        const int rr = min(l8, B - 1);
        double s = rb[rr * B] * rc[0];
#pragma unroll
        for (int k = 1; k < B; ++k) s += rb[rr * B + k] * rc[k];
        xl = s;
        wave_sync();
        break;
      }
#pragma unroll
      for (int e = 0; e < BM; ++e) tmp[e] = rb[e];
      double gnew[B], bu[B];
      if (p == 0) {
        // gamma_0 = b_0, zeta_0 = r_0
#pragma unroll
        for (int r = 0; r < B; ++r) gnew[r] = is_z ? a[r] : rb[r * B + q];
      } else {
        double T[B];
        mat_col<B>(tmp, ai, T);  // T = b ainv_{p-1}
        wave_sync();
        if (is_c) {
#pragma unroll
          for (int r = 0; r < B; ++r) rb[r * B + q] = T[r];
        }
        wave_sync();
#pragma unroll
        for (int e = 0; e < BM; ++e) tmp[e] = rb[e];
        mat_col<B>(tmp, gm, x);  // T gamma_{p-1}, lane B: T zeta_{p-1}
#pragma unroll
        for (int r = 0; r < B; ++r)
          gnew[r] = is_z ? a[r] - x[r] : p < n - 2 ? -x[r] : c[r] - x[r];
        mat_col<B>(tmp, U, x);
#pragma unroll
        for (int r = 0; r < B; ++r) a[r] = a[r] - x[r];
        mat_col<B>(bf, U, bu);  // beta_{p-1} U_{p-1}
        if (p == n - 2) {       // L_{n-1} - beta_{n-3} U_{n-3}
#pragma unroll
          for (int r = 0; r < B; ++r) bu[r] = rb[BM + r * B + q] - bu[r];
        }
        wave_sync();
        if (is_c) {
#pragma unroll
          for (int r = 0; r < B; ++r) rc[r * B + q] = bu[r];
        }
        wave_sync();
#pragma unroll
        for (int e = 0; e < BM; ++e) bf[e] = rc[e];
      }
#pragma unroll
      for (int r = 0; r < B; ++r) inv[r] = (r == q) ? 1.0 : 0.0;
      gj_oct<B, false>(a, inv, ok);
      mat_col<B>(bf, inv, bu);  // beta_p
      if (p > 0 && p < n - 2) {
#pragma unroll
        for (int r = 0; r < B; ++r) bu[r] = -bu[r];
      }
      wave_sync();
      if (is_c) {
#pragma unroll
        for (int r = 0; r < B; ++r) rc[r * B + q] = bu[r];
      }
      wave_sync();
#pragma unroll
      for (int e = 0; e < BM; ++e) bf[e] = rc[e];
      mat_col<B>(bf, gnew, x);
#pragma unroll
      for (int r = 0; r < B; ++r) {
        sb[r] = sb[r] + x[r];
        ai[r] = inv[r];
        U[r] = c[r];
        gm[r] = gnew[r];
      }
      wave_sync();
      if (l8 <= B) {
#pragma unroll
        for (int r = 0; r < B; ++r) {
          rc[r * NC + (is_z ? 0 : 1 + B + q)] = gnew[r];
          if (is_c) {
            rc[r * NC + 1 + q] = c[r];
            rb[r * B + q] = inv[r];
          }
        }
      }
    }
    as.land();
    wave_sync();
    flush(p0, m);
    wave_sync();
  }
  if (!ok && line < nl) atomicOr(status, 1);
  archive_fence();
  // the way back, top chunk first: lane r holds component r of x
  double2 buf[PAIRS];
  LineCell<NM, DIR> cell;
  auto length = [&](int p0) { return p0 == 0 ? min(first, n) : min(OCT, n - p0); };
  auto fetch = [&](int p0) {
    const int m = length(p0);
    const double2* src = ar + (long long)p0 * PAIRS * nl + min(line, nl - 1) * m + min(l8, m - 1);
#pragma unroll
    for (int k = 0; k < PAIRS; ++k) buf[k] = src[(long long)k * nl * m];
    cell.load(L, w, du, o, t, lo + p0 + min(l8, m - 1), false);
  };
  auto land = [&]() {
#pragma unroll
    for (int k = 0; k < PAIRS; ++k) {
      landed(buf[k].x);
      landed(buf[k].y);
    }
    cell.land();
  };
  const int rr = min(l8, B - 1);
  double xv = xl;
  int p0 = n <= first ? 0 : first + (n - 1 - first) / OCT * OCT;
  fetch(p0);
  land();
  while (true) {
    const int m = length(p0);
    wave_sync();
    {
      double* c = cols + lane * COLS;
      double* b = bms + lane * BM;
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) {
        const int e0 = 2 * k, e1 = 2 * k + 1;
        (e0 < COLS ? c[e0] : b[e0 - COLS]) = buf[k].x;
        (e1 < COLS ? c[e1] : b[e1 - COLS]) = buf[k].y;
      }
    }
    const LineCell<NM, DIR> mine = cell;
    const int next = p0 == 0 ? -1 : p0 == first ? 0 : p0 - OCT;
    if (next >= 0) fetch(next);
    wave_sync();
    for (int l = m - 1; l >= 0; --l) {
      double* rc = cols + (lane - l8 + l) * COLS + rr * NC;
      const double* rb = bms + (lane - l8 + l) * BM + rr * B;
      if (p0 + l < n - 1) {
        double ux = 0.0;
        if (p0 + l < n - 2) ux = OctDot<B>::dot(rc + 1, xv);
        const double gx = OctDot<B>::dot(rc + 1 + B, xl);
        const double tv = (rc[0] - ux) - gx;
        xv = OctDot<B>::dot(rb, tv);
      }
      if (l8 < B) rc[0] = xv;
    }
    wave_sync();
    Vt<B> d;
#pragma unroll
    for (int r = 0; r < B; ++r) d.v[r] = cols[lane * COLS + r * NC];
    land();
    if (l8 < m && line < nl)
      line_store<NM, B, DIR, true>(d, mine, du, o + (long long)(lo + p0 + l8) * L.sl, L.sn);
    if (next < 0) break;
    p0 = next;
  }
}

// The x1 columns of a block as lines (lanes along x2, as the column tables
// of a run).
__device__ __forceinline__ KLines column_lines(const KGrid& g) {
  KLines L;
  L.nf = g.nx2;
  L.nline = (long long)g.nx2 * g.nx3;
  L.n = g.nx1;
  L.lo = g.is;
  L.org0 = (long long)g.js * g.c.j + (long long)g.ks * g.c.k;
  L.sf = g.c.j;
  L.ss = g.c.k;
  L.sl = g.c.i;
  L.sn = g.c.n;
  const double area = g.dx2 * g.dx3, vol = g.dx1 * g.dx2 * g.dx3;
  const double s2v = 1. / (2. * vol);
  L.sla = area * s2v;
  L.sra = area * s2v;
  L.sda = 0.0;
  L.grav = g.grav;
  L.td0 = 1;
  L.td1 = 2;
  L.t0s = g.js;
  L.t1s = g.ks;
  L.nc1 = g.nc1;
  L.nc2 = g.nc2;
  L.nc3 = g.nc3;
  L.c = g.c;
  return L;
}

// A stage's column solve and update of a run (k_implicit_fused_batch), eight
// columns per wavefront over the same group table: wavefront v takes columns
// 8 (v % 8) .. + 7 of group v / 8.  A block's archive keeps its place
// (aoff); the columns of a wavefront are contiguous in it.  The x1 sides are
// walls or outflow.
template <int NM, int B>
__global__ void __launch_bounds__(64 * RWAVES)
    k_rows_update_batch(const KBlockPtr* __restrict__ bp, const KGroup* __restrict__ grp,
                        int ngroups, KThermo th, double dt, const double* __restrict__ dtp,
                        KUpdate up, double* __restrict__ arch, int* __restrict__ status) {
  constexpr int N = 5 + NM, IVX = 1 + NM, IPR = 4 + NM;
  constexpr int PERG = 64 / RLINES;  // wavefronts per group
  __shared__ double shm[RWAVES * RowRec<B>::WAVE];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int v = blockIdx.x * RWAVES + wv;
  const int gq = v / PERG;
  if (gq >= ngroups) return;  // whole wavefronts; no workgroup barrier below
  const int b = __builtin_amdgcn_readfirstlane(grp[gq].b);
  const int line0 = __builtin_amdgcn_readfirstlane(grp[gq].col0) + (v % PERG) * RLINES;
  const long long aoff = grp[gq].aoff;
  const KGrid g = bp[b].g;
  const KLines L = column_lines(g);
  if (line0 >= L.nline) return;
  const double* w0 = gptr(bp[b].w);
  double *w = gptr(bp[b].w), *u = gptr(bp[b].u), *u1 = gptr(bp[b].u1);
  double *psf = gptr(bp[b].psf), *psv = gptr(bp[b].psv);
  const double* du = gptr(bp[b].du);
  double* sh = shm + wv * RowRec<B>::WAVE;
  const int lane = threadIdx.x & 63, line = lane / OCT, l8 = lane & (OCT - 1);
  const int nl = (int)min((long long)RLINES, L.nline - line0);
  const bool live = line < nl;
  const int t = line0 + min(line, nl - 1);
  const long long o = L.org(t), pc = (long long)t * g.ps_c;
  const OctArchive<B> ar{
      reinterpret_cast<double2*>(arch + aoff + (long long)line0 * L.n * (B * B + B)), L.n, nl};
  if (dtp) dt = dt * dtp[0];
  const bool hs = g.grav != 0.0;
  {
    RowAsm<NM, B, 0> as(L, th, w0, du, o, dt, psv + pc, g.ps_i, hs && g.bc[0] == 2,
                        hs && g.bc[1] == 2);
    const bool ok = oct_forward<NM, B, 0>(as, sh, ar, g.bc[0] != 1, g.bc[1] != 1);
    if (!ok && live) atomicOr(status, 1);
  }
  archive_fence();
  const int is = g.is, ie = g.ie;
  const long long sn = L.sn, si = L.sl;
  const double grav = g.grav, dx = g.dx1;
  // LDS of the way back: the solution, the hydrostatic steps grav rho dx of
  // a chunk, and per line the top face pressure and the densities of the three
  // cells next to each side
  double* sd = sh + 64 * OctArchive<B>::LS;
  double* st = sd + 64 * B + line * OCT;
  double* sx = sd + 64 * B + 64 + line * OCT;
  OctBack<B> bk{ar, 0.0};
  double pf_next = 0.0, pf_top = 0.0;
  const int ptop = (L.n - 1) / OCT * OCT;
  double nduo[N], nwsp[N], nuo[N], nu1o[N];
  auto fetch = [&](int p0) {  // the chunk's archive and the lane's cell
    bk.fetch(p0);
    const long long ci = o + (long long)min(is + max(p0, 0) + l8, ie) * si;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      nduo[n] = (n <= NM || B == 3) ? du[ci + n * sn] : 0.0;
      nwsp[n] = (n >= 1 && n <= NM) ? w0[ci + n * sn] : 0.0;
      nuo[n] = u[ci + n * sn];
      nu1o[n] = (up.stage == 0) ? 0.0 : u1[ci + n * sn];
    }
  };
  auto land = [&]() {
    bk.land();
#pragma unroll
    for (int n = 0; n < N; ++n) {
      if (n <= NM || B == 3) landed(nduo[n]);
      if (n >= 1 && n <= NM) landed(nwsp[n]);
      landed(nuo[n]);
      landed(nu1o[n]);
    }
  };
  fetch(ptop);
  land();
  for (int p0 = ptop; p0 >= 0; p0 -= OCT) {
    const int i = is + p0 + l8;
    const bool cell = live && i <= ie;
    const long long ci = o + (long long)min(i, ie) * si;
    bk.to_lds(sh);
    double duo[N], wsp[N], uo[N], u1o[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      duo[n] = nduo[n];
      wsp[n] = nwsp[n];
      uo[n] = nuo[n];
      u1o[n] = nu1o[n];
    }
    fetch(p0 - OCT);
    bk.chunk(p0, sh, sd);
    double wc[N], dun[N], uc[N];
    {
      Vt<B> d;
#pragma unroll
      for (int r = 0; r < B; ++r) d.v[r] = sd[lane * B + r];
      write_back<NM, B>(d, duo, wsp, dun);
    }
    land();
    if (cell) {
      update_cell_pre<NM>(th, up, uo, u1o, u1, ci, sn, dun, uc, wc, status);
      const int mt = ie - i, mb = i - is;  // distance from the sides
#pragma unroll
      for (int n = 0; n < N; ++n) {
        u[ci + n * sn] = uc[n];
        w[ci + n * sn] = wc[n];
        // x1 ghosts: mirrored at a wall, copies of the last cell at outflow
        const double mir = (n == IVX) ? -wc[n] : wc[n];
        if (mt < NG && g.bc[1] == 0) w[ci + n * sn + (2 * mt + 1) * si] = mir;
        if (mb < NG && g.bc[0] == 0) w[ci + n * sn - (2 * mb + 1) * si] = mir;
        if (mt == 0 && g.bc[1] == 2)
          for (int gh = 1; gh <= NG; ++gh) w[ci + n * sn + gh * si] = wc[n];
        if (mb == 0 && g.bc[0] == 2)
          for (int gh = 1; gh <= NG; ++gh) w[ci + n * sn - gh * si] = wc[n];
      }
      if (hs) {
        st[l8] = grav * wc[0] * dx;
        if (mt == 0) {
          const double RdTv = wc[IPR] / wc[0];
          sx[0] = wc[IPR] * exp_d(grav * dx / (2 * RdTv));
        }
        if (mt < NG) sx[1 + mt] = wc[0];
        if (mb < NG) sx[4 + mb] = wc[0];
      }
    }
    if (!hs) continue;
    wave_sync();
    if (p0 == ptop) pf_top = pf_next = sx[0];
    double mine = 0.0, above = 0.0;
    double step[OCT];
#pragma unroll
    for (int l = 0; l < OCT; ++l) step[l] = st[l];
#pragma unroll
    for (int l = OCT - 1; l >= 0; --l) {
      if (p0 + l >= L.n) continue;
      const double lowr = pf_next - step[l];
      if (l == l8) {
        mine = lowr;
        above = pf_next;
      }
      pf_next = lowr;
    }
    if (cell) {
      psf[pc + i * g.ps_i] = mine;
      psv[pc + i * g.ps_i] = log_mean(mine, above);
      if (i == ie) psf[pc + (ie + 1) * g.ps_i] = pf_top;
    }
  }
  if (!hs || !live || l8 > 1) return;
  // pressures of the ghosts, lane 0 below (psf(is-1..is-3)), lane 1 above
  // (psf(ie+2..ie+4)); a ghost's density is that of the mirrored cell at a
  // wall and of the last cell at an outflow side
  if (l8 == 0) {
    const double gb = (g.bc[0] == 0) ? -grav : grav;
    double cur = pf_next;
    for (int gh = 1; gh <= NG; ++gh) {
      const double rho = sx[4 + (g.bc[0] == 0 ? gh - 1 : 0)];
      const double lowr = cur - gb * rho * dx;
      psf[pc + (is - gh) * g.ps_i] = lowr;
      psv[pc + (is - gh) * g.ps_i] = log_mean(lowr, cur);
      cur = lowr;
    }
  } else {
    const double gt = (g.bc[1] == 0) ? -grav : grav;
    double cur = pf_top;
    for (int gh = 1; gh <= NG; ++gh) {
      const double rho = sx[1 + (g.bc[1] == 0 ? gh - 1 : 0)];
      const double high = cur + gt * rho * dx;
      psf[pc + (ie + gh + 1) * g.ps_i] = high;
      psv[pc + (ie + gh) * g.ps_i] = log_mean(cur, high);
      cur = high;
    }
  }
}

}  // namespace cg
