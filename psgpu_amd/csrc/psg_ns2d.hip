// 2D Navier-Stokes vorticity stepper: four RK4 stages without viscosity and
// an end-of-step Crank-Nicolson factor.
//   stage 1,2 (Step1):  Zs = dt N(Z0);  Z0 = Z + Zs/2
//   stage 3   (Step2):  Z3 = dt N(Z0);  Z0 = Z + Z3
//   final     (Step):   Z = [(1 - dt nu k^2/2) Z + (Z1 + 2 Z2 + 2 Z3 + dt N(Z0))/6] / (1 + dt nu k^2/2)
// with N = -i(kx FFT(u w) + ky FFT(v w)) and forcing NZKX -= A at (0,+-KF);
// off-mask modes of Z are zeroed at every stage.
// (2D_NavierStokes/src_RK4/src_gmres/cuda.cu:44-76, kernels.h:247-435)
// Each stage is two kernels: the shared x-pass, and a column pass (k2_col) that
// transforms the products forward in y, applies the stage update and, while the
// column is still on chip, transforms the next stage's (w, u, v) back in y.
#include "psg_launch.hpp"

namespace psg {

// RK4 stage update of one mode.  The stage input Z0 goes straight on to the
// inverse transforms, so only the state and one running sum of the increments
// are kept: (Z1 + 2 Z2) + 2 Z3, added in the order of the closing formula.
// acc is private to the run and stored like the columns that the pass works on,
// [m][ikx][iky].
template <int STAGE> struct Upd2D {
  cpx<double> *z, *acc;
  long nkt;
  const int8_t *L;
  double dt, v2, famp, kf;
  const double *dtm = nullptr;   // per-member steps (batched Newton flows); dt 0 leaves a member unchanged
  int *cnt = nullptr;            // step counter of a recorded base, advanced by the last stage
  struct In {
    cpx<double> z, a;
    bool on;
  };
  __device__ __forceinline__ In fetch(int m, long ik, long it) const {
    In q{{0.0, 0.0}, {0.0, 0.0}, L[ik] == 1};
    q.z = z[(long)m * nkt + ik];
    if constexpr (STAGE > 0) q.a = acc[(long)m * nkt + it];
    return q;
  }
  // N0 = FFT(v w)/NR, N1 = FFT(u w)/NR (the reference's NZK halves); returns Z0
  __device__ __forceinline__ cpx<double> apply(const In &q, int m, long ik, long it, double kx, double ky,
                                               cpx<double> N0, cpx<double> N1) const {
    if (!q.on) {
      if constexpr (STAGE == 3) z[(long)m * nkt + ik] = cpx<double>{0.0, 0.0};
      return cpx<double>{0.0, 0.0};
    }
    const double h = dtm ? dtm[m] : dt;
    double NZKX = kx * N1.y + ky * N0.y;
    double NZKY = -kx * N1.x - ky * N0.x;
    if (kx == 0.0 && fabs(ky) == kf) NZKX += famp;
    const double ZX = h * NZKX, ZY = h * NZKY;
    if constexpr (STAGE < 3) {
      cpx<double> *A = acc + (long)m * nkt + it;
      if constexpr (STAGE == 0) *A = cpx<double>{ZX, ZY};
      else *A = cpx<double>{q.a.x + 2 * ZX, q.a.y + 2 * ZY};
      const double f = STAGE == 2 ? 1.0 : 0.5;
      return cpx<double>{q.z.x + f * ZX, q.z.y + f * ZY};
    } else {
      const double wk = kx * kx + ky * ky;
      const double damp1 = 1 - 0.5 * h * v2 * wk;
      const double damp2 = 1. / (1 + 0.5 * h * v2 * wk);
      const cpx<double> r{damp2 * (damp1 * q.z.x + (q.a.x + ZX) / 6.), damp2 * (damp1 * q.z.y + (q.a.y + ZY) / 6.)};
      z[(long)m * nkt + ik] = r;
      return r;
    }
  }
  __device__ __forceinline__ void once() const {
    if constexpr (STAGE == 3) {
      if (cnt) *cnt = *cnt + 1;
    }
  }
};

// masked state L Z into the inverse transforms (setVelocity, kernels.h:112-147)
struct Load2D {
  const cpx<double> *z;
  long nkt;
  const int8_t *L;
  struct In {
    cpx<double> z;
  };
  __device__ __forceinline__ In fetch(int m, long ik, long) const {
    return In{L[ik] ? z[(long)m * nkt + ik] : cpx<double>{0.0, 0.0}};
  }
  __device__ __forceinline__ cpx<double> apply(const In &q, int, long, long, double, double, cpx<double>,
                                               cpx<double>) const {
    return q.z;
  }
  __device__ __forceinline__ void once() const {}
};

// masked N + F into out (nonlinear right-hand side, no viscous term)
struct Store2D {
  cpx<double> *out;
  long nkt;
  const int8_t *L;
  double famp, kf;
  struct In {
    double l;
  };
  __device__ __forceinline__ In fetch(int, long ik, long) const { return In{(double)L[ik]}; }
  __device__ __forceinline__ cpx<double> apply(const In &q, int m, long ik, long, double kx, double ky,
                                               cpx<double> N0, cpx<double> N1) const {
    double NZKX = kx * N1.y + ky * N0.y;
    double NZKY = -kx * N1.x - ky * N0.x;
    if (kx == 0.0 && fabs(ky) == kf) NZKX += famp;
    out[(long)m * nkt + ik] = cpx<double>{q.l * NZKX, q.l * NZKY};
    return cpx<double>{0.0, 0.0};
  }
  __device__ __forceinline__ void once() const {}
};

// Column pass: one kx column per block, three teams of N/8 threads.
//   FWD: teams 0 and 1 transform the products (v w) and (u w) forward in y;
//        the block's threads update the column's modes from them
//   INV: the updated column (or the loaded state) with the Hermitian fill of
//        kx = 0 (in place in the reference, 2D_NavierStokes/src_RK4/kernels.h:82-96)
//        and Biot-Savart (kernels.h:112-147): team f transforms field f of (w, u, v)
// A 2D launch has few columns, so its time is the latency of one block, not
// bandwidth.  With forward and inverse in one launch a stage takes two launches
// instead of three, with a team per field the transforms of a column run side
// by side, and everything a block reads is requested at its start.  At 512^2 in
// FP64 it takes 8.2 us where separate y-forward and y-inverse passes took 9.3
// and 7.6 us (a step 102 -> 69 us; at 128^2 89 -> 46 us), with 8 members 21.5 us.
// Single columns ask for column-major buffers: from row-major products the pass
// took 8.8 us, and 29.5 us with 8 members.
// NG independent groups (blockIdx.y: base, perturbation) take their own update
// and field range.
template <int N> struct Col2 {
  static constexpr int TP = N / EPT, THREADS = 3 * TP;
  // twiddles and three rows; the updated column lies in the third row, whose
  // team has no forward transform, where its FP64 modes fit (FP64 rows do: at
  // 512 points five blocks then share a CU instead of four)
  template <typename P> static constexpr bool alias() { return sizeof(P) == 8; }
  template <typename P> static constexpr size_t lds() {
    return (size_t)4 * N * sizeof(cpx<P>) + (alias<P>() ? 0 : (size_t)(2 * (N / 3) + 1) * sizeof(cpx<double>));
  }
};
template <typename P, int N, bool FWD, bool INV, class UPD, int NG>
__global__ void __launch_bounds__(Col2<N>::THREADS)
k2_col(const cpx<P> *__restrict__ in, long in_ms, cpx<P> *__restrict__ out, long out_ms, Grid g,
       const cpx<P> *__restrict__ tw, UPD upd0, UPD upd1) {
  constexpr int TP = Col2<N>::TP, NT = Col2<N>::THREADS;
  constexpr int NI = (2 * (N / 3) + 1 + NT - 1) / NT;   // modes of the column per thread
  constexpr bool WAVE = TP <= 64;
  constexpr int SW = row_swizzle<EPT>();
  PSG_TWIDDLES_REQUEST(P, N, EPT, NT);
  const int team = threadIdx.x / TP, j = threadIdx.x % TP;
  const TileId tid = xcd_tile();
  const int ikx = tid.x, grp = NG > 1 ? tid.y : 0, m = tid.z;
  const UPD upd = NG > 1 && grp ? upd1 : upd0;
  const double kx = (double)ikx * g.alpha;
  cpx<P> *row = lds + team * N;
  constexpr bool ALIAS = Col2<N>::template alias<P>();
  cpx<double> *col = reinterpret_cast<cpx<double> *>(lds + (ALIAS ? 2 : 3) * N);
  cpx<P> v[EPT];
  if constexpr (FWD) {
    const cpx<P> *src = in + (long)m * in_ms + (long)(grp * 2 + (team < 2 ? team : 0)) * g.ysz + YCol::col(g, ikx);
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) v[mm] = team < 2 ? src[j + TP * mm] : cpx<P>{0, 0};
  }
  typename UPD::In q[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int iky = threadIdx.x + i * NT, iy = iky < g.ikty ? iky : 0;
    q[i] = upd.fetch(m, (long)iy * g.iktx + ikx, (long)ikx * g.ikty + iy);
  }
  PSG_TWIDDLES_READY(P);
  if constexpr (FWD) {
    fft_pencil<P, N, EPT, false, WAVE, SW>(v, row, j, 1, 0, tw);
    team_sync<WAVE>();
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) row[j + TP * mm] = v[mm];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int iky = threadIdx.x + i * NT, ky = iky - g.kty;
    if (iky < g.ikty) {
      cpx<double> n0{0.0, 0.0}, n1{0.0, 0.0};
      if constexpr (FWD) {
        const int p = ky < 0 ? ky + N : ky;
        const cpx<double> a = up(lds[p]), b = up(lds[N + p]);
        n0 = cpx<double>{a.x * g.inr, a.y * g.inr};
        n1 = cpx<double>{b.x * g.inr, b.y * g.inr};
      }
      const cpx<double> w = upd.apply(q[i], m, (long)iky * g.iktx + ikx, (long)ikx * g.ikty + iky, kx, (double)ky, n0, n1);
      if constexpr (INV) col[iky] = w;
    }
  }
  if (FWD && tid.x == 0 && tid.y == 0 && tid.z == 0 && threadIdx.x == 0) upd.once();
  if constexpr (INV) {
    __syncthreads();
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) {
      const int ky = wrapk(j + TP * mm, g.ny, g.kty);
      cpx<double> w{0.0, 0.0};
      if (ky != PSG_NOK) {
        const bool mirror = ikx == 0 && ky < 0;
        w = col[(mirror ? -ky : ky) + g.kty];
        if (mirror) w.y = -w.y;
        if (team > 0) {
          const double kyd = (double)ky, wk = kx * kx + kyd * kyd;
          const double wki = 1.0 / (wk > 0.001 ? wk : 0.001);
          w = team == 1 ? cpx<double>{-kyd * w.y * wki, kyd * w.x * wki} : cpx<double>{kx * w.y * wki, -kx * w.x * wki};
        }
      }
      v[mm] = to<P>(w);
    }
    if constexpr (ALIAS) __syncthreads();
    fft_pencil<P, N, EPT, true, WAVE, SW>(v, row, j, 1, 0, tw);
    cpx<P> *o = out + (long)m * out_ms + (long)(grp * 3 + team) * g.ysz + YCol::col(g, ikx);
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) o[j + TP * mm] = v[mm];
  }
}

// members (and NG groups) of one column pass; in: 2 NG fields, out: 3 NG fields a member
template <typename P, bool FWD, bool INV, class UPD, int NG = 1>
static int launch_col2(Ctx *c, const cpx<P> *in, cpx<P> *out, int nm, UPD u0, UPD u1) {
  const Grid &g = c->g;
  PSG_DISPATCH_N(g.ny, {
    const size_t lds = Col2<N>::template lds<P>();
    auto k = k2_col<P, N, FWD, INV, UPD, NG>;
    PSG_HIP(lds_attr(k, lds));
    hipLaunchKernelGGL(k, dim3(g.iktx, NG, nm), dim3(Col2<N>::THREADS), lds, c->stream, in, 2 * NG * g.ysz, out,
                       3 * NG * g.ysz, g, twp<P>(c, 1), u0, u1);
  });
  PSG_HIP(hipGetLastError());
  return 0;
}
template <typename P, bool FWD, bool INV, class UPD>
static int launch_col2(Ctx *c, const cpx<P> *in, cpx<P> *out, int nm, UPD u) {
  return launch_col2<P, FWD, INV, UPD, 1>(c, in, out, nm, u, u);
}

template <typename P, int FI, int FO, class PROD>
static int launch_xpass2(Ctx *c, const cpx<P> *in, cpx<P> *out, long nrow_m, int nm, PROD prod) {
  const Grid &g = c->g;
  PSG_DISPATCH_N(g.nx, {
    if (g.iktx != xband<N>()) {
      set_error("x-pass: IKTX %d is not NX/3+1", g.iktx);
      return PSG_EINVAL;
    }
    long nrows = nrow_m * nm;
    if (nrows >= (1L << 31)) {
      set_error("x-pass: %ld rows exceed the 32-bit row index", nrows);
      return PSG_EINVAL;
    }
    // few rows: one row per block, its field pairs transformed side by side.  Several rows
    // a block gather whole pieces of lines, but are fewer blocks with a longer chain each:
    // they win from 2048 rows on at every length (from 1024 rows on also at 1024 points)
    // and lose on the few rows of a single small grid.  Us, one row a block and several:
    //   step, FP64, one context (three at a time):
    //      64 points   512 rows 40.4, 40.8 (15.8, 15.9)   2048 rows 47.4, 42.2 (21.1, 18.1)
    //     128 points   512 rows 44.2, 49.1 (19.1, 20.7)   2048 rows 59.1, 51.1 (29.6, 23.3)
    //     256 points  1024 rows 64.8, 62.9 (30.3, 26.7)   2048 rows 78.4, 62.5 (47.7, 34.9)
    //     512 points   512 rows 68.9, 65.6 (31.8, 28.1)   1024 rows 97.6, 83.8 (50.7, 36.4)
    //    1024 points   256 rows 75.9, 77.4 (40.6, 32.6)   1024 rows  190,  154 ( 109, 80.2)
    //   the same in FP32: 16 points 2048 rows 44.6, 41.7 (15.9, 16.1), 64 points 2048 rows
    //     40.7, 37.6 (17.1, 15.5), 1024 points 256 rows 61.6, 68.2 (28.1, 28.8), 1024 rows
    //     149, 112 (84.9, 54.0)
    //   tangent of 20 steps (6 fields in, 4 out), one context, FP64 and FP32: 64 points 2048
    //     rows 1288, 1293 and 1077, 1098; 128 points 2048 rows 1747, 1661 and 1398, 1288;
    //     512^2 2364, 2295 and 1875, 1900; 1024^2 8656, 6033 and 5849, 4137
    if (nrows < (N >= 1024 ? 1024 : 2048)) {
      constexpr int NT = xsplit_teams<FI, FO>() * Row<N>::TPX;
      static_assert(NT <= 1024, "split-row x-pass block size");
      const size_t lds = xsplit_lds<P, N, FI, FO>();
      auto k = k_xpass_split<P, N, FI, FO, PROD>;
      PSG_HIP(lds_attr(k, lds));
      hipLaunchKernelGGL(k, dim3((unsigned)nrows), dim3(NT), lds, c->stream, in, out, nrow_m, nrows, g,
                         twp<P>(c, 0), prod);
    } else {
      // rows per block: 256 threads, 512 for the long rows in FP32 (128 rows at 16 points, 4 at
      // 512 and 2 at 1024 in FP64, 8 and 4 in FP32).  They gather pieces of 128 bytes and more
      // in FP64 up to 256 points, of 64 at 512 and 32 at 1024.  Twice the rows leaves one or two
      // blocks a CU, whose barriers then stand alone (FP64 us, this and twice: 512^2 x 8 23.6,
      // 27.3; 1024^2 x 4 48.1, 64.3); half of them halves the pieces (FP32 512^2 x 8 15.3,
      // 15.8; 1024^2 x 2 20.3, 21.7)
      constexpr int TE = Row<N>::TEAMS * (sizeof(P) == 4 && N >= 512 ? 2 : 1);
      constexpr size_t lds = xcol_lds<P, N, TE>();
      static_assert(TE * Row<N>::TPX <= 1024 && lds <= 160 * 1024, "column x-pass block size");
      auto k = k_xpass_col<P, N, TE, FI, FO, PROD>;
      PSG_HIP(lds_attr(k, lds));
      hipLaunchKernelGGL(k, dim3((unsigned)((nrows + TE - 1) / TE)), dim3(TE * Row<N>::TPX), lds, c->stream, in, out,
                         nrow_m, nrows, g, twp<P>(c, 0), prod);
    }
  });
  PSG_HIP(hipGetLastError());
  return 0;
}

#define PSG_TRY2(x)     \
  do {                  \
    int r_ = (x);       \
    if (r_) return r_;  \
  } while (0)

static double famp2(const Ctx *c) { return c->cfg.force == PSG_FORCE_NONE ? 0.0 : c->cfg.ampfor; }
// stage update of the context's state; of the perturbation (no forcing)
template <int S> static Upd2D<S> upd2(const Ctx *c, int *cnt = nullptr) {
  return Upd2D<S>{c->state, c->rh, c->g.nkt, c->mask, c->cfg.dt, c->cfg.v2, famp2(c), c->cfg.kf, c->dtm_on ? c->dtm : nullptr,
                  cnt};
}
template <int S> static Upd2D<S> pert2(const Ctx *c, int *cnt = nullptr) {
  return Upd2D<S>{c->tl_state, c->tl_rh, c->g.nkt, c->mask, c->cfg.dt, c->cfg.v2, 0.0, c->cfg.kf, nullptr, cnt};
}
static Load2D load2(const Ctx *c, const cpx<double> *z) { return Load2D{z, c->g.nkt, c->mask}; }

// the column pass that ends a stage; a run's last stage (end) only updates the state
template <typename P, int S, int NG = 1>
static int col2_stage(Ctx *c, const cpx<P> *in, cpx<P> *out, int nm, Upd2D<S> u0, Upd2D<S> u1, bool end) {
  if constexpr (S == 3) {
    if (end) return launch_col2<P, true, false, Upd2D<S>, NG>(c, in, out, nm, u0, u1);
  }
  return launch_col2<P, true, true, Upd2D<S>, NG>(c, in, out, nm, u0, u1);
}

// one stage from the y-space fields in B, which it leaves ready for the next
template <typename P, int S> static int stage2(Ctx *c, Upd2D<S> upd, int nm, bool end) {
  const Grid &g = c->g;
  cpx<P> *B = (cpx<P> *)c->bufB, *Cb = (cpx<P> *)c->bufC;
  const long Y = (long)g.iktx * g.ny;
  const size_t b = sizeof(cpx<P>);
  prof_begin(c, "xpass2", (long)(5 * Y * b) * nm);
  PSG_TRY2((launch_xpass2<P, 3, 2>(c, B, Cb, g.ny, nm, Prod2D<P>{})));
  prof_end(c);
  prof_begin(c, "ycol2_update", (long)(5 * Y * b + 3 * g.nkt * 16) * nm);
  PSG_TRY2((col2_stage<P, S>(c, Cb, B, nm, upd, upd, end)));
  prof_end(c);
  return 0;
}

// first, last: the first and the last steps of a run.  It starts from the masked state,
// every later stage finds its fields in B, and its last stage makes none (runs of one
// step, 1024^2 x 4 in three contexts: 389 us with the unused transforms, 367 without)
template <typename P> static int run2_t(Ctx *c, int nsteps, bool first, bool last) {
  if (first) PSG_TRY2((launch_col2<P, false, true>(c, (const cpx<P> *)nullptr, (cpx<P> *)c->bufB, c->batch, load2(c, c->state))));
  for (int nt = 0; nt < nsteps; nt++) {
    const bool end = last && nt == nsteps - 1;
    PSG_TRY2((stage2<P>(c, upd2<0>(c), c->batch, end)));
    PSG_TRY2((stage2<P>(c, upd2<1>(c), c->batch, end)));
    PSG_TRY2((stage2<P>(c, upd2<2>(c), c->batch, end)));
    PSG_TRY2((stage2<P>(c, upd2<3>(c), c->batch, end)));
  }
  return 0;
}

int ns2d_run(Ctx *c, int nsteps, bool first, bool last) {
  return c->cfg.precision == PSG_FP32BULK ? run2_t<float>(c, nsteps, first, last) : run2_t<double>(c, nsteps, first, last);
}

template <typename P> static int nonlin2_t(Ctx *c, const cpx<double> *in, cpx<double> *out) {
  cpx<P> *B = (cpx<P> *)c->bufB, *Cb = (cpx<P> *)c->bufC;
  PSG_TRY2((launch_col2<P, false, true>(c, (const cpx<P> *)nullptr, B, 1, load2(c, in))));
  PSG_TRY2((launch_xpass2<P, 3, 2>(c, B, Cb, c->g.ny, 1, Prod2D<P>{})));
  return launch_col2<P, true, false>(c, Cb, (cpx<P> *)nullptr, 1, Store2D{out, c->g.nkt, c->mask, famp2(c), c->cfg.kf});
}

int ns2d_nonlin(Ctx *c, int, const cpx<double> *in_dev, cpx<double> *out_dev) {
  return c->cfg.precision == PSG_FP32BULK ? nonlin2_t<float>(c, in_dev, out_dev)
                                          : nonlin2_t<double>(c, in_dev, out_dev);
}

template <typename P, int N, int TE>
__global__ void __launch_bounds__(TE *(N / EPT))
k2_xphys(const cpx<P> *__restrict__ in, double *__restrict__ out, long nrow, Grid g, const cpx<P> *__restrict__ tw) {
  PSG_TWIDDLES_REQUEST(P, N, EPT, TE *(N / EPT));
  constexpr int TPX = N / EPT;
  const int team = threadIdx.x / TPX, j = threadIdx.x % TPX;
  const long row = (long)blockIdx.x * TE + team;
  const bool valid = row < nrow;
  const int f = blockIdx.y;
  const cpx<P> *ra = in + (long)f * g.ysz + YCol::row(g, valid ? (int)row : 0, 0);
  cpx<P> v[EPT];
#pragma unroll
  for (int mm = 0; mm < EPT; mm++) {
    const int k = j + TPX * mm;
    cpx<P> a{0, 0};
    if (valid) {
      if (k < g.iktx) { a = ra[YCol::col(g, k)]; if (k == 0) a.y = 0; }
      else if (k > N - g.iktx) { a = ra[YCol::col(g, N - k)]; a.y = -a.y; }
    }
    v[mm] = a;
  }
  PSG_TWIDDLES_READY(P);
  fft_pencil<P, N, EPT, true>(v, lds + team * N, j, 1, 0, tw);
  if (valid) {
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) out[((long)f * nrow + row) * N + j + TPX * mm] = (double)v[mm].x;
  }
}

template <typename P> static int physical2_t(Ctx *c, int member, double *out) {
  const Grid &g = c->g;
  cpx<P> *B = (cpx<P> *)c->bufB;
  // physical fields of the masked state (w, u, v)
  PSG_TRY2((launch_col2<P, false, true>(c, (const cpx<P> *)nullptr, B, 1, load2(c, c->state + (long)member * g.nkt))));
  long nrow = g.ny;
  PSG_DISPATCH_N(g.nx, {
    constexpr int TE = Row<N>::TEAMS;
    dim3 grid((unsigned)((nrow + TE - 1) / TE), 3);
    size_t lds = (size_t)(N * TE + N) * sizeof(cpx<P>);
    auto k = k2_xphys<P, N, TE>;
    PSG_HIP(lds_attr(k, lds));
    hipLaunchKernelGGL(k, grid, dim3(Row<N>::THREADS), lds, c->stream, B, out, nrow, g, twp<P>(c, 0));
  });
  PSG_HIP(hipGetLastError());
  return 0;
}

int ns2d_physical(Ctx *c, int member, double *out_dev) {
  return c->cfg.precision == PSG_FP32BULK ? physical2_t<float>(c, member, out_dev)
                                          : physical2_t<double>(c, member, out_dev);
}

// ------------------------------------------------------------------ tangent linear
// Base and perturbation advance together through the same RK4/CN stages:
// the perturbation stage increments use the linearised nonlinear term
// dN = -i(kx FFT(du w + u dw) + ky FFT(dv w + v dw)) (no forcing) with the
// same damping factors and masks as the base update.  The x-pass mixes them;
// the column pass takes them as two independent groups.
template <typename P, int S> static int stage2_tl(Ctx *c, bool end) {
  cpx<P> *B = (cpx<P> *)c->tl_bufB, *Cb = (cpx<P> *)c->tl_bufC;
  Upd2D<S> base = upd2<S>(c);
  base.dtm = nullptr;
  PSG_TRY2((launch_xpass2<P, 6, 4>(c, B, Cb, c->g.ny, c->batch, Prod2DTL<P>{})));
  return col2_stage<P, S, 2>(c, Cb, B, c->batch, base, pert2<S>(c), end);
}

template <typename P> static int run2tl_t(Ctx *c, int nsteps, bool first, bool last) {
  if (first)
    PSG_TRY2((launch_col2<P, false, true, Load2D, 2>(c, nullptr, (cpx<P> *)c->tl_bufB, c->batch, load2(c, c->state),
                                                     load2(c, c->tl_state))));
  for (int nt = 0; nt < nsteps; nt++) {
    const bool end = last && nt == nsteps - 1;
    PSG_TRY2((stage2_tl<P, 0>(c, end)));
    PSG_TRY2((stage2_tl<P, 1>(c, end)));
    PSG_TRY2((stage2_tl<P, 2>(c, end)));
    PSG_TRY2((stage2_tl<P, 3>(c, end)));
  }
  return 0;
}

int ns2d_tl_run(Ctx *c, int nsteps, bool first, bool last) {
  return (c->cfg.precision == PSG_FP32BULK || c->tl_fp32) ? run2tl_t<float>(c, nsteps, first, last)
                                                          : run2tl_t<double>(c, nsteps, first, last);
}

// ------------------------------------------------------------------ recorded base
// A base flow whose x-pass uses Prod2DRec stores the physical (w, u, v) of
// every stage at slot 4*step + stage, step being the device counter that the
// last stage's column pass advances.  The perturbation-only flow
// (Prod2DTLRec) reads them back instead of transforming the base
// again, so one tangent-linear step costs the transforms of a plain step.
// Past the record's last slot nothing is stored and zeros are read; the host
// sizes the record so that this never happens.
__device__ __forceinline__ long rec_offset(const int *cnt, int stage, long slots, long plane) {
  const long slot = 4L * (long)(*cnt) + stage;
  return slot < slots ? slot * 3 * plane : -1;
}

template <typename P, typename RP> struct Prod2DRec {
  static constexpr bool ROW = true;
  RP *rec;
  const int *cnt;
  int stage;
  long slots;
  int nx, ny;
  struct Bound {
    RP *p;
    long plane;
    bool on;
    // in: w, u, v; out: (v w, u w) as Prod2D
    __device__ __forceinline__ void operator()(int n, const P *in, P *out) const {
      if (on) {
        p[n] = (RP)in[0];
        p[plane + n] = (RP)in[1];
        p[2 * plane + n] = (RP)in[2];
      }
      out[0] = in[2] * in[0];
      out[1] = in[1] * in[0];
    }
  };
  // every team forms the products; team 0 alone stores the row
  __device__ __forceinline__ Bound bind(unsigned, unsigned row, int team) const {
    const long plane = (long)ny * nx;
    const long o = rec_offset(cnt, stage, slots, plane);
    return Bound{o >= 0 ? rec + o + (long)row * nx : rec, plane, o >= 0 && team == 0};
  }
};

template <typename P, typename RP> struct Prod2DTLRec {
  static constexpr bool ROW = true;
  const RP *rec;
  const int *cnt;
  int stage;
  long slots;
  int nx, ny;
  struct Bound {
    const RP *p;
    long plane;
    bool on;
    // in: dw, du, dv; out: (dv w + v dw, du w + u dw) about the recorded (w, u, v)
    __device__ __forceinline__ void operator()(int n, const P *in, P *out) const {
      P w = 0, u = 0, v = 0;
      if (on) {
        w = (P)p[n];
        u = (P)p[plane + n];
        v = (P)p[2 * plane + n];
      }
      out[0] = in[2] * w + v * in[0];
      out[1] = in[1] * w + u * in[0];
    }
  };
  // only team 0's output pair is stored: the other team reads nothing
  __device__ __forceinline__ Bound bind(unsigned, unsigned row, int team) const {
    const long plane = (long)ny * nx;
    const long o = rec_offset(cnt, stage, slots, plane);
    return Bound{o >= 0 ? rec + o + (long)row * nx : rec, plane, o >= 0 && team == 0};
  }
};

__global__ void k2_zero_int(int *p) { *p = 0; }

// the split-row x-pass alone (the record is indexed by row)
template <typename P, int FI, int FO, class PROD>
static int launch_xpass2_split(Ctx *c, const cpx<P> *in, cpx<P> *out, PROD prod) {
  const Grid &g = c->g;
  PSG_DISPATCH_N(g.nx, {
    if (g.iktx != xband<N>()) {
      set_error("x-pass: IKTX %d is not NX/3+1", g.iktx);
      return PSG_EINVAL;
    }
    if (g.ny >= 2048) {
      set_error("recorded base: %d rows exceed the split-row x-pass", g.ny);
      return PSG_EINVAL;
    }
    constexpr int NT = xsplit_teams<FI, FO>() * Row<N>::TPX;
    const size_t lds = xsplit_lds<P, N, FI, FO>();
    auto k = k_xpass_split<P, N, FI, FO, PROD>;
    PSG_HIP(lds_attr(k, lds));
    hipLaunchKernelGGL(k, dim3((unsigned)g.ny), dim3(NT), lds, c->stream, in, out, (long)g.ny, (long)g.ny, g,
                       twp<P>(c, 0), prod);
  });
  PSG_HIP(hipGetLastError());
  return 0;
}

template <typename P, typename RP> static int run2rec_t(Ctx *c, int nsteps, bool first, bool last) {
  const Grid &g = c->g;
  if (c->batch != 1 || !c->rec || !c->rec_cnt) {
    set_error("recorded base: one member and an allocated record only");
    return PSG_EINVAL;
  }
  cpx<P> *B = (cpx<P> *)c->bufB, *Cb = (cpx<P> *)c->bufC;
  if (first) PSG_TRY2((launch_col2<P, false, true>(c, (const cpx<P> *)nullptr, B, 1, load2(c, c->state))));
  for (int nt = 0; nt < nsteps; nt++) {
    const bool end = last && nt == nsteps - 1;
#define PSG_REC_STAGE(S)                                                           \
    {                                                                              \
      Prod2DRec<P, RP> pr{(RP *)c->rec, c->rec_cnt, S, c->rec_slots, g.nx, g.ny};  \
      PSG_TRY2((launch_xpass2_split<P, 3, 2>(c, B, Cb, pr)));                      \
      const Upd2D<S> u = upd2<S>(c, c->rec_cnt);                                   \
      PSG_TRY2((col2_stage<P, S>(c, Cb, B, 1, u, u, end)));                        \
    }
    PSG_REC_STAGE(0) PSG_REC_STAGE(1) PSG_REC_STAGE(2) PSG_REC_STAGE(3)
#undef PSG_REC_STAGE
  }
  return 0;
}

template <typename P> static int run2tlrec_t(Ctx *c, int nsteps, bool first, bool last) {
  const Grid &g = c->g;
  if (c->batch != 1 || !c->rec || !c->rec_cnt || c->rec_p != (int)sizeof(P)) {
    set_error("recorded tangent linear: one member and a record of the pass precision only");
    return PSG_EINVAL;
  }
  cpx<P> *B = (cpx<P> *)c->tl_bufB, *Cb = (cpx<P> *)c->tl_bufC;
  if (first) PSG_TRY2((launch_col2<P, false, true>(c, (const cpx<P> *)nullptr, B, 1, load2(c, c->tl_state))));
  for (int nt = 0; nt < nsteps; nt++) {
    const bool end = last && nt == nsteps - 1;
#define PSG_TLR_STAGE(S)                                                                \
    {                                                                                   \
      Prod2DTLRec<P, P> pr{(const P *)c->rec, c->rec_cnt, S, c->rec_slots, g.nx, g.ny}; \
      PSG_TRY2((launch_xpass2_split<P, 3, 2>(c, B, Cb, pr)));                           \
      const Upd2D<S> u = pert2<S>(c, c->rec_cnt);                                       \
      PSG_TRY2((col2_stage<P, S>(c, Cb, B, 1, u, u, end)));                             \
    }
    PSG_TLR_STAGE(0) PSG_TLR_STAGE(1) PSG_TLR_STAGE(2) PSG_TLR_STAGE(3)
#undef PSG_TLR_STAGE
  }
  return 0;
}

int ns2d_rec_run(Ctx *c, int nsteps, bool first, bool last) {
  if (c->cfg.precision == PSG_FP32BULK) {
    if (c->rec_p != 4) { set_error("recorded base: an FP32-bulk context records FP32"); return PSG_EINVAL; }
    return run2rec_t<float, float>(c, nsteps, first, last);
  }
  return c->rec_p == 4 ? run2rec_t<double, float>(c, nsteps, first, last) : run2rec_t<double, double>(c, nsteps, first, last);
}

int ns2d_tlrec_run(Ctx *c, int nsteps, bool first, bool last) {
  return c->rec_p == 4 ? run2tlrec_t<float>(c, nsteps, first, last) : run2tlrec_t<double>(c, nsteps, first, last);
}

int ns2d_rec_reset(Ctx *c) {
  hipLaunchKernelGGL(k2_zero_int, dim3(1), dim3(1), 0, c->stream, c->rec_cnt);
  PSG_HIP(hipGetLastError());
  return 0;
}

int ns2d_init(Ctx *c) {
  const Grid &g = c->g;
  size_t b = c->cfg.precision == PSG_FP32BULK ? sizeof(cpx<float>) : sizeof(cpx<double>);
  c->szB = (size_t)3 * g.ysz * c->batch * b;
  c->szC = (size_t)2 * g.ysz * c->batch * b;
  PSG_HIP(hipMalloc(&c->bufB, c->szB));
  PSG_HIP(hipMalloc(&c->bufC, c->szC));
  PSG_HIP(hipMalloc(&c->rh, sizeof(cpx<double>) * g.nkt * c->batch));
  PSG_HIP(hipMemsetAsync(c->rh, 0, sizeof(cpx<double>) * g.nkt * c->batch, c->stream));
  return 0;
}

}  // namespace psg
