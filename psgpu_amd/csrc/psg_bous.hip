// 3D Boussinesq stepper: RK4 with per-stage Crank-Nicolson factors, buoyancy
// with gravity tilted by theta (radians), Leray projection after each step.
//   stage 1,2 (Step1): X_s = dt C(Z0);  Z0 = d_{1/4} (X^n + dt/2 C)
//   stage 3   (Step2): X_3 = dt C(Z0);  Z0 = d_{1/2} (X^n + dt C)
//   final     (Step) : X^{n+1} = L [(1 - dt nu k^2/2) X^n + (X_1 + dt C)/6 + (X_2 + X_3)/3] / (1 + dt nu k^2/2)
//                      Z0 = X^{n+1} (before projection); w^{n+1} <- w - k (k.w)/|k|^2
// with d_q = (1 - q dt nu k^2)/(1 + q dt nu k^2) (nu/Sc for the buoyancy),
//   C_w   = L [curl(u x w) - Ri (buoyancy torque with sin/cos theta)] + F,
//   C_rho = -L [FFT(u.grad rho) - v cos theta - w sin theta].
// (3D_Boussinesq/src/cuda.cu:65-101, kernels.h:331-621; RHS for Newton kernels.h:624-692)
// One right-hand side: pass 1 from the stage state (vorticity, Biot-Savart
// velocity and i k rho), y-inverse of 9 fields, x-pass product (-(u x w),
// u.grad rho), y-forward of 4 fields, z-forward ending in the stage update.
#include "psg_ns3d.hpp"

namespace psg {

// The stage input Z0 and the increments X_s live in z runs (LayRun): a z-pass
// block then reads and writes them as one run per (tile, ky), as the
// Navier-Stokes working copy (LayW) is; the state stays in the reference order.
typedef LayRun<4> LayZ0;
typedef LayRun<12> LayXS;

// pass 1: outputs w(3), u(3), i kx rho, i ky rho, i kz rho; with nout = 7 the
// seventh field is rho itself (physical-space dumps, 3D_Boussinesq/src/out_low.h:79-110)
// LAY: layout of st (its field stride fs); the mask is in the reference order.
// Gather- and register-bound: vorticity becomes velocity in its own registers,
// in FP64 until the transforms, and every index is a constant, so that with whole
// pencils of up to 512 points nothing lies in scratch memory and two waves share a
// SIMD (split fields in FP64 keep up to 52 bytes there, 1024 points 232 to 472; an earlier
// form, with the field loop rolled, indexed its registers at run time: 400 bytes
// of scratch a lane and one wave per SIMD; capped for three waves this one spills
// and is slower again).  512^3 FP64 2.11 -> 1.54 ms, 256^3 0.289 -> 0.195 ms, in
// FP32 1.91 -> 1.34 and 0.230 -> 0.165 ms.
// SPLIT: blockIdx.z also picks vorticity, velocity or density, for grids whose
// few blocks would run their eight transforms one after the other.
template <typename P, int N, int T, class LAY, bool SPLIT>
__global__ void __launch_bounds__(T *(N / EPT)) PSG_WAVES_PER_EU((N <= 512 ? 2 : 1))
k_zinv_bous(const cpx<double> *__restrict__ st, long st_ms, long fs, cpx<P> *__restrict__ out, long out_ms, Grid g,
            const cpx<P> *__restrict__ tw, const int8_t *__restrict__ mask, int umask, int nout) {
  PSG_TWIDDLES_REQUEST(P, N, EPT, T *(N / EPT));
  constexpr int TP = N / EPT;
  const int col = threadIdx.x % T, j = threadIdx.x / T;
  const TileId tid = xcd_tile();
  const int ikx = tid.x * T + col, iky = tid.y, m = SPLIT ? tid.z / 3 : tid.z, part = SPLIT ? tid.z % 3 : -1;
  const bool vort = !SPLIT || part == 0, vel = !SPLIT || part == 1, dens = !SPLIT || part == 2;
  const bool valid = ikx < g.iktx;
  const int ky = iky - g.kty;
  const double kx = (double)ikx * g.alpha, kyd = (double)ky;
  const cpx<double> *s0 = st + (long)m * st_ms;
  cpx<P> *o = out + (long)m * out_ms;
  cpx<double> w[3][EPT];
#pragma unroll
  for (int mm = 0; mm < EPT; mm++) {
    const int kz = valid ? wrapk(j + TP * mm, g.nz, g.ktz) : PSG_NOK;
    const FillIdx q = fill_index<LAY>(g, ikx, iky, ky, kz);
#pragma unroll
    for (int f = 0; f < 3; f++) w[f][mm] = SPLIT && part == 2 ? (f == 0 ? ld_fill(s0 + 3 * fs, q) : cpx<double>{0, 0}) : ld_fill(s0 + f * fs, q);
  }
  PSG_TWIDDLES_READY(P);
  // transform one field and store it into output f
  auto field = [&](cpx<P>(&v)[EPT], int f) {
    fft_pencil<P, N, EPT, true>(v, lds, fresh(j), T, col, tw);
    const int jo = fresh(j);
    if (valid) {
#pragma unroll
      for (int mm = 0; mm < EPT; mm++)
        st_pass<NT<P, PASS_ZINV>::st>(&o[(long)f * g.zsz + zoff<P>(g, ikx, iky, jo + TP * mm)], v[mm]);
    }
  };
  if (vort) {
#pragma unroll
    for (int f = 0; f < 3; f++) {
      cpx<P> v[EPT];
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) v[mm] = to<P>(w[f][mm]);
      field(v, f);
    }
  }
  if (vel) {
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) {
      const int kz = valid ? wrapk(fresh(j) + TP * mm, g.nz, g.ktz) : PSG_NOK;
      const double kzd = kz == PSG_NOK ? 0.0 : (double)kz;
      const double wk = kx * kx + kyd * kyd + kzd * kzd;
      double wki = 1.0;
      if (umask) {
        const FillIdx q = fill_index<LAY>(g, ikx, iky, ky, kz);
        if (q.idx >= 0) wki = (double)mask[q.tidx];
      }
      wki = wki / (wk > 0.001 ? wk : 0.001);
      cpx<double> u, vv, ww;
      biot_savart(kx, kyd, kzd, w[0][mm], w[1][mm], w[2][mm], wki, u, vv, ww);
      w[0][mm] = u;
      w[1][mm] = vv;
      w[2][mm] = ww;
      PSG_COMPILER_FENCE();
    }
#pragma unroll
    for (int f = 0; f < 3; f++) {
      cpx<P> v[EPT];
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) v[mm] = to<P>(w[f][mm]);
      // the density is requested before the last velocity transform, into
      // registers that the vorticity has left
      if (!SPLIT && f == 1) {
#pragma unroll
        for (int mm = 0; mm < EPT; mm++) {
          const int kz = valid ? wrapk(fresh(j) + TP * mm, g.nz, g.ktz) : PSG_NOK;
          w[0][mm] = ld_fill(s0 + 3 * fs, fill_index<LAY>(g, ikx, iky, ky, kz));
        }
      }
      field(v, 3 + f);
    }
  }
  if (!dens) return;
  cpx<P> v[EPT];
#pragma unroll
  for (int mm = 0; mm < EPT; mm++) v[mm] = to<P>(w[0][mm]);
  if (nout == 7) {
    field(v, 6);
    return;
  }
  // setFFK: i kx rho and i ky rho are one transform of rho scaled by constants
  // of the pencil, so nine outputs take eight transforms
  fft_pencil<P, N, EPT, true>(v, lds, fresh(j), T, col, tw);
  if (valid) {
    const int jo = fresh(j);
    const P px = (P)kx, py = (P)kyd;
    cpx<P> *o6 = o + 6 * g.zsz, *o7 = o6 + g.zsz;
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) {
      const long at = zoff<P>(g, ikx, iky, jo + TP * mm);
      st_pass<NT<P, PASS_ZINV>::st>(&o6[at], cpx<P>{-px * v[mm].y, px * v[mm].x});
      st_pass<NT<P, PASS_ZINV>::st>(&o7[at], cpx<P>{-py * v[mm].y, py * v[mm].x});
    }
  }
#pragma unroll
  for (int mm = 0; mm < EPT; mm++) {
    const int kz = wrapk(fresh(j) + TP * mm, g.nz, g.ktz);
    const double kzd = kz == PSG_NOK ? 0.0 : (double)kz;
    v[mm] = to<P>(cpx<double>{-kzd * w[0][mm].y, kzd * w[0][mm].x});   // i kz rho
  }
  field(v, 8);
}

// x-pass product: (U,V,W) <- -(u x w), rx <- u . grad rho  (3D_Boussinesq/src/kernels.h:298-328)
template <typename P> struct ProdBous {
  __device__ __forceinline__ void operator()(const P *in, P *out) const {
    const P tx = in[0], te = in[1], tz = in[2], tu = in[3], tv = in[4], tw = in[5];
    out[0] = -(tv * tz - tw * te);
    out[1] = -(tw * tx - tu * tz);
    out[2] = -(tu * te - tv * tx);
    out[3] = tu * in[6] + tv * in[7] + tw * in[8];
  }
};

struct BousPar {
  double dt, v2, sc, ri, sinth, costh, kf, ampfor;
};

// C (8 reals: xi, eta, zeta, rho as re/im) from the transformed products and the stage state
__device__ __forceinline__ void bous_rhs(const BousPar &p, double kx, double ky, double kz, double LC,
                                         const cpx<double> (&N)[4], cpx<double> x0, cpx<double> e0,
                                         cpx<double> z0, cpx<double> r0, double *C) {
  const double UKX = N[0].x, UKY = N[0].y, VKX = N[1].x, VKY = N[1].y, WKX = N[2].x, WKY = N[2].y;
  const double wk = kx * kx + ky * ky + kz * kz;
  const double wki = 1.0 / (wk > 0.001 ? wk : 0.001);
  const double rXR = -kx * r0.y, rXC = kx * r0.x, rYR = -ky * r0.y, rYC = ky * r0.x, rZR = -kz * r0.y,
               rZC = kz * r0.x;
  const double ri = p.ri, s = p.sinth, co = p.costh;
  C[0] = LC * (ky * WKY - kz * VKY - ri * (rYR * s - rZR * co));
  C[1] = LC * (kz * VKX - ky * WKX - ri * (rYC * s - rZC * co));
  C[2] = LC * (kz * UKY - kx * WKY + ri * rXR * s);
  C[3] = LC * (kx * WKX - kz * UKX + ri * rXC * s);
  C[4] = LC * (kx * VKY - ky * UKY - ri * rXR * co);
  C[5] = LC * (ky * UKX - kx * VKX - ri * rXC * co);
  C[6] = -LC * (N[3].x + (kz * x0.y - kx * z0.y) * wki * co + (kx * e0.y - ky * x0.y) * wki * s);
  C[7] = -LC * (N[3].y + (kx * z0.x - kz * x0.x) * wki * co + (ky * x0.x - kx * e0.x) * wki * s);
  if (kx == 0.0 && kz == 0.0 && ky == p.kf) C[4] += p.ampfor;
}

template <int STAGE> struct UpdBous {
  cpx<double> *st, *s0, *xs;  // state [m][4][nkt]; stage input (LayZ0) and increments (LayXS, field 4 stage + f)
  long nkt, nktw;
  const int8_t *L;
  BousPar p;
  Grid g;
  __device__ __forceinline__ void operator()(int m, long ik, int ikx, double kx, double ky, double kz,
                                             cpx<double> (&N)[4]) const {
    const int iky = (int)ky + g.kty, ikz = (int)kz + g.ktz;
    cpx<double> *S = st + (long)m * 4 * nkt + ik;
    cpx<double> *Z = s0 + (long)m * 4 * nktw + LayZ0::at(g, ikx, iky, ikz);
    cpx<double> *X = xs + (long)m * 12 * nktw + LayXS::at(g, ikx, iky, ikz);
    constexpr int zf = 8;
    const double wk = kx * kx + ky * ky + kz * kz;
    const double dt = p.dt;
    const double LC = (double)L[ik];
    double C[8];
    if constexpr (STAGE < 3) {
      bous_rhs(p, kx, ky, kz, LC, N, Z[0], Z[zf], Z[2 * zf], Z[3 * zf], C);
      const double q = STAGE < 2 ? 0.25 : 0.5, h = STAGE < 2 ? 0.5 : 1.0;
      const double d1 = (1. - q * dt * p.v2 * wk) / (1. + q * dt * p.v2 * wk);
      const double d2 = (1. - q * dt * p.v2 * wk / p.sc) / (1. + q * dt * p.v2 * wk / p.sc);
#pragma unroll
      for (int f = 0; f < 4; f++) {
        X[(STAGE * 4 + f) * zf] = cpx<double>{dt * C[2 * f], dt * C[2 * f + 1]};
        const double d = f < 3 ? d1 : d2;
        const cpx<double> sn = S[f * nkt];
        Z[f * zf] = cpx<double>{d * (sn.x + h * dt * C[2 * f]), d * (sn.y + h * dt * C[2 * f + 1])};
      }
    } else {
      bous_rhs(p, kx, ky, kz, 1.0, N, Z[0], Z[zf], Z[2 * zf], Z[3 * zf], C);
      const double d1 = 1. - 0.5 * dt * p.v2 * wk, d2 = 1. - 0.5 * dt * p.v2 * wk / p.sc;
      const double den1 = 1. + 0.5 * dt * p.v2 * wk, den2 = 1. + 0.5 * dt * p.v2 * wk / p.sc;
      const double sixth = 1.0 / 6.0, third = 1.0 / 3.0;
      cpx<double> r[4];
#pragma unroll
      for (int f = 0; f < 4; f++) {
        const double d = f < 3 ? d1 : d2, den = f < 3 ? den1 : den2;
        const cpx<double> sn = S[f * nkt], x1 = X[f * zf], x2 = X[(4 + f) * zf], x3 = X[(8 + f) * zf];
        r[f].x = LC * (d * sn.x + sixth * (x1.x + dt * C[2 * f]) + third * (x2.x + x3.x)) / den;
        r[f].y = LC * (d * sn.y + sixth * (x1.y + dt * C[2 * f + 1]) + third * (x2.y + x3.y)) / den;
        Z[f * zf] = r[f];
      }
      const double wki = 1.0 / (wk > 0.001 ? wk : 0.001);
      const double phiR = (kx * r[0].y + ky * r[1].y + kz * r[2].y) * wki;
      const double phiC = -(kx * r[0].x + ky * r[1].x + kz * r[2].x) * wki;
      r[0].x -= -kx * phiC; r[0].y -= kx * phiR;
      r[1].x -= -ky * phiC; r[1].y -= ky * phiR;
      r[2].x -= -kz * phiC; r[2].y -= kz * phiR;
#pragma unroll
      for (int f = 0; f < 4; f++) S[f * nkt] = r[f];
    }
  }
};

// dz/dt for Newton (3D_Boussinesq/src/kernels.h:624-692): out = -nu k^2 z + C
struct UpdBousRHS {
  const cpx<double> *st;       // the state, which is also the stage input
  cpx<double> *out;
  long nkt;
  const int8_t *L;
  BousPar p;
  __device__ __forceinline__ void operator()(int m, long ik, int, double kx, double ky, double kz,
                                             cpx<double> (&N)[4]) const {
    const cpx<double> *S = st + (long)m * 4 * nkt + ik;
    double C[8];
    bous_rhs(p, kx, ky, kz, (double)L[ik], N, S[0], S[nkt], S[2 * nkt], S[3 * nkt], C);
    const double wk = kx * kx + ky * ky + kz * kz;
    const double d1 = -p.v2 * wk, d2 = -p.v2 * wk / p.sc;
    cpx<double> *o = out + (long)m * 4 * nkt + ik;
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const double d = f < 3 ? d1 : d2;
      o[f * nkt] = cpx<double>{d * S[f * nkt].x + C[2 * f], d * S[f * nkt].y + C[2 * f + 1]};
    }
  }
};

// stage input = state (setVelocity), in LayZ0 (padding columns zero)
__global__ void k_stage_bous(const cpx<double> *__restrict__ a, cpx<double> *__restrict__ b, Grid g, long nktw, long total) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long m = i / (4 * nktw), w = i - m * 4 * nktw, run = w / 32;
    const int f = (int)((w >> 3) & 3), ikz = (int)(run % g.iktz);
    const long t = run / g.iktz;
    const int iky = (int)(t % g.ikty), ikx = (int)(t / g.ikty) * 8 + (int)(w & 7);
    b[i] = ikx < g.iktx ? a[(m * 4 + f) * g.nkt + LayNKT::at(g, ikx, iky, ikz)] : cpx<double>{0, 0};
  }
}

// ------------------------------------------------------------------ launches
#define PSG_TRYB(x)     \
  do {                  \
    int r_ = (x);       \
    if (r_) return r_;  \
  } while (0)

// LAY: LayZ0 (the stage input) or LayNKT (a state)
template <typename P, class LAY>
static int launch_zinv_b(Ctx *c, const cpx<double> *st, int umask, int nm, int nout = 9) {
  const Grid &g = c->g;
  cpx<P> *A = (cpx<P> *)c->bufA;
  PSG_DISPATCH_N(g.nz, {
    constexpr int T = Col<N, P>::T;
    dim3 grid((g.iktx + T - 1) / T, g.ikty, nm);
    size_t lds = (size_t)(N * T + N) * sizeof(cpx<P>);
    constexpr bool RUN = std::is_same<LAY, LayZ0>::value;
    // with blocks for three quarters of the CUs or fewer: 32^3 FP64 19.4 -> 13.9 us, 64^3
    // (129 blocks) 21.5 -> 17.0; at 128^3 (255 blocks) the split costs, 30 -> 34.3
    const bool split = grid.x * grid.y * grid.z <= 192;
    auto k = split ? k_zinv_bous<P, N, T, LAY, true> : k_zinv_bous<P, N, T, LAY, false>;
    PSG_HIP(lds_attr(k, lds));
    if (split) grid.z *= 3;
    hipLaunchKernelGGL(k, grid, dim3(Col<N, P>::THREADS), lds, c->stream, st, 4 * (RUN ? c->nktw : g.nkt),
                       RUN ? 8L : g.nkt, A, 9 * g.zsz, g, twp<P>(c, 2), c->mask, umask, nout);
  });
  PSG_HIP(hipGetLastError());
  return 0;
}

template <typename P> int launch_xphys(Ctx *c, const cpx<P> *in, double *out, int nf);

// x-pass shapes of the Boussinesq product (9 inputs, 4 outputs), chosen per
// context by psg_autotune: the variants of the Navier-Stokes x-pass (points per
// thread, input front-loading, per-pair product re-evaluation, rows per block,
// register caps)
template <typename P> static int xpass_bous(Ctx *c, const cpx<P> *B, cpx<P> *Cb, int nm) {
  const long nr = (long)c->g.ny * c->g.nz;
  const ProdBous<P> pb{};
  // variant 0 is the shape measured fastest for the length and precision (us):
  //   FP64, 256 points on: 3 (8 points a thread 516, this 394 at 256^3; 4530, 3543 at 512^3), 32 to 128: 4
  //     (16.8, 14.2 at 32^3; 17.9, 15.0 at 64^3; 70.0, 60.3 at 128^3; 117, 98.8 at 64^3 with 16 members)
  //   FP32, 32 and 64: 4 (15.8, 12.8; 15.1, 13.0), 128: 2 (37.2, 35.6), above: 8 points, product kept
  //   16 points: 8 points a thread although 4 is faster (19.1, 10.8).  This is not a matter of
  //     speed or of accuracy: a two-shift Newton solve at 16^3 whose Jacobian is singular stops
  //     at a shift of 1.34e-5 with the radix-4 shapes (3, 4, 7, 8, 9, 11) and below 1e-5, the
  //     bound that is asked of it, with the radix-8 ones
  // Shape 3 and 4 add in another order (radix 4 throughout): one 512^3 step is 1.8e-16 of its
  // state off its 64-bit value, and 1.6e-16 with radix 8
  const int n = c->g.nx;
  const int best = n < 32 ? 0 : sizeof(P) == 8 ? (n >= 256 ? 3 : 4) : (n <= 64 ? 4 : n == 128 ? 2 : 0);
  const int xv = c->xvar ? c->xvar : best;
  switch (xv) {
    case 1: return launch_xpass<P, 9, 4, ProdBous<P>, 8, true, true>(c, B, Cb, nr, nm, pb);
    case 2: return launch_xpass<P, 9, 4, ProdBous<P>, 8, false, true>(c, B, Cb, nr, nm, pb);
    case 3: return launch_xpass<P, 9, 4, ProdBous<P>, 4, true, false>(c, B, Cb, nr, nm, pb);
    case 4: return launch_xpass<P, 9, 4, ProdBous<P>, 4, false, true>(c, B, Cb, nr, nm, pb);
    case 5: return launch_xpass<P, 9, 4, ProdBous<P>, 8, false, true, 2>(c, B, Cb, nr, nm, pb);
    case 6: return launch_xpass<P, 9, 4, ProdBous<P>, 8, false, true, 4>(c, B, Cb, nr, nm, pb);
    case 7: return launch_xpass<P, 9, 4, ProdBous<P>, 4, false, true, 1>(c, B, Cb, nr, nm, pb);
    case 8:
    case 9:
      if constexpr (std::is_same<P, float>::value) {
        if (xv == 8) return launch_xpass<P, 9, 4, ProdBous<P>, 16, false, true>(c, B, Cb, nr, nm, pb);
        return launch_xpass<P, 9, 4, ProdBous<P>, 16, false, true, 4>(c, B, Cb, nr, nm, pb);
      }
      return launch_xpass<P, 9, 4, ProdBous<P>, 4, false, true, 2>(c, B, Cb, nr, nm, pb);
    case 10:
      return launch_xpass<P, 9, 4, ProdBous<P>, 8, false, true, 0, sizeof(P) == 8 ? 4 : 5>(c, B, Cb, nr, nm, pb);
    case 11:
      return launch_xpass<P, 9, 4, ProdBous<P>, 4, false, true, 0, sizeof(P) == 8 ? 5 : 6>(c, B, Cb, nr, nm, pb);
    default: return launch_xpass<P, 9, 4, ProdBous<P>>(c, B, Cb, nr, nm, pb);
  }
}

template <typename P, class UPD> static int launch_zfwd_b(Ctx *c, const cpx<P> *in, UPD upd, int nm) {
  const Grid &g = c->g;
  PSG_DISPATCH_N(g.nz, {
    constexpr int T = Col<N, P>::T;
    dim3 grid((g.iktx + T - 1) / T, g.ikty, nm);
    size_t lds = (size_t)(N * T + N) * sizeof(cpx<P>);
    // short transforms: all loads of a block in flight at once, whatever the
    // registers (up to 290 in FP64, one wave per SIMD).  From 256 points on there
    // are blocks enough for occupancy to count: the update's loads stay within
    // pairs of modes, and in FP64 each field is loaded at its own transform
    // (256^3 FP64 297 -> 229 us, FP32 209 -> 201; at 64^3 it would be 21 -> 26).  Two
    // waves per SIMD leave 256 registers a thread: FP64 keeps 104 to 200 bytes a lane
    // in scratch, FP32 none.  Either way it waits for memory for 61 to 81% of its time
    constexpr bool LONG = N >= 256;
    auto k = k_zfwd<P, N, T, 4, UPD, (sizeof(P) == 4 || !LONG), 1, (LONG ? 2 : 0), (LONG && N <= 512 ? 2 : 1)>;
    PSG_HIP(lds_attr(k, lds));
    hipLaunchKernelGGL(k, grid, dim3(Col<N, P>::THREADS), lds, c->stream, in, g, twp<P>(c, 2), upd);
  });
  PSG_HIP(hipGetLastError());
  return 0;
}

template <typename P, class LAY, class UPD> static int rhs_b(Ctx *c, const cpx<double> *s0, int umask, UPD upd, int nm) {
  const Grid &g = c->g;
  cpx<P> *A = (cpx<P> *)c->bufA, *B = (cpx<P> *)c->bufB, *Cb = (cpx<P> *)c->bufC;
  const long Z = (long)g.iktx * g.ikty * g.nz, Y = (long)g.iktx * g.ny * g.nz;
  const long b = sizeof(cpx<P>);
  prof_begin(c, "zinv_bous", (4 * g.nkt * 16 + 9 * Z * b) * nm);
  PSG_TRYB((launch_zinv_b<P, LAY>(c, s0, umask, nm)));
  prof_end(c);
  prof_begin(c, "yinv", 9 * (Z + Y) * b * nm);
  PSG_TRYB(launch_yinv_g<P>(c, A, B, 9 * nm));
  prof_end(c);
  prof_begin(c, "xpass_bous", 13 * Y * b * nm);
  PSG_TRYB(xpass_bous<P>(c, B, Cb, nm));
  prof_end(c);
  prof_begin(c, "yfwd", 4 * (Y + Z) * b * nm);
  PSG_TRYB(launch_yfwd_g<P>(c, Cb, A, 4 * nm));
  prof_end(c);
  prof_begin(c, "zfwd_update_bous", (4 * Z * b + 16 * g.nkt * 16) * nm);
  PSG_TRYB((launch_zfwd_b<P>(c, A, upd, nm)));
  prof_end(c);
  return 0;
}

static BousPar bpar(const Ctx *c) {
  return BousPar{c->cfg.dt, c->cfg.v2, c->cfg.sc, c->cfg.ri, sin(c->cfg.theta), cos(c->cfg.theta), c->cfg.kf,
                 c->cfg.ampfor};
}

template <typename P> static int runb_t(Ctx *c, int nsteps, bool first) {
  const Grid &g = c->g;
  if (first) {
    // stage input = state (setVelocity); later steps leave it equal to the state themselves
    const long tot = 4 * c->nktw * c->batch;
    hipLaunchKernelGGL(k_stage_bous, dim3((unsigned)std::min<long>(8192, (tot + 255) / 256)), dim3(256), 0, c->stream,
                       c->state, c->stage, g, c->nktw, tot);
    PSG_HIP(hipGetLastError());
  }
  const BousPar p = bpar(c);
  for (int nt = 0; nt < nsteps; nt++) {
#define PSG_BOUS_STAGE(S)                                                                         \
    {                                                                                             \
      UpdBous<S> u{c->state, c->stage, c->rh, g.nkt, c->nktw, c->mask, p, g};                     \
      PSG_TRYB((rhs_b<P, LayZ0>(c, c->stage, (S == 0 && first && nt == 0) ? 1 : 0, u, c->batch))); \
    }
    PSG_BOUS_STAGE(0) PSG_BOUS_STAGE(1) PSG_BOUS_STAGE(2) PSG_BOUS_STAGE(3)
#undef PSG_BOUS_STAGE
  }
  return 0;
}

int bous_run(Ctx *c, int nsteps, bool first) {
  return c->cfg.precision == PSG_FP32BULK ? runb_t<float>(c, nsteps, first) : runb_t<double>(c, nsteps, first);
}

template <typename P> static int rhsb_t(Ctx *c, const cpx<double> *in, cpx<double> *out) {
  UpdBousRHS u{in, out, c->g.nkt, c->mask, bpar(c)};
  return rhs_b<P, LayNKT>(c, in, 1, u, 1);
}

int bous_timederiv(Ctx *c, const cpx<double> *in_dev, cpx<double> *out_dev) {
  return c->cfg.precision == PSG_FP32BULK ? rhsb_t<float>(c, in_dev, out_dev) : rhsb_t<double>(c, in_dev, out_dev);
}

// physical fields of one member: w(3), u(3), rho, NR doubles each, x fastest
template <typename P> static int physb_t(Ctx *c, const cpx<double> *st, double *out) {
  const Grid &g = c->g;
  PSG_TRYB((launch_zinv_b<P, LayNKT>(c, st, 1, 1, 7)));
  PSG_TRYB(launch_yinv_g<P>(c, (const cpx<P> *)c->bufA, (cpx<P> *)c->bufB, 7));
  return launch_xphys<P>(c, (const cpx<P> *)c->bufB, out, 7);
}

int bous_physical_state(Ctx *c, const cpx<double> *st, double *out_dev) {
  return c->cfg.precision == PSG_FP32BULK ? physb_t<float>(c, st, out_dev) : physb_t<double>(c, st, out_dev);
}

int bous_physical(Ctx *c, int member, double *out_dev) {
  return bous_physical_state(c, c->state + (long)member * 4 * c->g.nkt, out_dev);
}

int bous_init(Ctx *c) {
  const Grid &g = c->g;
  size_t b = c->cfg.precision == PSG_FP32BULK ? sizeof(cpx<float>) : sizeof(cpx<double>);
  c->szA = (size_t)9 * g.zsz * c->batch * b;
  c->szB = (size_t)9 * g.ysz * c->batch * b;
  c->szC = (size_t)4 * g.ysz * c->batch * b;
  PSG_HIP(hipMalloc(&c->bufA, c->szA));
  PSG_HIP(hipMalloc(&c->bufB, c->szB));
  PSG_HIP(hipMalloc(&c->bufC, c->szC));
  c->nktw = (long)((g.iktx + 7) / 8) * 8 * g.ikty * g.iktz;
  PSG_HIP(hipMalloc(&c->rh, sizeof(cpx<double>) * 12 * c->nktw * c->batch));
  PSG_HIP(hipMalloc(&c->stage, sizeof(cpx<double>) * 4 * c->nktw * c->batch));
  PSG_HIP(hipMemsetAsync(c->rh, 0, sizeof(cpx<double>) * 12 * c->nktw * c->batch, c->stream));
  PSG_HIP(hipMemsetAsync(c->stage, 0, sizeof(cpx<double>) * 4 * c->nktw * c->batch, c->stream));
  return 0;
}

}  // namespace psg
