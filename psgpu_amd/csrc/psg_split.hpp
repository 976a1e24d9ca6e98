// Two-kernel right-hand side of the 3D Navier-Stokes/Euler steppers.
//
// The y transform is split between the two kernels (N_y = 16 RA, four-step
// form): position p = k1 + 16 k2 of the padded spectrum and row y = y2 + RA y1,
//   W^(p y) = W_RA^(k2 y2) W_N^(k1 y2) W_16^(k1 y1),
// so the RA-point part runs where the whole z axis is on chip and the 16-point
// part where the whole x axis is:
//   z kernel (k_zsplit): forward y2 and z transforms of the products, Heun/CN
//     update of the modes, velocity and inverse z and y2 transforms of the next
//     stage's six fields, for two or three kx columns and one k1
//   xy kernel (k_xysplit): inverse y1 and x transforms, product, forward x and
//     y1 transforms, for one (z, y2): 16 rows
// Between them move F (six fields, [f][kx group][k1][y2][z][kb]) and G (three
// products, [f][z][y2][k1][kx]).  A step is four launches instead of ten, with
// fewer barriers and memory latencies in a row inside them, and the state is not
// read again for the inverse transforms.  Each kernel writes whole runs and
// gathers its reads in pieces of kb points; workgroups that share the gathered
// lines run next to each other on one XCD.
#pragma once
#include "psg_ns3d.hpp"

namespace psg {

constexpr int SPLIT_RB = 16;   // rows of the xy kernel, points of its y transform

// kx columns per z-kernel block: G and F move in pieces of kb points.  Two make
// pieces of 32 bytes in FP64; in FP32 they make 16, and from 1024 (z, y2) points a
// column on three are taken: fewer pieces, for more threads a block (864 instead of
// 576) and fewer blocks.  In FP64 the larger blocks cost more than they give.  One
// step in us, one context / three at a time, two columns and three:
//   FP64 32x128x128 84.8 / 43.7, 117 / 50.8; 64x128x128 96.9 / 71.8, 127 / 85.9
//   FP32 128^3 130 / 95.1, 105 / 89.1; 64x128x128 x 2 131 / 97.1, 105 / 92.7;
//        64x128x128 84.5 / 52.8, 91.1 / 46.6; 32x128x128 74.1 / 33.4, 84.7 / 35.2
__host__ __device__ constexpr int split_kb(bool fp32, int nz, int ra) { return fp32 && nz * ra >= 1024 ? 3 : 2; }

// sizes and pitches of the split buffers and of the working layout
struct Split {
  int ra, kb, ng;    // y2 count; kx columns of a z-kernel block (split_kb); groups of kb columns
  int pa;            // points of one (group, k1) chunk of F: ra nz kb, and 8 so that in FP64 chunks
                     // start an odd number of 128-byte lines apart (in FP32 of half lines)
  int xq, zp;        // kx pitch of a G row; points of one z plane of G (likewise padded)
  int kzp;           // kz pitch of the working state [ikx][iky][f][kz], kz = 0..KTZ, -KTZ..-1
  long fs, gs;       // points per field of F and G
  long nkts;         // working modes per field
  static Split of(const Ctx *c) {
    const Grid &g = c->g;
    Split s;
    s.ra = g.ny / SPLIT_RB;
    s.kb = split_kb(c->cfg.precision == PSG_FP32BULK, g.nz, s.ra);
    s.ng = (g.iktx + s.kb - 1) / s.kb;
    s.pa = s.ra * g.nz * s.kb + 8;
    s.xq = (g.iktx + 7) / 8 * 8;
    s.zp = g.ny * s.xq + 8;
    s.kzp = (g.iktz + 7) / 8 * 8;
    s.fs = (long)s.ng * SPLIT_RB * s.pa;
    s.gs = (long)g.nz * s.zp;
    s.nkts = (long)g.iktx * g.ikty * s.kzp;
    return s;
  }
  __device__ __forceinline__ long at(const Grid &g, int ikx, int iky, int kz) const {
    return ((long)ikx * g.ikty + iky) * 3 * kzp + (kz < 0 ? kz + g.iktz : kz);
  }
  __device__ __forceinline__ long tab(const Grid &g, int ikx, int iky, int kz) const {
    return ((long)ikx * g.ikty + iky) * kzp + (kz < 0 ? kz + g.iktz : kz);
  }
};

// what a z kernel does with the modes it holds
struct SplitUpd {
  int fwd;           // 0: load the state and transform back only (first stage of a run)
  int phase, euler;  // Heun half-step, flavour
  int umask;         // velocity masked by L (first stage of a run)
  int last;          // update only (last stage of a run)
  double dt;
  Force F;
};

template <typename P, int NZ, int RA> struct ZShape {
  static constexpr int TP = NZ / EPT;
  static constexpr int NC = 2 * RA / 3 + 1;      // columns p = k1 + 16 k2 inside the 2/3 band, at most
  static constexpr int KB = split_kb(sizeof(P) == 4, NZ, RA), COLS = KB * NC;
  static constexpr int NT = 3 * COLS * TP;
  static constexpr size_t lds() { return (size_t)(NZ + 3 * COLS * NZ) * sizeof(cpx<P>); }
};

// One block: kb columns of kx, one k1, all k2 and kz, three fields side by side
// (a team of NZ/8 threads per field and column, one LDS row each).  The update
// reads the state from st and writes it to sn: the fill of kx = 0 takes half of
// its modes from the mirrored ones, which another block updates.  A block makes
// their new values itself, from its own transforms (the products are real, so
// N(-k) = conj N(k)), and must find their old values whole.
template <typename P, int NZ, int RA>
__global__ void __launch_bounds__((ZShape<P, NZ, RA>::NT)) PSG_WAVES_PER_EU((sizeof(P) == 4 ? 4 : 3))
k_zsplit(const cpx<P> *__restrict__ G, cpx<P> *__restrict__ F, const cpx<P> *__restrict__ st, cpx<P> *__restrict__ sn,
         cpx<P> *__restrict__ rh, const double *__restrict__ nuzn, const double *__restrict__ nu1,
         const int8_t *__restrict__ L, Grid g, Split d, const cpx<P> *__restrict__ tw, SplitUpd u) {
  using Z = ZShape<P, NZ, RA>;
  constexpr int E = EPT, TP = Z::TP, NT = Z::NT, KB = Z::KB, COLS = Z::COLS;
  constexpr int SW = row_swizzle<E>();
  PSG_TWIDDLES_REQUEST(P, NZ, E, NT);
  // groups of one k1 next to each other on an XCD: they share the lines of G
  const TileId tid = xcd_tile();
  const int grp = tid.x, k1 = tid.y, m = tid.z;
  const int t = threadIdx.x, team = t / TP, j = t % TP, fld = team / COLS, tq = team % COLS;
  cpx<P> *row = lds + team * NZ;
  // element z of row (f, column q), rotated so that the columns of a gather lie on different banks
  auto el = [&](int f, int q, int z) -> cpx<P> & { return lds[(f * COLS + q) * NZ + ((z + (q % KB) * (8 / KB + KB % 2)) & (NZ - 1))]; };
  const cpx<P> *S = st + (long)m * 3 * d.nkts;
  cpx<P> *SN = sn + (long)m * 3 * d.nkts, *R = rh + (long)m * 3 * d.nkts;
  const int fs = d.kzp;
  // columns of k1: k2 < nlo (ky >= 0) and k2 >= RA - nhi (ky < 0)
  const int nlo = k1 <= g.kty ? (g.kty - k1) / SPLIT_RB + 1 : 0;
  const int nhi = RA - (g.ny - g.kty - k1 + SPLIT_RB - 1) / SPLIT_RB;
  // column q = ci KB + c: its kx index and ky; false where there is none
  auto column = [&](int q, int &ikx, int &ky) {
    const int ci = q / KB, k2 = ci < nlo ? ci : RA - nhi + ci - nlo, p = k1 + SPLIT_RB * k2;
    ikx = grp * KB + q % KB;
    ky = ci < nlo ? p : p - g.ny;
    return ikx < g.iktx && ci < nlo + nhi;
  };
  // mode i of the block, kz fastest
  struct Mode {
    int q, p, ikx, ky, kz;   // column, row position, wavenumbers
    bool on, mirror;         // there is such a mode; the fill takes it from -k
  };
  auto mode = [&](int i) {
    Mode o;
    o.q = i / g.iktz;
    const int c = i - o.q * g.iktz;
    o.kz = c <= g.ktz ? c : c - g.iktz;
    o.p = o.kz < 0 ? o.kz + NZ : o.kz;
    o.on = o.q < COLS && column(o.q, o.ikx, o.ky);
    o.mirror = o.on && o.ikx == 0 && (o.ky < 0 || (o.ky == 0 && o.kz < 0));
    return o;
  };
  // everything the update reads of one mode, requested ahead of its use
  struct In {
    cpx<P> s[3], r[3];
    double zn, n1;
    int8_t l;
  };
  auto fetch = [&](bool on, int ikx, int ky, int kz) {
    In a{};
    if (on) {
      const long ik = d.at(g, ikx, ky + g.kty, kz), it = d.tab(g, ikx, ky + g.kty, kz);
      a.l = L[it];
      if (!u.euler) a.n1 = nu1[it];
      if (!u.euler && u.phase == 0) a.zn = nuzn[it];
#pragma unroll
      for (int f = 0; f < 3; f++) a.s[f] = S[ik + f * fs];
      if (u.phase == 1) {
#pragma unroll
        for (int f = 0; f < 3; f++) a.r[f] = R[ik + f * fs];
      }
    }
    return a;
  };
  // new values n of the mode (kx, ky, kz) from its transformed products N, and its RH
  auto heun = [&](double kx, double ky, double kz, const cpx<double> (&N)[3], const In &a, cpx<P> (&n)[3], cpx<P> (&rn)[3]) {
    PSG_CURL
    cpx<double> C[3] = {{xiX, xiY}, {etX, etY}, {ztX, ztY}};
    const double ll = (double)a.l;
    if (!u.euler) add_forcing(u.F, kx, ky, kz, C[0].x, C[1].y, C[2].x, C[2].y);
    // phase 0: RH = rl C, w* = n1 (zn w + cl C); phase 1: w = ll (w* + n2 (C - RH))
    const double zn = u.euler ? 1.0 : a.zn, n1 = u.euler ? 1.0 : ll * a.n1, rl = u.euler ? ll : 1.0,
                 cl = u.euler ? u.dt : 1.0, n2 = 0.5 * (u.euler ? u.dt : a.n1);
#pragma unroll
    for (int f = 0; f < 3; f++) {
      const cpx<double> w = up(a.s[f]), r = up(a.r[f]);
      if (u.phase == 0) {
        rn[f] = to<P>(cpx<double>{rl * C[f].x, rl * C[f].y});
        n[f] = to<P>(cpx<double>{n1 * (zn * w.x + cl * C[f].x), n1 * (zn * w.y + cl * C[f].y)});
      } else {
        n[f] = to<P>(cpx<double>{ll * (w.x + n2 * (C[f].x - r.x)), ll * (w.y + n2 * (C[f].y - r.y))});
      }
    }
  };
  auto update = [&](const Mode &o, const In &a) {
    if (!o.on) return;
    const double kx = (double)o.ikx * g.alpha, ky = (double)o.ky, kz = (double)o.kz;
    const long ik = d.at(g, o.ikx, o.ky + g.kty, o.kz);
    cpx<double> N[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
      const cpx<double> v = up(el(f, o.q, o.p));
      N[f] = cpx<double>{v.x * g.inr, v.y * g.inr};
    }
    cpx<P> n[3], rn[3];
    heun(kx, ky, kz, N, a, n, rn);
#pragma unroll
    for (int f = 0; f < 3; f++) {
      if (u.phase == 0) R[ik + f * fs] = rn[f];
      SN[ik + f * fs] = n[f];
    }
    if (o.mirror) {
      const In b = fetch(true, 0, -o.ky, -o.kz);
#pragma unroll
      for (int f = 0; f < 3; f++) N[f].y = -N[f].y;
      heun(kx, -ky, -kz, N, b, n, rn);
#pragma unroll
      for (int f = 0; f < 3; f++) n[f].y = -n[f].y;
    } else if (o.ikx == 0 && o.ky == 0 && o.kz == 0) {
      n[0] = n[1] = n[2] = cpx<P>{0, 0};
    }
#pragma unroll
    for (int f = 0; f < 3; f++) el(f, o.q, o.p) = n[f];
  };
  constexpr int NI = (COLS * (2 * (NZ / 3) + 1) + NT - 1) / NT;   // modes per thread
  constexpr int NJ = (3 * KB * NZ + NT - 1) / NT;                 // y2 transforms per thread
  if (u.fwd) {
    // y2 transforms at fixed z; a thread's inputs of all its work are requested first
    cpx<P> r[NJ][RA];
#pragma unroll
    for (int i = 0; i < NJ; i++) {
      const int job = t + i * NT, c = job % KB, z = job / KB % NZ, f = job / (KB * NZ);
      const cpx<P> *src = G + ((long)m * 3 + f) * d.gs + (long)z * d.zp + k1 * d.xq + grp * KB + c;
#pragma unroll
      for (int y2 = 0; y2 < RA; y2++) r[i][y2] = f < 3 ? src[y2 * SPLIT_RB * d.xq] : cpx<P>{0, 0};
    }
    In in[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const Mode o = mode(t + i * NT);
      in[i] = fetch(o.on, o.ikx, o.ky, o.kz);
    }
    PSG_TWIDDLES_READY(P);
#pragma unroll
    for (int i = 0; i < NJ; i++) {
      const int job = t + i * NT, c = job % KB, z = job / KB % NZ, f = job / (KB * NZ);
      dftR<P, false, RA>(r[i]);
#pragma unroll
      for (int k2 = 0; k2 < RA; k2++) {
        const int cc = k2 < nlo ? k2 : k2 - (RA - nhi) + nlo;
        if (f < 3 && (k2 < nlo || k2 >= RA - nhi)) el(f, cc * KB + c, z) = r[i][k2];
      }
    }
    __syncthreads();
    cpx<P> v[E];
#pragma unroll
    for (int mm = 0; mm < E; mm++) v[mm] = el(fld, tq, j + TP * mm);
    team_sync<true>();
    fft_pencil<P, NZ, E, false, true, SW>(v, row, j, 1, 0, tw);
    team_sync<true>();
#pragma unroll
    for (int mm = 0; mm < E; mm++) el(fld, tq, j + TP * mm) = v[mm];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NI; i++) update(mode(fresh(t) + i * NT), in[i]);
    if (u.last) return;
  } else {
    // the state with the Hermitian fill of kx = 0
    PSG_TWIDDLES_READY(P);
#pragma unroll 1
    for (int i = t; i < COLS * g.iktz; i += NT) {
      const Mode o = mode(i);
      if (!o.on) continue;
      const long ik = d.at(g, o.ikx, (o.mirror ? -o.ky : o.ky) + g.kty, o.mirror ? -o.kz : o.kz);
#pragma unroll
      for (int f = 0; f < 3; f++) {
        cpx<P> a = S[ik + f * fs];
        if (o.ikx == 0 && o.ky == 0 && o.kz == 0) a = cpx<P>{0, 0};
        if (o.mirror) a.y = -a.y;
        el(f, o.q, o.p) = a;
      }
    }
  }
  __syncthreads();
  // this team's component of vorticity and velocity; component fld of i k x w
  // takes the other two components in cyclic order
  cpx<P> v[E], vel[E];
  {
    const int f1 = fld == 2 ? 0 : fld + 1, f2 = fld == 0 ? 2 : fld - 1;
    int ikx, iky;
    const bool on = column(tq, ikx, iky);
    const double kx = (double)ikx * g.alpha, kyd = (double)iky;
#pragma unroll
    for (int mm = 0; mm < E; mm++) {
      const int p = fresh(j) + TP * mm, kz = wrapk(p, NZ, g.ktz);
      v[mm] = vel[mm] = cpx<P>{0, 0};
      if (on && kz != PSG_NOK) {
        v[mm] = el(fld, tq, p);
        const double kzd = (double)kz, wk = kx * kx + kyd * kyd + kzd * kzd;
        double wki = 1.0 / (wk > 0.001 ? wk : 0.001);
        if (u.umask) {
          const bool mirror = ikx == 0 && (iky < 0 || (iky == 0 && kz < 0));
          wki *= (double)L[d.tab(g, ikx, (mirror ? -iky : iky) + g.kty, mirror ? -kz : kz)];
        }
        const double ka = fld == 0 ? kyd : (fld == 1 ? kzd : kx), kb = fld == 0 ? kzd : (fld == 1 ? kx : kyd);
        const cpx<double> a = up(el(f1, tq, p)), b = up(el(f2, tq, p));
        vel[mm] = to<P>(cpx<double>{-(ka * b.y - kb * a.y) * wki, -(kb * a.x - ka * b.x) * wki});
      }
      PSG_COMPILER_FENCE();
    }
  }
  __syncthreads();
#pragma unroll
  for (int half = 0; half < 2; half++) {
    if (half == 1) {
#pragma unroll
      for (int mm = 0; mm < E; mm++) v[mm] = vel[mm];
    }
    fft_pencil<P, NZ, E, true, true, SW>(v, row, j, 1, 0, tw);
    team_sync<true>();
#pragma unroll
    for (int mm = 0; mm < E; mm++) el(fld, tq, j + TP * mm) = v[mm];
    __syncthreads();
#pragma unroll 1
    for (int job = fresh(t); job < 3 * KB * NZ; job += NT) {
      const int c = job % KB, z = job / KB % NZ, f = job / (KB * NZ);
      cpx<P> r[RA];
#pragma unroll
      for (int k2 = 0; k2 < RA; k2++) {
        const int cc = k2 < nlo ? k2 : k2 - (RA - nhi) + nlo;
        r[k2] = (k2 < nlo || k2 >= RA - nhi) ? el(f, cc * KB + c, z) : cpx<P>{0, 0};
      }
      dftR<P, true, RA>(r);
      cpx<P> *o = F + ((long)m * 6 + half * 3 + f) * d.fs + (long)(grp * SPLIT_RB + k1) * d.pa + z * KB + c;
#pragma unroll
      for (int y2 = 0; y2 < RA; y2++) o[y2 * (KB * NZ)] = r[y2];
    }
    if (half == 0) __syncthreads();
  }
}

// ------------------------------------------------------------------ xy kernel
template <int NX> struct XShape {
  static constexpr int TP = NX / EPT, NT = SPLIT_RB * TP, IX = xband<NX>();
  template <typename P> static constexpr size_t lds() {
    return (size_t)(NX + SPLIT_RB * NX + 4 * SPLIT_RB * IX) * sizeof(cpx<P>);
  }
};

// Persistent blocks, one (z, y2) unit after the other, z fastest.  The next
// unit's values of F are requested as soon as this unit's y1 transforms have
// taken theirs out of the registers, and are in flight during its x transforms:
// a CU holds two such blocks in FP64, too few to hide that latency otherwise.
// Thread t transforms column kx < IX - 1 of field f in y1 (t = f (IX-1) + kx; six
// fields fill 252 of the 256 threads at NX = 128); the last column's values are
// loaded one per thread and summed directly.
// LDS-bound: at 128^3 in FP64 the LDS pipe is busy for 22 of its 42 us, the
// vector ALUs for 15; at 64^3 it takes 12.4 us, the z kernel 14.7 us.
template <typename P, int NX>
__global__ void __launch_bounds__((XShape<NX>::NT)) PSG_WAVES_PER_EU(sizeof(P) == 8 ? 2 : 4)
k_xysplit(const cpx<P> *__restrict__ F, cpx<P> *__restrict__ G, Grid g, Split d, const cpx<P> *__restrict__ tw,
          const cpx<P> *__restrict__ twy, int units) {
  using X = XShape<NX>;
  constexpr int RB = SPLIT_RB, TP = X::TP, NT = X::NT, IX = X::IX, SW = row_swizzle<EPT>();
  constexpr int NE = (6 * RB + NT - 1) / NT;   // last-column values per thread
  static_assert(6 * (IX - 1) <= NT && 3 * IX <= NT, "one y1 column per thread");
  static_assert(2 * RB * IX + 6 * RB <= RB * NX, "pair 0 and the last column fit the exchange rows");
  PSG_TWIDDLES_REQUEST(P, NX, EPT, NT);
  PSG_TWIDDLES_READY(P);
  cpx<P> *ex = lds, *hs = lds + RB * NX;        // exchange rows (and pair 0), pairs 1 and 2 (then the products)
  cpx<P> *last = ex + 2 * RB * IX;
  const int nz = g.nz;
  // field f of the unit's rows
  auto rows = [&](int f) { return f < 2 ? ex + f * RB * IX : hs + (f - 2) * RB * IX; };
  const bool job = threadIdx.x < 6 * (IX - 1);
  cpx<P> r[RB], e[NE];
  auto request = [&](int un) {
    const int z = un % nz, t = un / nz, y2 = t % d.ra, m = t / d.ra;
    const int th = fresh(threadIdx.x), jf = th / (IX - 1), jk = th % (IX - 1);
    const cpx<P> *f0 = F + (long)m * 6 * d.fs + (y2 * nz + z) * d.kb;
    const cpx<P> *src = f0 + (long)(job ? jf : 0) * d.fs + (long)(jk / d.kb) * RB * d.pa + jk % d.kb;
#pragma unroll
    for (int k1 = 0; k1 < RB; k1++) r[k1] = job ? src[(long)k1 * d.pa] : cpx<P>{0, 0};
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int q = threadIdx.x + i * NT, qf = q / RB, qk = q % RB;
      e[i] = q < 6 * RB ? f0[(long)qf * d.fs + ((long)((IX - 1) / d.kb) * RB + qk) * d.pa + (IX - 1) % d.kb] : cpx<P>{0, 0};
    }
  };
  // XCD x = block % 8 takes one contiguous range of units, its blocks next to each other
  const int per = (units + 7) / 8, x = blockIdx.x % 8, slots = gridDim.x / 8;
  const int uend = (x + 1) * per < units ? (x + 1) * per : units;
  int un = x * per + blockIdx.x / 8;
  if (un < uend) request(un);
  for (; un < uend; un += slots) {
    const int z = un % nz, zr = un / nz, y2 = zr % d.ra, m = zr / d.ra;
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int q = threadIdx.x + i * NT;
      if (q < 6 * RB) last[q] = e[i];
    }
#pragma unroll
    for (int k1 = 1; k1 < RB; k1++) r[k1] = mulc(r[k1], twy[k1 * y2]);
    dft16<P, true>(r);
    if (job) {
      const int th = fresh(threadIdx.x), jf = th / (IX - 1), jk = th % (IX - 1);
      cpx<P> *o = rows(jf) + jk;
#pragma unroll
      for (int y1 = 0; y1 < RB; y1++) o[y1 * IX] = r[y1];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int q = threadIdx.x + i * NT, qf = q / RB, qy = q % RB;
      if (q < 6 * RB) {
        const cpx<P> wv = twy[y2 + d.ra * qy];
        cpx<P> a = last[qf * RB + RB - 1];
        for (int k1 = RB - 2; k1 >= 0; k1--) a = add(mulc(a, wv), last[qf * RB + k1]);
        rows(qf)[qy * IX + IX - 1] = a;
      }
    }
    if (un + slots < uend) request(un + slots);
    __syncthreads();
    P phys[6][EPT];
#pragma unroll
    for (int p = 0; p < 3; p++) {
      const int t = fresh(threadIdx.x), team = t / TP, j = t % TP;
      cpx<P> *tl = ex + team * NX;
      cpx<P> v[EPT];
      const cpx<P> *ra = rows(2 * p) + team * IX, *rb = rows(2 * p + 1) + team * IX;
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) {
        const int k = j + TP * mm;
        v[mm] = cpx<P>{0, 0};
        if (k < IX) {
          cpx<P> a = ra[k], b = rb[k];
          if (k == 0) a.y = b.y = 0;
          v[mm] = cpx<P>{a.x - b.y, a.y + b.x};
        } else if (k > NX - IX) {
          const cpx<P> a = ra[NX - k], b = rb[NX - k];
          v[mm] = cpx<P>{a.x + b.y, b.x - a.y};
        }
      }
      if (p == 0) __syncthreads();   // the exchange rows hold pair 0
      fft_pencil<P, NX, EPT, true, true, SW>(v, tl, j, 1, 0, tw);
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) { phys[2 * p][mm] = v[mm].x; phys[2 * p + 1][mm] = v[mm].y; }
    }
    P res[3][EPT];
#pragma unroll
    for (int mm = 0; mm < EPT; mm++) {
      const P in[6] = {phys[0][mm], phys[1][mm], phys[2][mm], phys[3][mm], phys[4][mm], phys[5][mm]};
      P out[3];
      ProdNS<P>{}(in, out);
      res[0][mm] = out[0]; res[1][mm] = out[1]; res[2][mm] = out[2];
    }
    __syncthreads();   // every row of pairs 1 and 2 is read
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int t = fresh(threadIdx.x), team = t / TP, j = t % TP;
      cpx<P> *tl = ex + team * NX;
      cpx<P> v[EPT];
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) v[mm] = cpx<P>{res[2 * q][mm], q == 0 ? res[1][mm] : (P)0};
      fft_pencil<P, NX, EPT, false, true, SW>(v, tl, j, 1, 0, tw);
      team_sync<true>();
#pragma unroll
      for (int mm = 0; mm < EPT; mm++) {
        const int k = j + TP * mm;
        if (k < IX || k > NX - IX) tl[lpos<SW>(k)] = v[mm];
      }
      team_sync<true>();
#pragma unroll 1
      for (int k = j; k < IX; k += TP) {
        cpx<P> A, B;
        split_pair(tl[lpos<SW>(k)], tl[lpos<SW>((NX - k) & (NX - 1))], A, B);
        hs[(2 * q * RB + team) * IX + k] = A;
        if (q == 0) hs[(RB + team) * IX + k] = B;
      }
    }
    __syncthreads();
    if (threadIdx.x < 3 * IX) {
      const int th = fresh(threadIdx.x), f = th / IX, kx = th % IX;
      cpx<P> o[RB];
#pragma unroll
      for (int y1 = 0; y1 < RB; y1++) o[y1] = hs[(f * RB + y1) * IX + kx];
      dft16<P, false>(o);
      cpx<P> *dst = G + ((long)m * 3 + f) * d.gs + (long)z * d.zp + y2 * RB * d.xq + kx;
#pragma unroll
      for (int k1 = 0; k1 < RB; k1++) dst[k1 * d.xq] = k1 ? mul(o[k1], twy[k1 * y2]) : o[0];
    }
    __syncthreads();
  }
}

inline bool split_len(int n) { return n == 32 || n == 64 || n == 128; }
// Grids whose tiles fit the LDS, with F and G of all members within a quarter
// of the 256 MB last-level cache, and the default kernel shapes (the others are
// those of the five pencil passes).  What the split saves is launches and their
// latency; its pieces of kb points cost more than the pencil passes' 128-byte
// ones once F and G come from HBM.  One step in us, pencil passes -> two kernels:
//   one context: FP64 32x128x128 108 -> 84, 64x128x128 132 -> 98, 128x128x64 129 -> 113;
//     FP32 64x128x128 x 2 148 -> 105, 128^3 138 -> 105
//   three at a time: FP64 32^3 25.6 -> 14.5, 64^3 37.6 -> 22.7, 64^3 x 4 (52 MB)
//     87.0 -> 54.4, 128x128x64 (51 MB) 86.2 -> 80.8; FP32 128^3 98 -> 88
// Beyond the line it depends on what else runs: at about 100 MB a context that has
// the cache to itself still gains (FP64 128^3 206 -> 183, FP32 128x128x64 x 4
// 242 -> 229), three of them lose (167 -> 177, 196 -> 214) or, with short rows, not
// (64^3 x 8 188 -> 137).  A context cannot know its neighbours, and no grid within
// the line is slower either way, so the line stands where both agree.
inline bool split_usable(const Ctx *c) {
  if (c->g.dim != 3 || c->cfg.flavour == PSG_BOUS3D || !split_len(c->g.nx) || !split_len(c->g.ny) || !split_len(c->g.nz))
    return false;
  if (c->xvar || c->zvar || c->slvar) return false;
  const Split d = Split::of(c);
  const size_t b = c->cfg.precision == PSG_FP32BULK ? 8 : 16;
  return (6 * d.fs + 3 * d.gs) * (size_t)c->batch * b <= (size_t)64 << 20;
}

// st: the working copies; phase 0 (and the first stage's load) reads the first
// and writes the second, phase 1 the other way round
template <typename P> static int launch_zsplit(Ctx *c, cpx<P> *st, SplitUpd u) {
  const Grid &g = c->g;
  const Split d = Split::of(c);
  cpx<P> *st2 = st + 3 * d.nkts * c->batch;
  auto go = [&](auto k, int nt, size_t lds) -> int {
    PSG_HIP(lds_attr(k, lds));
    hipLaunchKernelGGL(k, dim3(d.ng, SPLIT_RB, c->batch), dim3(nt), lds, c->stream, (const cpx<P> *)c->bufC,
                       (cpx<P> *)c->bufB, (const cpx<P> *)(u.phase ? st2 : st), u.phase ? st : st2, (cpx<P> *)c->rh,
                       (const double *)c->wnuzn, (const double *)c->wnu1, (const int8_t *)c->wmask, g, d, twp<P>(c, 2), u);
    PSG_HIP(hipGetLastError());
    return 0;
  };
  auto len = [&](auto ra) -> int {
    constexpr int RA = decltype(ra)::value;
    switch (g.nz) {
#define PSG_ZS(NZ) case NZ: return go(k_zsplit<P, NZ, RA>, ZShape<P, NZ, RA>::NT, ZShape<P, NZ, RA>::lds());
      PSG_ZS(32) PSG_ZS(64) PSG_ZS(128)
#undef PSG_ZS
    }
    set_error("split z kernel: length %d", g.nz);
    return PSG_EINVAL;
  };
  switch (d.ra) {
    case 2: return len(std::integral_constant<int, 2>{});
    case 4: return len(std::integral_constant<int, 4>{});
    case 8: return len(std::integral_constant<int, 8>{});
  }
  set_error("split z kernel: NY %d", g.ny);
  return PSG_EINVAL;
}

template <typename P> static int launch_xysplit(Ctx *c) {
  const Grid &g = c->g;
  const Split d = Split::of(c);
  const int units = g.nz * d.ra * c->batch;
  auto go = [&](auto k, int nt, size_t lds) -> int {
    PSG_HIP(lds_attr(k, lds));
    // as many blocks as the CUs hold: by LDS, and by registers 8 wavefronts in FP64, 16 in FP32
    const int waves = (nt + 63) / 64, bl = (int)(163840 / lds), bw = (sizeof(P) == 8 ? 8 : 16) / waves;
    const int bpc = bl < bw ? bl : bw;
    int nb = c->cus * (bpc < 1 ? 1 : bpc);
    if (nb > units) nb = units;
    nb = (nb + 7) / 8 * 8;
    hipLaunchKernelGGL(k, dim3(nb), dim3(nt), lds, c->stream, (const cpx<P> *)c->bufB, (cpx<P> *)c->bufC, g, d,
                       twp<P>(c, 0), twp<P>(c, 1), units);
    PSG_HIP(hipGetLastError());
    return 0;
  };
  switch (g.nx) {
#define PSG_XS(NX) case NX: return go(k_xysplit<P, NX>, XShape<NX>::NT, XShape<NX>::template lds<P>());
    PSG_XS(32) PSG_XS(64) PSG_XS(128)
#undef PSG_XS
  }
  set_error("split xy kernel: length %d", g.nx);
  return PSG_EINVAL;
}

// Heun steps of the working copy st (layout Split::at).  F holds the inverse
// transforms of the state before every xy kernel: the first call of a run
// makes them from the state, each update but a run's last makes the next stage's.
// (runs of one step, one context: 64x128x128 FP32 133 us with the unused transforms,
// 120 without, 64^3 FP64 84 and 79)
template <typename P> int split_run(Ctx *c, cpx<P> *st, int nsteps, bool first, bool last) {
  const Grid &g = c->g;
  const bool euler = c->cfg.flavour == PSG_EULER3D;
  SplitUpd u{0, 0, euler ? 1 : 0, 1, 0, c->cfg.dt, Force{c->cfg.force, c->cfg.kf, c->cfg.ampfor}};
  const long b = sizeof(cpx<P>), Y = (long)g.iktx * g.ny * g.nz;
  if (first) PSG_TRY(launch_zsplit<P>(c, st, u));
  u.fwd = 1;
  u.umask = 0;
  for (int nt = 0; nt < nsteps; nt++)
    for (int phase = 0; phase < 2; phase++) {
      prof_begin(c, "xy", 9 * Y * b * c->batch);
      PSG_TRY(launch_xysplit<P>(c));
      prof_end(c);
      u.phase = phase;
      u.last = last && phase == 1 && nt == nsteps - 1;
      prof_begin(c, "z_update", (9 * Y * b + 9 * g.nkt * b + 17 * g.nkt) * c->batch);
      PSG_TRY(launch_zsplit<P>(c, st, u));
      prof_end(c);
    }
  return 0;
}

extern template int split_run<float>(Ctx *, cpx<float> *, int, bool, bool);
extern template int split_run<double>(Ctx *, cpx<double> *, int, bool, bool);

}  // namespace psg
