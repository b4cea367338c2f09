// sac_tile.h -- an RK stage's x and y work and its register update on 16 x 16
// tiles staged in LDS: whole stages of 2-D grids and patches, and the last
// pass of 3-D stages.
//
// The work per mesh cell is that of the line tiles (sac_line.h) along x and
// y with the same arithmetic per value -- 4th-order flux divergence with the
// background energy terms (centdiff4, src/vaccd.t:35-70), Powell's sources,
// setnu for the 2*ndim+1 variables of each axis (src/vacusr.viscosity.t:
// 224-455), the hyperdiffusion line terms and the cross-term factors
// (src/vacusr.viscosity.t:2-221) -- then the cross terms between x and y,
//   m_1 += d_x(rho_t Tm_{1,0}), e += d_x(m_1 Tm_{1,0}), b_1 -= d_x(Tb_{1,0}), e -= d_x(b_1 Tb_{1,0})
//   m_0 += d_y(rho_t Tm_{0,1}), e += d_y(m_0 Tm_{0,1}), b_0 -= d_y(Tb_{0,1}), e -= d_y(b_0 Tb_{0,1})
// (central differences, zero at a non-periodic edge, T = 0 outside the
// mesh), the rate of other kernels (f.R: the z work, resistivity), gravity,
// and the update with the cmax of the result (update_cells).  Neither the
// rate of x and y nor T_{0,1}, T_{1,0} leave the CU.
//
// Schedule.  A block of 512 threads owns a tile of one plane.  Each thread
// loads and evaluates one point of the 22 x 22 around it (the corners that
// nothing reads left out): 13 fields, coalesced along x, into setnu's q
// values, rho_t, m and the x and y fluxes in LDS.  After one barrier the
// lower four wavefronts do the x work of the 256 cells and the upper four
// the y work at the same time; the y rates and the factors are handed over
// through the space of the fluxes, and the lower four finish the cells.
// What bounds such a tile is latency: its FP64 chains are long, and its LDS
// (75 KB in 3-D) lets two blocks into a CU.  Two axes on twice the
// wavefronts halve the chain and give four wavefronts per SIMD instead of
// two.  A 2-D stage of 501 x 299 cells was an x and a y line kernel and an
// update, 19.8 + 16.3 + 15.5 us; here 21.3.  512 patches (4.8 M cells): 0.996
// ms before, 0.65 now.  Reading the cell's background, c_tot and dx before
// the points, and the base register while the axes are handed over, is 15 %
// of that.  In 3-D a tile is bound by both its VALU issue (2350 instructions
// per 64 cells, 60 % of the time at the 2.07 GHz the card runs FP64 work at)
// and the waits between its barriers: 128 VGPRs keep the four wavefronts per
// SIMD (144 let in one block per CU: 2.07 -> 2.78 ms at 256^3).
//
// Grid edges follow the line tiles: a point beyond the grid along x (y) is
// the mirror cell 6 inward (src/vacusr.viscosity.t:378-400), read only by
// the x (y) work of cells in the grid.
#pragma once
#include "sac_device.h"

namespace sac {
namespace tile {

constexpr int TX = 16, TY = 16, HALO = 3;
constexpr int PX = TX + 2 * HALO, PY = TY + 2 * HALO;  // 22 x 22 points
constexpr int NC = TX * TY;  // cells, and threads of each axis
constexpr int NT = 2 * NC;

// LDS layout (elements).  q of rho', thermal energy, v_l (and b_2 in 3-D) on
// all 22 x 22 points; b_0, which only the y work takes differences of, on
// columns -1..16, b_1 on rows -1..16; rho_t and m_l on -1..16 both ways; the
// x fluxes on columns -2..17 of the tile's rows, the y fluxes on rows -2..17
// of its columns.  The flux of b_K along K is zero and has no slot; Powell's
// sources keep b_K + bg_K in one (slot NE-1).
//
// In FP64, 16 lanes read one tile row of 16 doubles (128 bytes: every bank
// once).  In FP32 a half-wave (32 lanes, served together) reads two tile
// rows; they are rows r and r+8 (see cell_row), and every pitch is 2 (mod 4)
// floats, so the two rows' reads fall 8 * pitch = 16 (mod 32) banks apart and
// never share a bank.
template <int NDIM, int NDIR, typename C, bool DIVB>
struct Lay {
  static constexpr bool F32 = sizeof(C) == 4;
  static constexpr int NE = 2 + 2 * NDIR;
  static constexpr int QP = PX;                      // pitch of the full planes
  static constexpr int NFULL = 2 + NDIM + (NDIM == 3 ? 1 : 0);
  static constexpr int SP = TX + 2;                  // pitch of the 18-wide planes
  static constexpr int B0 = NFULL * PY * QP;         // [22][18]
  static constexpr int B1 = B0 + PY * SP;            // [18][22]
  static constexpr int RT = B1 + (TY + 2) * QP;      // [18][18]
  static constexpr int M0 = RT + (TY + 2) * SP;      // [NDIM][18][18]
  static constexpr int FXP = F32 ? TX + 6 : TX + 4;  // pitch of the x fluxes
  static constexpr int FYP = F32 ? TX + 2 : TX;      // and of the y fluxes
  static constexpr int NF = DIVB ? NE : NE - 1;
  static constexpr int FX = M0 + NDIM * (TY + 2) * SP;  // [NF][16][FXP]
  static constexpr int FY = FX + NF * TY * FXP;         // [NF][20][FYP]
  static constexpr int END = FY + NF * (TY + 4) * FYP;
  // after the fluxes are read, in their place
  static constexpr int RY = FX;                     // y rates [NE][16][FYP]
  static constexpr int T01 = RY + NE * TY * FYP;    // Tm_{0,1}, Tb_{0,1}: [2][18][FYP], rows -1..16
  static constexpr int T10 = T01 + 2 * (TY + 2) * FYP;  // Tm_{1,0}, Tb_{1,0}: [2][16][18], cols -1..16
  static_assert(T10 + 2 * TY * SP <= END, "the exchange fits the space of the fluxes");
};

template <int NDIM, int NDIR, typename C, bool DIVB>
struct Smem {
  C v[Lay<NDIM, NDIR, C, DIVB>::END];
};

template <bool B>
struct Bool {
  static constexpr bool value = B;
};

// flux slot of field n along K
__host__ __device__ constexpr int fslot(int ndir, int K, int n) {
  return n > 2 + ndir + K ? n - 1 : n;
}

// tile row of thread t (0..255) of its axis: t / 16 in FP64; in FP32 lanes
// 0-15, 16-31, 32-47, 48-63 of wave w take rows 2w, 2w+8, 2w+1, 2w+9
template <typename C>
__device__ __forceinline__ int cell_row(int t) {
  if constexpr (sizeof(C) == 4)
    return 2 * (t >> 6) + ((t >> 5) & 1) + 8 * ((t >> 4) & 1);
  else
    return t / TX;
}

// tiles of a plane along x and y
__host__ __device__ inline int ntx(const GridDesc& g) {
  return (g.Mhi[0] - g.Mlo[0] + 1 + TX - 1) / TX;
}
__host__ __device__ inline int nty(const GridDesc& g) {
  return (g.Mhi[1] - g.Mlo[1] + 1 + TY - 1) / TY;
}
__host__ __device__ inline long long nblocks(const GridDesc& g) {
  return (long long)ntx(g) * nty(g) * (g.Mhi[2] - g.Mlo[2] + 1);
}
// 32-bit byte offsets reach the 22 rows of a tile's points
__host__ __device__ inline bool rows_fit(long long pitch) { return pitch < (1LL << 32) / (8 * PY); }

// One cell's line terms along axis K (0 or 1) from the staged plane, as in
// line_tile: flux divergence, background energy terms, Powell's sources,
// setnu face ratios, hyperdiffusion line terms; returns the factors
// T_{K,1-K} in Tm, Tb.  fget(s, d) is flux slot s at offset d along K,
// qget(p, d) the q of setnu's variable p of axis K (rho', thermal energy,
// v_0.., b_l (l != K)), rget(d) rho_t, mget(l, d) m_l.  EDGE: some cell of
// the wavefront may lie within two cells of an end of the mesh along K, where
// terms are replaced by zero; the other wavefronts go without those selects
// (about 60 of the 700 instructions of an axis).
template <int NDIM, int NDIR, int K, typename S, typename C, bool DIVB, bool EDGE, typename FG,
          typename QG, typename RG, typename MG>
__device__ __forceinline__ void cell_axis(const FinalArgs& f, const GridDesc& g, long long icell,
                                          const Pt<NDIR, C>& pbg, C (&R)[2 + 2 * NDIR], int c,
                                          C dxk, C idx, C inv12, C ctk,
                                          bool valid, C& numax, FG fget, QG qget, RG rget, MG mget,
                                          C& Tm, C& Tb) {
  constexpr int NE = 2 + 2 * NDIR, NP = 2 * NDIM + 1;
  const long long fs = g.fs;
  const double* __restrict__ Bg = f.bg;
  const int MloK = g.Mlo[K], MhiK = g.Mhi[K];
  {
    const bool fluxc = !EDGE || (c >= MloK + 2 && c <= MhiK - 2);
#pragma unroll
    for (int n = 0; n < NE; n++) {
      if (n == 2 + NDIR + K) {
        R[n] = 0;
        continue;
      }
      const int s = fslot(NDIR, K, n);
      C E1, e2;
      const C D1 = two_diff(fget(s, 1), fget(s, -1), E1);
      const C D2 = two_diff(fget(s, 2), fget(s, -2), e2);
      R[n] = ((D2 - (C)8 * D1) + (e2 - (C)8 * E1)) * inv12;
    }
    const C pTb0 = (C)ptotal_bg<NDIR, C>(pbg, f.gamma);
    const C bgk = (C)pbg.bg[K];
    C re = 0;
#pragma unroll
    for (int l = 0; l < NDIM; l++) {
      const C dv1 = qget(2 + l, 1) - qget(2 + l, -1);
      const C dv2 = qget(2 + l, 2) - qget(2 + l, -2);
      const C Dv = -(dv2 - (C)8 * dv1) * inv12;
      if (l == K) re -= Dv * pTb0;
      re += bgk * (C)pbg.bg[l] * Dv;
    }
    R[1 + NDIR] += re;
#pragma unroll
    for (int n = 0; n < NE; n++) R[n] = fluxc ? R[n] : (C)0;
    // Powell's div B sources (see line_tile)
    if (DIVB && fluxc && valid) {
      const S* __restrict__ Wf = (const S*)f.wct;
      const C D1b = fget(NE - 1, 1) - fget(NE - 1, -1);
      const C D2b = fget(NE - 1, 2) - fget(NE - 1, -2);
      const C gK = -((D2b - (C)8 * D1b) * inv12);
      const double rt = (double)Wf[icell] + Bg[fs + icell];
      double sm = 0.0;
#pragma unroll
      for (int cd = 0; cd < NDIR; cd++) {
        const double m = (double)Wf[(1 + cd) * fs + icell];
        const double bt = (double)Wf[(2 + NDIR + cd) * fs + icell] + Bg[(2 + cd) * fs + icell];
        R[1 + cd] -= (C)bt * gK;
        R[2 + NDIR + cd] -= (C)(m / rt) * gK;
        sm = (cd == 0) ? m * bt : sm + m * bt;
      }
      R[1 + NDIR] -= (C)(sm / rt) * gK;
    }
  }
  if (f.visc_on) {
#pragma clang fp contract(off)
    const bool z1 =
        EDGE && ((c == MloK && !g.per_lo[K]) || (c == MhiK && !g.per_hi[K]));
    C nmax = 0;
    const HyperAxis<C> ha(ctk, dxk, idx);
    const C rt0 = rget(0), rhoL = rt0 + rget(-1), rhoR = rget(1) + rt0;  // twice the means
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const bool vel = p >= 2 && p < 2 + NDIM;
      C q[7], ratL, ratR, tL, tR;
#pragma unroll
      for (int s = 0; s < 7; s++) q[s] = qget(p, s - 3);
      face_pair<C>(q, ratL, ratR);
      const C T = hyper_faces<C>(q, vel ? ha.kv : ha.ks, ratL, ratR, z1, tL, tR, nmax);
      if (p == 0) {
        R[0] = fma_(tR - tL, ha.i2, R[0]);
      } else if (p == 1) {
        R[1 + NDIR] = fma_(tR - tL, ha.i2, R[1 + NDIR]);
      } else if (vel) {
        const int l = p - 2;
        const C m0 = mget(l, 0), mL = m0 + mget(l, -1), mR = mget(l, 1) + m0;
        const C f = (l == K) ? ha.i2h : ha.i2q;  // the i==k branch runs twice for l==k
        R[1 + l] = fma_(fma_(rhoR, tR, -(rhoL * tL)), f, R[1 + l]);
        R[1 + NDIR] = fma_(fma_(mR, tR, -(mL * tL)), f, R[1 + NDIR]);
        if (l == 1 - K) Tm = T * ha.it;
      } else {
        const int n = p - 2 - NDIM;
        const int lb = (n < K) ? n : n + 1;
        const C BL = q[3] + q[2], BR = q[4] + q[3];
        R[2 + NDIR + lb] = fma_(tR - tL, ha.i2, R[2 + NDIR + lb]);
        R[1 + NDIR] = fma_(fma_(BR, tR, -(BL * tL)), ha.i2h, R[1 + NDIR]);
        if (lb == 1 - K) Tb = (C)2 * T * ha.it;
      }
    }
    numax = valid ? ha.nu(nmax) : (C)0;
  }
}

// The factor T_{K,1-K} of one halo cell for one of its two variables (which
// 0: the velocity, 1: the field), from q[0..6] along K; the same arithmetic
// as cell_axis.
template <typename C>
__device__ __forceinline__ C cross_factor(const C (&q)[7], int which, bool z1, C dxk, C idx,
                                          C ctk) {
#pragma clang fp contract(off)
  const HyperAxis<C> ha(ctk, dxk, idx);
  C ratL, ratR, tL, tR, nmax = 0;
  face_pair<C>(q, ratL, ratR);
  const C T = hyper_faces<C>(q, which ? ha.ks : ha.kv, ratL, ratR, z1, tL, tR, nmax);
  return which ? (C)2 * T * ha.it : T * ha.it;
}

// The stage of the tile with its first cell at grid column x0 and row y0 of
// plane z.  True for the threads that stored a cell (at c).  Off: the type of
// the points' byte offsets (see rows_fit).
template <int NDIM, int NDIR, typename S, typename C, bool RK4L, bool DIVB, typename Off = unsigned>
__device__ __forceinline__ bool stage_tile(const FinalArgs& f, const GridDesc& g, int x0, int y0,
                                           int z, C* __restrict__ sm, C& numax,
                                           double (&redv)[2 * NDIM], int (&c)[3]) {
  using L = Lay<NDIM, NDIR, C, DIVB>;
  constexpr int NE = L::NE;
  const long long fs = g.fs;
  const long long zoff = (long long)z * g.st[2];
  const int tid = (int)threadIdx.x;
  const bool xgrp = tid < NC;  // uniform over a wavefront
  const int t = tid & (NC - 1);
  const int tx = t % TX, ty = cell_row<C>(t);

  // ---- the thread's cell ----
  const int cx = x0 + tx, cy = y0 + ty;
  const bool valid = cx >= g.Mlo[0] && cx <= g.Mhi[0] && cy <= g.Mhi[1];
  const int cxc = (cx > g.G[0] - 1) ? g.G[0] - 1 : cx;
  const int cyc = (cy > g.G[1] - 1) ? g.G[1] - 1 : cy;
  const long long icell = zoff + (long long)cyc * g.st[1] + cxc;
  // the cell's widths: of the wavefront's axis, and half over both
  const double* dxc = xgrp ? f.dx[0] + cxc : f.dx[1] + cyc;
  const C dxk = (C)dxc[0], idx = (C)dxc[kDxInv * f.dxs], inv12 = (C)dxc[kDxInv12 * f.dxs];
  const C hx = (C)f.dx[0][kDxHalf * f.dxs + cxc], hy = (C)f.dx[1][kDxHalf * f.dxs + cyc];
  const C ctk = f.visc_on ? (C)red_get(f.ctot_src, xgrp ? 0 : 1) : (C)0;
  Pt<NDIR, C> own;  // the cell's background
  own.eb = f.bg[icell];
  own.rhob = f.bg[fs + icell];
#pragma unroll
  for (int cd = 0; cd < NDIR; cd++) own.bg[cd] = f.bg[(2 + cd) * fs + icell];
  const bool xlo = !g.per_lo[0], xhi = !g.per_hi[0], ylo = !g.per_lo[1], yhi = !g.per_hi[1];

  // ---- one point per thread: the tile's cells, then the halo ----
  {
    int ix, iy;
    bool point = true, fx = true, fy = true;
    if (xgrp) {
      ix = tx + HALO;
      iy = ty + HALO;
    } else if (t < 96) {  // columns -3..-1 and 16..18 of the tile's rows
      const int r = t / 6, k = t - 6 * r;
      ix = k < 3 ? k : k + TX;
      iy = r + HALO;
      fy = false;
      fx = ix >= 1 && ix <= PX - 2;
    } else if (t < 192) {  // rows -3..-1 and 16..18 of its columns
      const int k = (t - 96) / TX;
      ix = (t - 96) % TX + HALO;
      iy = k < 3 ? k : k + TY;
      fx = false;
      fy = iy >= 1 && iy <= PY - 2;
    } else {  // of the corners what the factors of the halo rows and columns take
      const int u = t - 192;
      fx = fy = false;
      point = u < 20;
      if (u < 12) {
        const int k = u % 6;
        ix = k < 3 ? k : k + TX;
        iy = u < 6 ? HALO - 1 : TY + HALO;
      } else {
        const int k = u & 3;
        ix = u < 16 ? HALO - 1 : TX + HALO;
        iy = k < 2 ? k : k + TY + 2;
      }
    }
    if (point) {
      int gx = x0 - HALO + ix, gy = y0 - HALO + iy;
      // mirror layer beyond the grid (used only along its own axis)
      if (gx < 0) gx = g.Mlo[0] + 3;
      if (gx > g.G[0] - 1) gx = g.Mhi[0] - 3;
      if (gy < 0) gy = g.Mlo[1] + 3;
      if (gy > g.G[1] - 1) gy = g.Mhi[1] - 3;
      // offsets from the tile's first row (a mirrored row lies in the tile too)
      const int yb = y0 > HALO ? y0 - HALO : 0;
      const long long ob0 = zoff + yb * g.st[1];
      const Off i = (Off)(gy - yb) * (Off)g.st[1] + (Off)gx;
      const char* __restrict__ Wp = (const char*)((const S*)f.wct + ob0);
      const char* __restrict__ Bp = (const char*)(f.bg + ob0);
      const Off ow = i * (Off)sizeof(S), ob = i * (Off)8;
      auto wv = [&](int n) { return (C) * (const S*)(Wp + (size_t)n * fs * sizeof(S) + ow); };
      auto bv = [&](int n) { return *(const double*)(Bp + (size_t)n * fs * 8 + ob); };
      Pt<NDIR, C> p;
      p.rho = wv(0);
#pragma unroll
      for (int cd = 0; cd < NDIR; cd++) p.m[cd] = wv(1 + cd);
      p.e = wv(1 + NDIR);
#pragma unroll
      for (int cd = 0; cd < NDIR; cd++) p.b[cd] = wv(2 + NDIR + cd);
      p.eb = bv(0);
      p.rhob = bv(1);
#pragma unroll
      for (int cd = 0; cd < NDIR; cd++) p.bg[cd] = bv(2 + cd);
      const double rtd = (double)p.rho + p.rhob;
      const double inv = recip<C>(rtd);
      if (fx || fy) {
        const FluxPt<C> fc = flux_common<NDIR, C>(p, f.gamma, inv);
        if (fx) {
          C F[NE];
          flux_axis<NDIR, C>(p, fc, 0, F);
          C* o = sm + L::FX + (iy - HALO) * L::FXP + ix - 1;
#pragma unroll
          for (int n = 0; n < NE; n++)
            if (n != 2 + NDIR) o[fslot(NDIR, 0, n) * TY * L::FXP] = F[n];
          if constexpr (DIVB) o[(NE - 1) * TY * L::FXP] = (C)((double)p.b[0] + p.bg[0]);
        }
        if (fy) {
          C F[NE];
          flux_axis<NDIR, C>(p, fc, 1, F);
          C* o = sm + L::FY + (iy - 1) * L::FYP + ix - HALO;
#pragma unroll
          for (int n = 0; n < NE; n++)
            if (n != 3 + NDIR) o[fslot(NDIR, 1, n) * (TY + 4) * L::FYP] = F[n];
          if constexpr (DIVB) o[(NE - 1) * (TY + 4) * L::FYP] = (C)((double)p.b[1] + p.bg[1]);
        }
      }
      {
#pragma clang fp contract(off)
        double sb = 0.0, smm = 0.0;
#pragma unroll
        for (int cd = 0; cd < NDIR; cd++) {
          const double mc = (double)p.m[cd], bc = (double)p.b[cd];
          sb += bc * bc;
          smm += mc * mc;
        }
        C* q = sm + iy * L::QP + ix;
        q[0] = p.rho;
        q[PY * L::QP] = (C)((double)p.e - 0.5 * (sb + smm * inv));
#pragma unroll
        for (int l = 0; l < NDIM; l++) q[(2 + l) * PY * L::QP] = p.m[l] * (C)inv;
        if constexpr (NDIM == 3) q[5 * PY * L::QP] = p.b[2];
        const bool inx = ix >= HALO - 1 && ix <= TX + HALO, iny = iy >= HALO - 1 && iy <= TY + HALO;
        if (inx) sm[L::B0 + iy * L::SP + ix - (HALO - 1)] = p.b[0];
        if (iny) sm[L::B1 + (iy - (HALO - 1)) * L::QP + ix] = p.b[1];
        if (inx && iny) {
          C* r = sm + L::RT + (iy - (HALO - 1)) * L::SP + ix - (HALO - 1);
          r[0] = (C)rtd;
#pragma unroll
          for (int l = 0; l < NDIM; l++) r[(1 + l) * (TY + 2) * L::SP] = p.m[l];
        }
      }
    }
  }

  const C* qc = sm + (ty + HALO) * L::QP + tx + HALO;       // full planes
  const C* rc = sm + L::RT + (ty + 1) * L::SP + tx + 1;     // 18 x 18 planes
  const C* b0 = sm + L::B0 + (ty + HALO) * L::SP + tx + 1;  // b_0
  const C* b1 = sm + L::B1 + (ty + 1) * L::QP + tx + HALO;  // b_1
  constexpr int QA = PY * L::QP, RA = (TY + 2) * L::SP;     // array strides
  __syncthreads();

  C R[1][NE], Tm = 0, Tb = 0, Th = 0;
  if (xgrp) {
    const C* fc = sm + L::FX + ty * L::FXP + tx + 2;
    auto work = [&](auto edge) {
      cell_axis<NDIM, NDIR, 0, S, C, DIVB, decltype(edge)::value>(
          f, g, icell, own, R[0], cx, dxk, idx, inv12, ctk, valid, numax,
          [&](int s, int d) { return fc[s * TY * L::FXP + d]; },
          [&](int p, int d) {
            return p < 2 + NDIM ? qc[p * QA + d] : (p == 2 + NDIM ? b1[d] : qc[5 * QA + d]);
          },
          [&](int d) { return rc[d]; }, [&](int l, int d) { return rc[(1 + l) * RA + d]; }, Tm,
          Tb);
    };
    if (x0 < g.Mlo[0] + 2 || x0 + TX - 1 > g.Mhi[0] - 2) work(Bool<true>{});
    else work(Bool<false>{});
    // T_{0,1} of the rows below and above the tile, one variable per lane
    if (f.visc_on && t >= NC - 64) {
      const int hc = t & 15, hr = (t & 16) ? TY : -1, which = (t >> 5) & 1;
      const int hcx = x0 + hc, hcxc = (hcx > g.G[0] - 1) ? g.G[0] - 1 : hcx;
      const double* dh = f.dx[0] + hcxc;
      const C* a = which ? sm + L::B1 + (hr + 1) * L::QP + hc + HALO
                         : sm + 3 * QA + (hr + HALO) * L::QP + hc + HALO;
      C q[7];
#pragma unroll
      for (int s = 0; s < 7; s++) q[s] = a[s - 3];
      const bool z1 = (hcx == g.Mlo[0] && xlo) || (hcx == g.Mhi[0] && xhi);
      Th = cross_factor<C>(q, which, z1, (C)dh[0], (C)dh[kDxInv * f.dxs], ctk);
    }
  } else {
    const C* fc = sm + L::FY + (ty + 2) * L::FYP + tx;
    auto work = [&](auto edge) {
      cell_axis<NDIM, NDIR, 1, S, C, DIVB, decltype(edge)::value>(
          f, g, icell, own, R[0], cy, dxk, idx, inv12, ctk, valid, numax,
          [&](int s, int d) { return fc[(s * (TY + 4) + d) * L::FYP]; },
          [&](int p, int d) {
            return p < 2 + NDIM ? qc[p * QA + d * L::QP]
                                : (p == 2 + NDIM ? b0[d * L::SP] : qc[5 * QA + d * L::QP]);
          },
          [&](int d) { return rc[d * L::SP]; },
          [&](int l, int d) { return rc[(1 + l) * RA + d * L::SP]; }, Tm, Tb);
    };
    if (y0 < g.Mlo[1] + 2 || y0 + TY - 1 > g.Mhi[1] - 2) work(Bool<true>{});
    else work(Bool<false>{});
    // T_{1,0} of the columns left and right of the tile
    if (f.visc_on && t >= NC - 64) {
      const int hr = t & 15, hc = (t & 16) ? TX : -1, which = (t >> 5) & 1;
      const int hcy = y0 + hr, hcyc = (hcy > g.G[1] - 1) ? g.G[1] - 1 : hcy;
      const double* dh = f.dx[1] + hcyc;
      const C* a = which ? sm + L::B0 + (hr + HALO) * L::SP + hc + 1
                         : sm + 2 * QA + (hr + HALO) * L::QP + hc + HALO;
      const int st = which ? L::SP : L::QP;
      C q[7];
#pragma unroll
      for (int s = 0; s < 7; s++) q[s] = a[(s - 3) * st];
      const bool z1 = (hcy == g.Mlo[1] && ylo) || (hcy == g.Mhi[1] && yhi);
      Th = cross_factor<C>(q, which, z1, (C)dh[0], (C)dh[kDxInv * f.dxs], ctk);
    }
  }
  // The rate of other kernels, the z factors of the cell's neighbours and the
  // base register: on their way while the axes are handed over.
  C Rin[NE], Tz[8];
  S base[NE];
  if (xgrp) {
#pragma unroll
    for (int n = 0; n < NE; n++) base[n] = ((const S*)f.base)[n * fs + icell];
  }
  if (xgrp && f.R) {
#pragma unroll
    for (int n = 0; n < NE; n++) Rin[n] = (C)((const S*)f.R)[n * fs + icell];
  }
  if constexpr (NDIM == 3) {
    if (xgrp && f.visc_on) {
      // in-grid indices: the neighbours of a mesh cell
      const long long ex = valid ? 1 : 0, ey = valid ? g.st[1] : 0;
      const S* __restrict__ T0 = (const S*)f.T + (long long)cross_index(NDIM, 2, 0) * fs + icell;
      const S* __restrict__ T1 = (const S*)f.T + (long long)cross_index(NDIM, 2, 1) * fs + icell;
      Tz[0] = (C)T0[ex], Tz[1] = (C)T0[-ex], Tz[2] = (C)T0[fs + ex], Tz[3] = (C)T0[fs - ex];
      Tz[4] = (C)T1[ey], Tz[5] = (C)T1[-ey], Tz[6] = (C)T1[fs + ey], Tz[7] = (C)T1[fs - ey];
    }
  }
  __syncthreads();  // the fluxes are read; their space takes the exchange
  if (xgrp) {
    sm[L::T01 + (ty + 1) * L::FYP + tx] = Tm;
    sm[L::T01 + ((TY + 2) + ty + 1) * L::FYP + tx] = Tb;
    if (t >= NC - 64)
      sm[L::T01 + (((t >> 5) & 1) * (TY + 2) + ((t & 16) ? TY + 1 : 0)) * L::FYP + (t & 15)] = Th;
  } else {
#pragma unroll
    for (int n = 0; n < NE; n++) sm[L::RY + (n * TY + ty) * L::FYP + tx] = R[0][n];
    sm[L::T10 + ty * L::SP + tx + 1] = Tm;
    sm[L::T10 + (TY + ty) * L::SP + tx + 1] = Tb;
    if (t >= NC - 64)
      sm[L::T10 + (((t >> 5) & 1) * TY + (t & 15)) * L::SP + ((t & 16) ? TX + 1 : 0)] = Th;
  }
  __syncthreads();
  if (!xgrp || !valid) return false;

#pragma unroll
  for (int n = 0; n < NE; n++) R[0][n] = R[0][n] + sm[L::RY + (n * TY + ty) * L::FYP + tx];
  if (f.R) {
#pragma unroll
    for (int n = 0; n < NE; n++) R[0][n] = R[0][n] + Rin[n];
  }
  if (f.visc_on) {
    // Cross terms with derivatives along l of the factors made along k.  The
    // factors of the z lines are zero outside the mesh in memory (never
    // written there), the tile's own are selected at the ends of the mesh.
    const C* t10 = sm + L::T10 + ty * L::SP + tx + 1;
    const C* t01 = sm + L::T01 + (ty + 1) * L::FYP + tx;
    auto cross = [&](auto ends) {
#pragma clang fp contract(off)
      constexpr bool E = decltype(ends)::value;
#pragma unroll
      for (int l = 0; l < 2; l++) {
        const int cl = (l == 0) ? cx : cy;
        const bool edge = (l == 0) ? ((cx == g.Mlo[0] && xlo) || (cx == g.Mhi[0] && xhi))
                                   : ((cy == g.Mlo[1] && ylo) || (cy == g.Mhi[1] && yhi));
        const C h = (l == 0) ? hx : hy;
        const bool inP = cl + 1 <= g.Mhi[l], inM = cl - 1 >= g.Mlo[l];
        const int rs = (l == 0) ? 1 : L::SP;  // neighbour along l in the 18-wide planes
        const int qs = (l == 0) ? 1 : L::QP;
        const C rtp = rc[rs], rtm = rc[-rs];
#pragma unroll
        for (int k = 0; k < NDIM; k++) {
          if (k == l) continue;
          C Tmp, Tmm, Tbp, Tbm, bkp, bkm;
          if (k == 2) {
            Tmp = Tz[4 * l], Tmm = Tz[4 * l + 1], Tbp = Tz[4 * l + 2], Tbm = Tz[4 * l + 3];
            bkp = qc[5 * QA + qs], bkm = qc[5 * QA - qs];
          } else if (l == 0) {
            Tmp = t10[1], Tmm = t10[-1], Tbp = t10[TY * L::SP + 1], Tbm = t10[TY * L::SP - 1];
            bkp = b1[1], bkm = b1[-1];
          } else {
            Tmp = t01[L::FYP], Tmm = t01[-L::FYP];
            Tbp = t01[(TY + 3) * L::FYP], Tbm = t01[(TY + 1) * L::FYP];
            bkp = b0[L::SP], bkm = b0[-L::SP];
          }
          if constexpr (E) {
            if (k < 2) {
              Tmp = inP ? Tmp : (C)0, Tmm = inM ? Tmm : (C)0;
              Tbp = inP ? Tbp : (C)0, Tbm = inM ? Tbm : (C)0;
            }
          }
          const C mkp = rc[(1 + k) * RA + rs], mkm = rc[(1 + k) * RA - rs];
          const C dm = fma_(rtp, Tmp, -(rtm * Tmm)) * h;
          const C de1 = fma_(mkp, Tmp, -(mkm * Tmm)) * h;
          const C db = (Tbp - Tbm) * h;
          const C de2 = fma_(Tbp, bkp, -(Tbm * bkm)) * h;
          const bool no = E && edge;
          R[0][1 + k] += no ? (C)0 : dm;
          R[0][1 + NDIR] += no ? (C)0 : de1;
          R[0][2 + NDIR + k] -= no ? (C)0 : db;
          R[0][1 + NDIR] -= no ? (C)0 : de2;
        }
      }
    };
    if (x0 <= g.Mlo[0] || x0 + TX > g.Mhi[0] || y0 <= g.Mlo[1] || y0 + TY > g.Mhi[1])
      cross(Bool<true>{});
    else
      cross(Bool<false>{});
  }
  c[0] = cx;
  c[1] = cy;
  c[2] = z;
  // gravity on rho' (gravity_cells), with m_d/rho_t from setnu's q of v_d
  {
    const C rho = qc[0];
    C rg = 0;
#pragma unroll
    for (int d = 0; d < NDIM; d++) {
      const bool on = f.grav_on[d] != 0;
      const C gr = (C)f.grav[d] * rho;
      R[0][1 + d] = on ? R[0][1 + d] + gr : R[0][1 + d];
      rg = on ? rg + gr * qc[(2 + d) * QA] : rg;
    }
    R[0][1 + NDIR] += rg;
  }
  update_cell<NDIM, NDIR, S, C, RK4L>(f, g, c, icell, base, own, R[0], redv);
  return true;
}

// ---------------------------------------------------------------------
// 3-D: the factors T_{0,2} and T_{1,2} of a tile's cells, made along x and y
// from v_2 and b_2, which the z work differentiates along z.  Making
// them in a pass of its own (4 fields read, 4 written) lets the z pass come
// before the x and y work, whose kernel can then finish the cell: the rate of
// x and y stays in registers and there is no combining pass.  A stage at
// 256^3 in FP64: plane tiles 1.84 ms, z lines 1.29, update 1.10 (1.68 RK4's
// last); now factors 0.27, z columns 0.83, this file's tiles 2.07 (2.37).  At
// 128^3: 0.266 + 0.177 + 0.158 (0.222), now 0.041 + 0.113 + 0.270 (0.319).
template <typename C>
struct TzSmem {
  C v[2][PY][PX];  // v_2, b_2
};

template <typename S, typename C>
__device__ __forceinline__ void tz_tile(const AxisArgs& a, int x0, int y0, int z, TzSmem<C>& sm) {
  constexpr int NDIM = 3, NDIR = 3;
  const GridDesc& g = a.g;
  const long long fs = g.fs, zoff = (long long)z * g.st[2];
  const int t = (int)threadIdx.x;
  const int tx = t % TX, ty = cell_row<C>(t);
  const int cx = x0 + tx, cy = y0 + ty;
  const int cxc = (cx > g.G[0] - 1) ? g.G[0] - 1 : cx;
  const int cyc = (cy > g.G[1] - 1) ? g.G[1] - 1 : cy;
  const C dxx = (C)a.dx[0][cxc], dxy = (C)a.dx[1][cyc];
  const C ix0 = (C)a.dx[0][kDxInv * a.dxs + cxc], iy0 = (C)a.dx[1][kDxInv * a.dxs + cyc];
  const C ctx = (C)red_get(a.ctot_src, 0), cty = (C)red_get(a.ctot_src, 1);
  const int yb = y0 > HALO ? y0 - HALO : 0;
  const long long ob = zoff + yb * g.st[1];
  const S* __restrict__ W = (const S*)a.wct + ob;
  const double* __restrict__ B = a.bg + ob;
  // the tile's points, then the columns and rows beside it (as in stage_tile)
#pragma unroll
  for (int k = 0; k < 2; k++) {
    int ix = tx + HALO, iy = ty + HALO;
    if (k == 1) {
      if (t >= 192) break;
      if (t < 96) {
        const int r = t / 6, u = t - 6 * r;
        ix = u < 3 ? u : u + TX;
        iy = r + HALO;
      } else {
        const int u = (t - 96) / TX;
        ix = (t - 96) % TX + HALO;
        iy = u < 3 ? u : u + TY;
      }
    }
    int gx = x0 - HALO + ix, gy = y0 - HALO + iy;
    if (gx < 0) gx = g.Mlo[0] + 3;
    if (gx > g.G[0] - 1) gx = g.Mhi[0] - 3;
    if (gy < 0) gy = g.Mlo[1] + 3;
    if (gy > g.G[1] - 1) gy = g.Mhi[1] - 3;
    const unsigned i = (unsigned)(gy - yb) * (unsigned)g.st[1] + (unsigned)gx;
    const unsigned ow = i * (unsigned)sizeof(S), o8 = i * 8u;
    auto wv = [&](int n) { return (C) * (const S*)((const char*)(W + (size_t)n * fs) + ow); };
    const C rho = wv(0), m = wv(1 + 2), b = wv(2 + NDIR + 2);
    const double rhob = *(const double*)((const char*)(B + fs) + o8);
    sm.v[0][iy][ix] = m * (C)recip<C>((double)rho + rhob);  // nothing to contract
    sm.v[1][iy][ix] = b;
  }
  __syncthreads();
  if (cx < g.Mlo[0] || cx > g.Mhi[0] || cy > g.Mhi[1]) return;
  const bool zx = (cx == g.Mlo[0] && !g.per_lo[0]) || (cx == g.Mhi[0] && !g.per_hi[0]);
  const bool zy = (cy == g.Mlo[1] && !g.per_lo[1]) || (cy == g.Mhi[1] && !g.per_hi[1]);
  const long long icell = zoff + (long long)cy * g.st[1] + cx;
  S* __restrict__ T = (S*)a.T;
#pragma unroll
  for (int w = 0; w < 2; w++) {
    const C* q0 = &sm.v[w][ty + HALO][tx + HALO];
    C q[7];
#pragma unroll
    for (int s = 0; s < 7; s++) q[s] = q0[s - 3];
    T[(long long)(cross_index(NDIM, 0, 2) + w) * fs + icell] =
        (S)cross_factor<C>(q, w, zx, dxx, ix0, ctx);
#pragma unroll
    for (int s = 0; s < 7; s++) q[s] = q0[(s - 3) * PX];
    T[(long long)(cross_index(NDIM, 1, 2) + w) * fs + icell] =
        (S)cross_factor<C>(q, w, zy, dxy, iy0, cty);
  }
}

}  // namespace tile
}  // namespace sac
