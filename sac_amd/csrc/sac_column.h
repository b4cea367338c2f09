// sac_column.h -- the z work of a 3-D stage with one thread per column.
//
// The work per cell is that of the line tiles along z (sac_line.h): flux
// divergence and background energy terms, Powell's sources, setnu and the
// hyperdiffusion line terms, the factors T_{2,0}, T_{2,1}, and the cross
// terms with derivatives along z of T_{0,2}, T_{1,2}; R is written.
//
// Schedule.  A thread marches its column upwards, one point per step; a
// wavefront holds 64 neighbouring columns, so every load and store is a row
// of x and everything that depends on z alone (edges, widths, mirrored
// points) is uniform.  The new point gives setnu's q values and the flux along
// z; the cell two points behind then has its flux divergence and z cross
// terms, the cell three behind its hyperdiffusion, and is stored.  The windows
// of q, rho_t and m stay in registers, each face's ratios are evaluated once
// and serve the cells on both its sides, and what does not fit waits in LDS
// (the fluxes, the oldest q) at places that only their own thread uses: there
// is no barrier.  The next point's 13 fields are loaded into the registers of
// the last one before the hyperdiffusion, which hides their latency.
//
// The line tiles evaluated both faces of each cell and waited at two barriers
// a chunk; half of their time was neither arithmetic nor memory.  z work at
// 128^3 in FP64 146 -> 113 us, at 256^3 0.97 -> 0.83 ms, at 250x90x77 in FP32
// storage 78 -> 69 us.  Each cell is 37 loads and stores of 8 bytes (0.97 ms
// at 256^3 without any reuse in L2): memory is what bounds it there.  Two
// wavefronts per SIMD take all registers in FP64; any spill costs more than
// the whole gain, because the waits for it wait for the prefetch too (220 us
// at 128^3).
#pragma once
#include "sac_device.h"

namespace sac {
namespace column {

constexpr int NT = 256;
constexpr int ROWS = 4;
constexpr int NDIM = 3, NDIR = 3, K = 2, NE = 8, NP = 7;
constexpr int SEG = 32;  // cells of a segment, at most

// LDS (elements): the fluxes' ring (b_2 has none along z; its slot keeps
// b_2 + bg_2 for Powell's sources), the oldest point of each q window, and
// the widths of the segment's cells
template <typename C, bool DIVB>
struct Lay {
  static constexpr int NF = DIVB ? NE : NE - 1;
  static constexpr int Q = ROWS * NF * NT;
  static constexpr int DX = Q + NP * NT;  // [4][SEG]
  static constexpr int R = DX + 4 * SEG;  // rates on their way to the next step, NR of them
  static constexpr int NR = (sizeof(C) == 8 && !DIVB) ? 3 : 0;
  static constexpr int END = R + NR * NT;
};
// flux slot of field n
__host__ __device__ constexpr int fslot(int n) { return n > 2 + NDIR + K ? n - 1 : n; }

// columns of a grid
__host__ __device__ inline long long ncolumns(const GridDesc& g) {
  return (long long)(g.Mhi[0] - g.Mlo[0] + 1) * (g.Mhi[1] - g.Mlo[1] + 1);
}

#define gas __attribute__((address_space(1)))
__device__ __forceinline__ gas char* plane(const void* p) {
  gas char* u = (gas char*)p;
  asm("" : "+s"(u));
  return u;
}

// setnu's ratio of the face between q[2] and q[3] (face_ratio; the divisor as
// in face_pair)
template <typename C>
__device__ __forceinline__ C face_one(C q0, const C (&q1)[5]) {
#pragma clang fp contract(off)
  const C q[6] = {q0, q1[0], q1[1], q1[2], q1[3], q1[4]};
  C s[5], d3[3];
#pragma unroll
  for (int j = 0; j < 5; j++) s[j] = q[j + 1] - q[j];
#pragma unroll
  for (int j = 0; j < 3; j++) d3[j] = fabs((C)3 * s[j + 1] - (q[j + 3] - q[j]));
  const C tiny = sizeof(C) == 8 ? (C)4.9406564584124654e-324 : (C)1.4012984643e-45f;
  const C md1 = fmax(fmax(fmax(fmax(fmax(tiny, fabs(s[0])), fabs(s[1])), fabs(s[2])), fabs(s[3])),
                     fabs(s[4]));
  return cdiv(fmax(fmax(d3[0], d3[1]), d3[2]), md1);
}

// Columns blockIdx.x * NT ..., cells Mlo + blockIdx.y * seg ... along z.
template <typename S, typename C, bool DIVB>
__device__ __forceinline__ void march(const AxisArgs& a, int seg, C* __restrict__ L, C& numax) {
  using Ly = Lay<C, DIVB>;
  const GridDesc& g = a.g;
  const long long fs = g.fs, sz = g.st[2];
  const double gamma = a.gamma;
  const int GK = g.G[2], lo = g.Mlo[2], hi = g.Mhi[2];
  const int tid = (int)threadIdx.x;
  const unsigned nx = (unsigned)(g.Mhi[0] - g.Mlo[0] + 1), ncol = (unsigned)ncolumns(g);
  unsigned col = blockIdx.x * (unsigned)NT + (unsigned)tid;
  if (col >= ncol) col = ncol - 1;  // threads past the end repeat the last column
  const unsigned ry = col / nx, rx = col - ry * nx;
  unsigned o = ((unsigned)g.Mlo[1] + ry) * (unsigned)g.st[1] + (unsigned)g.Mlo[0] + rx;
  const int cs = lo + (int)blockIdx.y * seg;
  const int ce = (cs + seg - 1 < hi) ? cs + seg - 1 : hi;

  // Field n of the state, the background or T at grid index z: a uniform
  // address plus the thread's offset in the plane, kept apart (the sum of an
  // offset and a field's address per thread takes two registers and an
  // addition for each load).
  auto wv = [&](int n, int z) {
    return (C) * (const gas S*)(plane((const S*)a.wct + n * fs + z * sz) + o * (unsigned)sizeof(S));
  };
  auto bv = [&](int n, int z) {
    return *(const gas double*)(plane(a.bg + n * fs + z * sz) + o * 8u);
  };
  auto tv = [&](int n, int z) {
    return (C) * (const gas S*)(plane((const S*)a.T + n * fs + z * sz) + o * (unsigned)sizeof(S));
  };
  auto put = [&](void* p, int n, int z, C v) {
    *(gas S*)(plane((S*)p + n * fs + z * sz) + o * (unsigned)sizeof(S)) = (S)v;
  };
  auto load = [&](int z, Pt<NDIR, C>& p) {
    if (z < 0) z = lo + 3;  // mirror layer beyond the grid
    if (z > GK - 1) z = hi - 3;
    p.rho = wv(0, z);
#pragma unroll
    for (int d = 0; d < NDIR; d++) p.m[d] = wv(1 + d, z);
    p.e = wv(1 + NDIR, z);
#pragma unroll
    for (int d = 0; d < NDIR; d++) p.b[d] = wv(2 + NDIR + d, z);
    p.eb = bv(0, z);
    p.rhob = bv(1, z);
#pragma unroll
    for (int d = 0; d < NDIR; d++) p.bg[d] = bv(2 + d, z);
  };
  // widths of cell c: dx, 1/dx, 1/(12 dx), 1/(2 dx)
  if (tid < 4 * SEG) {
    const int k = tid / SEG, c = cs + tid % SEG;
    const int tab = (k == 0) ? 0 : (k == 1) ? kDxInv : (k == 2) ? kDxInv12 : kDxHalf;
    L[Ly::DX + tid] = (C)a.dx[2][tab * a.dxs + (c < ce ? c : ce)];
  }
  auto dxv = [&](int c, int k) { return L[Ly::DX + k * SEG + c - cs]; };
  const C ctk = (C)red_get(a.ctot_src, K);

  // q of setnu at points p-4..p (p-5: q0): rho', thermal energy, v_l, b_0, b_1
  C q[NP][5], rat[NP], rt[5], m[NDIM][5], R[NE];
  auto q0 = [&](int v) -> C& { return L[Ly::Q + v * NT + tid]; };
  // flux slot s of point p + d
  auto at = [&](int s, int r) -> C& { return L[((r & 3) * Ly::NF + s) * NT + tid]; };
#pragma unroll
  for (int v = 0; v < NP; v++) {
    rat[v] = 0;
#pragma unroll
    for (int s = 0; s < 5; s++) q[v][s] = 0;
  }
#pragma unroll
  for (int s = 0; s < 5; s++) {
    rt[s] = 0;
#pragma unroll
    for (int l = 0; l < NDIM; l++) m[l][s] = 0;
  }
#pragma unroll
  for (int n = 0; n < NE; n++) R[n] = 0;

  // a new point: the windows move on
  auto point = [&](const Pt<NDIR, C>& pt) {
#pragma clang fp contract(off)
    const double rtd = (double)pt.rho + pt.rhob;
    const double inv = recip<C>(rtd);
#pragma unroll
    for (int v = 0; v < NP; v++)
#pragma unroll
      for (int s = 0; s < 4; s++) q[v][s] = q[v][s + 1];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      rt[s] = rt[s + 1];
#pragma unroll
      for (int l = 0; l < NDIM; l++) m[l][s] = m[l][s + 1];
    }
    double sb = 0.0, sm = 0.0;
#pragma unroll
    for (int d = 0; d < NDIR; d++) {
      const double mc = (double)pt.m[d], bc = (double)pt.b[d];
      sb += bc * bc;
      sm += mc * mc;
    }
    q[0][4] = pt.rho;
    q[1][4] = (C)((double)pt.e - 0.5 * (sb + sm * inv));
#pragma unroll
    for (int l = 0; l < NDIM; l++) q[2 + l][4] = pt.m[l] * (C)inv;
    q[5][4] = pt.b[0];
    q[6][4] = pt.b[1];
    rt[4] = (C)rtd;
#pragma unroll
    for (int l = 0; l < NDIM; l++) m[l][4] = pt.m[l];
  };
  auto flux = [&](const Pt<NDIR, C>& pt, C (&F)[NE]) {
    C v[NDIM];
    flux_pt<NDIR, NDIM, C>(pt, K, gamma, F, v);
    if constexpr (DIVB) F[2 + NDIR + K] = (C)((double)pt.b[K] + pt.bg[K]);
  };
  auto keep = [&](const C (&F)[NE], int p) {
#pragma unroll
    for (int n = 0; n < NE; n++)
      if (n != 2 + NDIR + K) at(fslot(n), p) = F[n];
    if constexpr (DIVB) at(NE - 1, p) = F[2 + NDIR + K];
  };

  // ---- the five points before the first face ----
  Pt<NDIR, C> nxt;
  load(cs - 3, nxt);
  __syncthreads();  // the widths
#pragma unroll 1
  for (int p = cs - 3; p < cs + 2; p++) {
    asm("" : "+v"(o));  // not widened ahead of the loop
    C F[NE];
    point(nxt);
    flux(nxt, F);
    keep(F, p);
    load(p + 1, nxt);
#pragma unroll
    for (int v = 0; v < NP; v++) q0(v) = q[v][0];
  }
#pragma unroll 1
  for (int p = cs + 2; p <= ce + 3; p++) {
    asm("" : "+v"(o));
    // of the cell two behind, whose divergence is due: background, and the
    // factors at its neighbours (of mesh cells; zero elsewhere)
    const int c2 = p - 2;  // ce + 1 in the last step, for nothing
    Pt<NDIR, C> pbg;
    C Tc[4 * K];
    pbg.eb = bv(0, c2);
#pragma unroll
    for (int d = 0; d < NDIR; d++) pbg.bg[d] = bv(2 + d, c2);
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int x = cross_index(NDIM, k, K);
      Tc[4 * k + 0] = tv(x, c2 + 1);
      Tc[4 * k + 1] = tv(x, c2 - 1);
      Tc[4 * k + 2] = tv(x + 1, c2 + 1);
      Tc[4 * k + 3] = tv(x + 1, c2 - 1);
    }
    point(nxt);
    __builtin_amdgcn_sched_barrier(0);

    C Rn[NE];
    // ---- the point's flux, and the divergence of the cell two behind ----
    // (point c2 + d: q[.][2 + d], rt and m [2 + d], ring row p - 2 + d)
    {
      C F[NE];
      flux(nxt, F);
      const int cd = c2 > ce ? ce : c2;
      const C inv12 = dxv(cd, 2), h = dxv(cd, 3);
      const bool fluxc = c2 >= lo + 2 && c2 <= hi - 2;
#pragma unroll
      for (int n = 0; n < NE; n++) {
        if (n == 2 + NDIR + K) {
          Rn[n] = 0;
          continue;
        }
        C E1, e2;
        const C D1 = two_diff(at(fslot(n), p - 1), at(fslot(n), p - 3), E1);
        const C D2 = two_diff(F[n], at(fslot(n), p), e2);
        Rn[n] = ((D2 - (C)8 * D1) + (e2 - (C)8 * E1)) * inv12;
      }
      const C pTb0 = (C)ptotal_bg<NDIR, C>(pbg, gamma);
      const C bgk = (C)pbg.bg[K];
      C re = 0;
#pragma unroll
      for (int l = 0; l < NDIM; l++) {
        const C dv1 = q[2 + l][3] - q[2 + l][1];
        const C dv2 = q[2 + l][4] - q[2 + l][0];
        const C Dv = -(dv2 - (C)8 * dv1) * inv12;
        if (l == K) re -= Dv * pTb0;
        re += bgk * (C)pbg.bg[l] * Dv;
      }
      Rn[1 + NDIR] += re;
#pragma unroll
      for (int n = 0; n < NE; n++) Rn[n] = fluxc ? Rn[n] : (C)0;
      if constexpr (DIVB) {  // Powell's div B sources (see line_tile)
        if (fluxc) {
          const C D1b = at(NE - 1, p - 1) - at(NE - 1, p - 3);
          const C D2b = F[2 + NDIR + K] - at(NE - 1, p);
          const C gK = -((D2b - (C)8 * D1b) * inv12);
          const double rc = (double)wv(0, c2) + bv(1, c2);
          double sm = 0.0;
#pragma unroll
          for (int d = 0; d < NDIR; d++) {
            const double mc = (double)wv(1 + d, c2);
            const double bt = (double)wv(2 + NDIR + d, c2) + bv(2 + d, c2);
            Rn[1 + d] -= (C)bt * gK;
            Rn[2 + NDIR + d] -= (C)(mc / rc) * gK;
            sm = (d == 0) ? mc * bt : sm + mc * bt;
          }
          Rn[1 + NDIR] -= (C)(sm / rc) * gK;
        }
      }
      const bool no = (c2 == lo && !g.per_lo[2]) || (c2 == hi && !g.per_hi[2]);
      const bool inP = c2 + 1 <= hi, inM = c2 - 1 >= lo;
#pragma unroll
      for (int k = 0; k < K; k++) {
        const C Tmp = inP ? Tc[4 * k + 0] : (C)0, Tmm = inM ? Tc[4 * k + 1] : (C)0;
        const C Tbp = inP ? Tc[4 * k + 2] : (C)0, Tbm = inM ? Tc[4 * k + 3] : (C)0;
        const C dm = (rt[3] * Tmp - rt[1] * Tmm) * h;
        const C de1 = (m[k][3] * Tmp - m[k][1] * Tmm) * h;
        const C db = (Tbp - Tbm) * h;
        const C de2 = (Tbp * q[5 + k][3] - Tbm * q[5 + k][1]) * h;
        Rn[1 + k] += no ? (C)0 : dm;
        Rn[1 + NDIR] += no ? (C)0 : de1;
        Rn[2 + NDIR + k] -= no ? (C)0 : db;
        Rn[1 + NDIR] -= no ? (C)0 : de2;
      }
      keep(F, p);
#pragma unroll
      for (int n = 0; n < Ly::NR; n++) {
        R[n] = L[Ly::R + n * NT + tid];
        L[Ly::R + n * NT + tid] = Rn[n];
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // nxt takes the registers of the point
    load(p < ce + 3 ? p + 1 : p, nxt);
    __builtin_amdgcn_sched_barrier(0);

    // ---- hyperdiffusion of the cell three behind ----
    // (point c + d: q[.][1 + d], rt and m [1 + d]).  The first step, with c
    // below the segment, is for the lower faces of its first cell; what it
    // stores there is written again by the next step.  (A branch around the
    // stores would let the compiler move the work above into the blocks
    // between them, and spill for it.)
    {
#pragma clang fp contract(off)
      const int c = p - 3;
      const bool z1 = (c == lo && !g.per_lo[2]) || (c == hi && !g.per_hi[2]);
      const int cd = c < cs ? cs : c;
      const HyperAxis<C> ha(ctk, dxv(cd, 0), dxv(cd, 1));
      C nmax = 0;
      const C rhoL = rt[1] + rt[0], rhoR = rt[2] + rt[1];  // twice the means
#pragma unroll
      for (int v = 0; v < NP; v++) {
        const bool vel = v >= 2 && v < 2 + NDIM;
        const C ratR = face_one<C>(q0(v), q[v]);
        C tL, tR;
        const C w[5] = {0, 0, q[v][0], q[v][1], q[v][2]};
        const C T = hyper_faces<C>(w, vel ? ha.kv : ha.ks, rat[v], ratR, z1, tL, tR, nmax);
        if (v == 0) {
          R[0] = fma_(tR - tL, ha.i2, R[0]);
        } else if (v == 1) {
          R[1 + NDIR] = fma_(tR - tL, ha.i2, R[1 + NDIR]);
        } else if (vel) {
          const int l = v - 2;
          const C mL = m[l][1] + m[l][0], mR = m[l][2] + m[l][1];
          const C f = (l == K) ? ha.i2h : ha.i2q;  // the i==k branch runs twice for l==k
          R[1 + l] = fma_(fma_(rhoR, tR, -(rhoL * tL)), f, R[1 + l]);
          R[1 + NDIR] = fma_(fma_(mR, tR, -(mL * tL)), f, R[1 + NDIR]);
          if (l != K) put(a.T, cross_index(NDIM, K, l), cd, T * ha.it);
        } else {
          const int lb = v - 2 - NDIM;
          const C BL = q[v][1] + q[v][0], BR = q[v][2] + q[v][1];
          R[2 + NDIR + lb] = fma_(tR - tL, ha.i2, R[2 + NDIR + lb]);
          R[1 + NDIR] = fma_(fma_(BR, tR, -(BL * tL)), ha.i2h, R[1 + NDIR]);
          put(a.T, cross_index(NDIM, K, lb) + 1, cd, (C)2 * T * ha.it);
        }
        rat[v] = ratR;
        q0(v) = q[v][0];
        __builtin_amdgcn_sched_barrier(0);
      }
      numax = fmax(numax, c < cs ? (C)0 : ha.nu(nmax));
#pragma unroll
      for (int n = 0; n < NE; n++) put(a.R, n, cd, R[n]);
    }
#pragma unroll
    for (int n = Ly::NR; n < NE; n++) R[n] = Rn[n];
  }
}

#undef gas
}  // namespace column
}  // namespace sac
