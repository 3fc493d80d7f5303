// The coarse end of the V-cycle, where a pass over a level costs its latency and not its bytes:
// the single-workgroup tail (k_mg_tail_lds) and the fused up-leg of a level (k_up).
//
// Included by wl_kernels.h after the per-cell pieces it uses (LRows, lcell, pro_map, TailDesc).
#pragma once
#include "wl_tail.h"

namespace wl {

// LDS image of a tail level: L (D arrays), x, r, ϵ, D, iD, indexed with 32-bit offsets.
template <class T>
struct SLev {
  int N0, N1, N2, s1, s2, n, cm;
  int nxp, npair;  // x pairs per row, pairs of the level
  int lx, ly;      // log2 of the row's and the plane's thread counts (pairs, rows)
  T *L, *x, *r, *e, *Dg, *iD;
};
__device__ __forceinline__ int log2_up(int v) { return v <= 1 ? 0 : 32 - __builtin_clz(v - 1); }

// Mixed precision with WL_COARSE_PCG=1: the coarsest level is solved by pcg! (src/Poisson.jl:166-186)
// in double by one thread, the Jacobi-preconditioned conjugate gradient on A·δ = r from δ = 0: at
// most 6 iterations with the reference's early exits (|ρ| < 10eps, |α| outside [1e-2, 1e2]).  δ,
// rounded to T, is the level's ϵ for increment!, in place of the GS-RB sweeps.
template <class T, int D>
__device__ __forceinline__ void tail_pcg(const SLev<T>& p, double (*cg)[TAIL_CG_MAX]) {
  double *X = cg[0], *ID = cg[1], *R = cg[2], *Z = cg[3], *E = cg[4];
  for (int I = 0; I < p.n; ++I) { X[I] = 0; ID[I] = 0; R[I] = 0; Z[I] = 0; E[I] = 0; }
  auto diag64 = [&](int I) {
    double sd = 0;
    sd -= ((double)p.L[I] + (double)p.L[I + 1]);
    sd -= ((double)p.L[p.n + I] + (double)p.L[p.n + I + p.s1]);
    if (D == 3) sd -= ((double)p.L[2 * p.n + I] + (double)p.L[2 * p.n + I + p.s2]);
    return sd;
  };
  auto each = [&](auto&& f) {
    for (int k = D == 3 ? 1 : 0; k <= (D == 3 ? p.N2 - 2 : 0); ++k)
      for (int j = 1; j <= p.N1 - 2; ++j)
        for (int i = 1; i <= p.N0 - 2; ++i) f(i + p.s1 * j + p.s2 * k);
  };
  auto dot64 = [&](const double* a, const double* b) {
    double acc = 0;
    each([&](int I) { acc += a[I] * b[I]; });
    return acc;
  };
  each([&](int I) {
    const double sd = diag64(I);
    ID[I] = sd == 0.0 ? 0.0 : 1.0 / sd;
    R[I] = (double)p.r[I];
    Z[I] = E[I] = R[I] * ID[I];
  });
  const double tiny = 10.0 * 2.220446049250313e-16;
  double rho = dot64(R, Z);
  if (fabs(rho) >= tiny) {
    for (int it = 1; it <= 6; ++it) {
      each([&](int I) {  // z = A·ϵ (mult, src/Poisson.jl:71-76; ghosts of ϵ are 0)
        double sv = E[I] * diag64(I);
        sv += (E[I - 1] * (double)p.L[I] + E[I + 1] * (double)p.L[I + 1]);
        sv += (E[I - p.s1] * (double)p.L[p.n + I] + E[I + p.s1] * (double)p.L[p.n + I + p.s1]);
        if (D == 3) sv += (E[I - p.s2] * (double)p.L[2 * p.n + I] + E[I + p.s2] * (double)p.L[2 * p.n + I + p.s2]);
        Z[I] = sv;
      });
      const double alpha = rho / dot64(Z, E);
      if (fabs(alpha) < 1e-2 || fabs(alpha) > 1e2) break;
      each([&](int I) {
        X[I] += alpha * E[I];
        R[I] -= alpha * Z[I];
      });
      if (it == 6) break;
      each([&](int I) { Z[I] = R[I] * ID[I]; });
      const double rho2 = dot64(R, Z);
      if (fabs(rho2) < tiny) break;
      const double beta = rho2 / rho;
      each([&](int I) { E[I] = beta * E[I] + Z[I]; });
      rho = rho2;
    }
  }
  each([&](int I) { p.e[I] = (T)X[I]; });
}

// The coarse tail with every level resident in LDS (L, r copied in, D and iD formed once), from
// Jacobi! on the first tail level down to the coarsest and back up through the first level's smooth!
// (src/MultiLevelPoisson.jl:88-101,106; src/Poisson.jl:100-148), perBC! where the reference has it.
//
// What bounds it is latency: about 29 dependent passes of at most a few thousand cells, one
// workgroup on an otherwise idle chip.  So
//  - in a half sweep a thread owns x pairs, one cell of which it updates, so no lane idles; in the other
//    passes it owns one cell where the level has no more than threads (in pairs 35 us against 27.5 on
//    32x32 and its three coarser levels), else pairs; both are dealt to the threads by shifts chosen
//    from the level's own extents;
//  - without KEEP, levels of at most 128 pairs run in the first wave alone, two pairs to a lane at most:
//    the LDS serves a wave in order, so their passes need no barrier (the other waves wait at one);
//    KEEP's passes over all cells take longer in one wave than the barriers cost (29 against 27.5 us);
//  - without KEEP (a flow's own solver, whose coarse levels nobody reads) the last increment! of a
//    level is x += ω·ϵ inside the fourth half sweep (its r is dead: the next V-cycle's restrict!
//    overwrites it), nothing but the first level's x is stored, and only r and L are loaded.
// KEEP holds the reference's whole level state (a standalone MultiLevelPoisson).
template <class T, int D, bool KEEP>
__device__ __forceinline__ void k_mg_tail_lds_body(const TailDesc<T>& d, const T* __restrict__ wp,
                                                   double (*cg)[TAIL_CG_MAX]) {
  constexpr int WAVE_PAIRS = 128;
  const T w = *wp;
  const int tid = threadIdx.x;
  const int lnt = 31 - __builtin_clz((int)blockDim.x);
  extern __shared__ __align__(16) unsigned char tail_smem[];
  T* sb = reinterpret_cast<T*>(tail_smem);
  auto lev = [&](int l) -> SLev<T> {
    SLev<T> q;
    const Geo& g = d.lv[l].g;
    q.N0 = g.N[0]; q.N1 = g.N[1]; q.N2 = D == 3 ? g.N[2] : 1;
    q.s1 = q.N0; q.s2 = q.N0 * q.N1; q.n = q.s2 * q.N2; q.cm = d.lv[l].cmask;
    q.nxp = (q.N0 - 1) >> 1;
    q.npair = q.nxp * (q.N1 - 2) * (D == 3 ? q.N2 - 2 : 1);
    q.lx = log2_up(q.nxp); q.ly = log2_up(q.N1 - 2);
    q.L = sb + d.lv[l].off;
    q.x = q.L + D * q.n; q.r = q.x + q.n; q.e = q.r + q.n; q.Dg = q.e + q.n; q.iD = q.Dg + q.n;
    return q;
  };
  // f(x, y, z) for each pair (x, x+1) of the level, over 2^ln threads; the second cell of a row's last
  // pair may be its ghost (x + 1 = N0 − 1), which f leaves alone
  auto pair_loop = [&](const SLev<T>& q, int ln, auto&& f) {
    const int sx = q.lx < ln ? q.lx : ln, sy = q.ly < ln - sx ? q.ly : ln - sx;
    const int bx = 1 << sx, by = 1 << sy, bz = 1 << (ln - sx - sy);
    const int tx = tid & (bx - 1), ty = (tid >> sx) & (by - 1), tz = tid >> (sx + sy);
    const int zlo = D == 3 ? 1 : 0, zhi = D == 3 ? q.N2 - 2 : 0;
    for (int z = zlo + tz; z <= zhi; z += bz)
      for (int y = 1 + ty; y <= q.N1 - 2; y += by)
        for (int p = tx; p < q.nxp; p += bx) f(1 + 2 * p, y, z);
  };
  // f(x, y, z) for each cell
  auto cell_loop = [&](const SLev<T>& q, int ln, auto&& f) {
    const int zlo = D == 3 ? 1 : 0, zhi = D == 3 ? q.N2 - 2 : 0;
    const int cx = log2_up(q.N0 - 2), cl = cx + q.ly;
    if (cl <= ln && ((zhi - zlo + 1) << cl) <= 1 << ln) {
      const int x = 1 + (tid & ((1 << cx) - 1)), y = 1 + ((tid >> cx) & ((1 << q.ly) - 1)), z = zlo + (tid >> cl);
      if (x <= q.N0 - 2 && y <= q.N1 - 2 && z <= zhi) f(x, y, z);
    } else {
      pair_loop(q, ln, [&](int x, int y, int z) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
          if (x + o <= q.N0 - 2) f(x + o, y, z);
      });
    }
  };
  // a pass's end: a barrier, or inside the first wave only the order of its LDS operations
  auto sync = [&](bool wave) {
    if (wave) {
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      __syncthreads();
    }
  };
  auto smult = [](const SLev<T>& q, const T* v, int I) -> T {
    T s = v[I] * q.Dg[I];
    s += (v[I - 1] * q.L[I] + v[I + 1] * q.L[I + 1]);
    s += (v[I - q.s1] * q.L[q.n + I] + v[I + q.s1] * q.L[q.n + I + q.s1]);
    if (D == 3) s += (v[I - q.s2] * q.L[2 * q.n + I] + v[I + q.s2] * q.L[2 * q.n + I + q.s2]);
    return s;
  };
  auto perbc = [&](const SLev<T>& q, T* a, int ln, bool wave) {  // periodic ghosts -> images
    if (!d.perdir) return;
    const int N[3] = {q.N0, q.N1, q.N2};
    for (int k = tid; k < q.n; k += 1 << ln) {
      const int c[3] = {k % q.N0, (k / q.s1) % q.N1, D == 3 ? k / q.s2 : 0};
      int m[3] = {c[0], c[1], c[2]};
      bool ghost = false;
#pragma unroll
      for (int r = 0; r < D; ++r) {
        if (!((d.perdir >> r) & 1)) continue;
        if (c[r] == 0) { m[r] = N[r] - 2; ghost = true; }
        else if (c[r] == N[r] - 1) { m[r] = 1; ghost = true; }
      }
      if (ghost) a[k] = a[m[0] + q.s1 * m[1] + q.s2 * m[2]];
    }
    sync(wave);
  };

  // ---- copy in; ghosts of ϵ are 0 (perBC! sets them where periodic) ----
  for (int l = 0; l < d.n; ++l) {
    const SLev<T> q = lev(l);
    const T* gL = d.lv[l].L;
    const T* gr = d.lv[l].r;
    const T* gx = d.lv[l].x;
    const T* ge = d.lv[l].e;
    const int nL = D * q.n, nt = blockDim.x;
#pragma unroll 4
    for (int k = tid; k < nL; k += nt) q.L[k] = gL[k];
    if (KEEP) {
      for (int k = tid; k < q.n; k += nt) { q.x[k] = gx[k]; q.r[k] = gr[k]; q.e[k] = ge[k]; }
    } else {
      if (l == 0) {
#pragma unroll 4
        for (int k = tid; k < q.n; k += nt) q.r[k] = gr[k];
      }
      for (int k = tid; k < q.n; k += nt) q.e[k] = T(0);
    }
  }
  __syncthreads();
  for (int l = 0; l < d.n; ++l) {  // D, iD on inside (src/Poisson.jl:43-46); the first level's ϵ = r·iD
    const SLev<T> q = lev(l);
    cell_loop(q, lnt, [&](int x, int y, int z) {
      const int I = x + q.s1 * y + q.s2 * z;
      T sd = 0;
      sd -= (q.L[I] + q.L[I + 1]);
      sd -= (q.L[q.n + I] + q.L[q.n + I + q.s1]);
      if (D == 3) sd -= (q.L[2 * q.n + I] + q.L[2 * q.n + I + q.s2]);
      const T id = inv_diag(sd);
      q.Dg[I] = sd;
      q.iD[I] = id;
      if (!KEEP && l == 0) {  // as restrict! left it
        q.x[I] = 0;
        q.e[I] = q.r[I] * id;
      }
    });
  }
  __syncthreads();

  // Jacobi!'s increment! (ω = 1): a cell reads ϵ, which no thread writes, and updates its own r and x
  auto jacobi = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l);
    perbc(f, f.e, ln, wave);
    cell_loop(f, ln, [&](int x, int y, int z) {
      const int I = x + f.s1 * y + f.s2 * z;
      f.r[I] = f.r[I] - T(1) * smult(f, f.e, I);
      f.x[I] = f.x[I] + T(1) * f.e[I];
    });
    sync(wave);
  };
  // restrict! to level l+1, fill!(x, 0) and ϵ = r·iD there: children summed in z, y, x order
  auto restrict_to = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l), c = lev(l + 1);
    cell_loop(c, ln, [&](int x, int y, int z) {
      const int cc[3] = {x, y, z};
      int a0[3], a1[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bool two = q < D && ((f.cm >> q) & 1);
        a0[q] = two ? 2 * cc[q] - 1 : cc[q];
        a1[q] = two ? 2 * cc[q] : cc[q];
      }
      T s = 0;
      for (int kk = a0[2]; kk <= a1[2]; ++kk)
        for (int jj = a0[1]; jj <= a1[1]; ++jj)
          for (int ii = a0[0]; ii <= a1[0]; ++ii) s += f.r[ii + f.s1 * jj + f.s2 * kk];
      const int Ic = x + c.s1 * y + c.s2 * z;
      c.r[Ic] = s;
      c.x[Ic] = 0;
      c.e[Ic] = s * c.iD[Ic];
    });
    sync(wave);
  };
  // smooth!(l): the four half sweeps (ϵ = r·iD is set) and increment!
  auto smooth = [&](int l, int ln, bool wave) {
    const SLev<T> p = lev(l);
    perbc(p, p.e, ln, wave);
    // a flow's x: the first level's goes straight to memory
    T* xg = d.lv[0].x;
    auto xinc = [&](int I) {
      const T v = p.x[I] + w * p.e[I];
      if (l == 0) xg[I] = v; else p.x[I] = v;
    };
    const bool exact = d.exact && l == d.n - 1 && p.n <= TAIL_CG_MAX && !d.perdir;
    // half_rangek (src/Poisson.jl:130-132) on the last axis
    const int klim = D == 3 ? 2 * (p.N2 / 2) - 2 : 2 * (p.N1 / 2) - 2;
    if (exact && d.exact == 2) {
      if (tid == 0) tail_pcg<T, D>(p, cg);
      sync(wave);
    } else if (exact) {
      // Mixed precision: smooth! of the coarsest level in double: ϵ = r·iD and the four GS-RB half
      // sweeps (src/Poisson.jl:141-148) with ϵ, D and iD held in double, then ϵ rounded to T for
      // increment!.  Same algorithm and order as the T sweeps below.  (pcg! here instead moved the
      // constant the Neumann problem leaves free in p away from the reference algorithm's: on a
      // 64x32x32 sphere, p 2.9e-3 and the force 7.5e-4 from the Float64 oracle, against 1e-4 and 5e-6.)
      double *E = cg[0], *ID = cg[1];
      for (int k = tid; k < p.n; k += 1 << ln) E[k] = 0;
      sync(wave);
      auto cells = [&](auto&& f) {
        pair_loop(p, ln, [&](int x, int y, int z) {
#pragma unroll
          for (int o = 0; o < 2; ++o)
            if (x + o <= p.N0 - 2) f(x + o + p.s1 * y + p.s2 * z);
        });
        sync(wave);
      };
      cells([&](int I) {
        double sd = 0;
        sd -= ((double)p.L[I] + (double)p.L[I + 1]);
        sd -= ((double)p.L[p.n + I] + (double)p.L[p.n + I + p.s1]);
        if (D == 3) sd -= ((double)p.L[2 * p.n + I] + (double)p.L[2 * p.n + I + p.s2]);
        ID[I] = sd == 0.0 ? 0.0 : 1.0 / sd;
        E[I] = (double)p.r[I] * ID[I];
      });
      for (int it = 1; it <= 4; ++it) {
        pair_loop(p, ln, [&](int x, int y, int z) {
          const int o = (x + y + z + it + D + 1) & 1;
          const int I = x + o + p.s1 * y + p.s2 * z;
          if (x + o <= p.N0 - 2 && (D == 3 ? z : y) <= klim) {
            double sv = (double)p.r[I];
            sv -= (E[I - 1] * (double)p.L[I] + E[I + 1] * (double)p.L[I + 1]);
            sv -= (E[I - p.s1] * (double)p.L[p.n + I] + E[I + p.s1] * (double)p.L[p.n + I + p.s1]);
            if (D == 3)
              sv -= (E[I - p.s2] * (double)p.L[2 * p.n + I] + E[I + p.s2] * (double)p.L[2 * p.n + I + p.s2]);
            E[I] = sv * ID[I];
          }
        });
        sync(wave);
      }
      cells([&](int I) { p.e[I] = (T)E[I]; });
    } else {
#pragma unroll 1
      for (int it = 1; it <= 4; ++it) {
        pair_loop(p, ln, [&](int x, int y, int z) {
          const int o = (x + y + z + it + D + 1) & 1;  // the pair's cell of this sweep's colour
          const int I = x + o + p.s1 * y + p.s2 * z;
          if (x + o <= p.N0 - 2 && (D == 3 ? z : y) <= klim) {
            T s = p.r[I];
            s -= (p.e[I - 1] * p.L[I] + p.e[I + 1] * p.L[I + 1]);
            s -= (p.e[I - p.s1] * p.L[p.n + I] + p.e[I + p.s1] * p.L[p.n + I + p.s1]);
            if (D == 3) s -= (p.e[I - p.s2] * p.L[2 * p.n + I] + p.e[I + p.s2] * p.L[2 * p.n + I + p.s2]);
            p.e[I] = s * p.iD[I];
          }
          if (!KEEP && it == 4) {  // both cells' ϵ are final: the other colour's since sweep 3
            const int J = x + p.s1 * y + p.s2 * z;
            xinc(J);
            if (x + 1 <= p.N0 - 2) xinc(J + 1);
          }
        });
        sync(wave);
      }
    }
    if (KEEP || exact) {
      perbc(p, p.e, ln, wave);
      cell_loop(p, ln, [&](int x, int y, int z) {
        const int I = x + p.s1 * y + p.s2 * z;
        if (KEEP) {
          p.r[I] = p.r[I] - w * smult(p, p.e, I);
          p.x[I] = p.x[I] + w * p.e[I];
        } else {
          xinc(I);
        }
      });
      sync(wave);
    }
  };
  // prolongate! from level l+1, increment!(l) and ϵ = r·iD for the smooth! that follows
  auto prolong = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l), p = lev(l + 1);
    const int N[3] = {f.N0, f.N1, f.N2};
    cell_loop(f, ln, [&](int x, int y, int z) {
      const int c[3] = {x, y, z};
      int q[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
      for (int dd = 0; dd < D; ++dd)
#pragma unroll
        for (int k = 0; k < 3; ++k) q[dd][k] = pro_map(c[dd] + k - 1, N[dd], (d.perdir >> dd) & 1, (f.cm >> dd) & 1);
      auto xcv = [&](int a, int b, int zz) -> T {
        const bool ok = a >= 0 && b >= 0 && zz >= 0;
        const T v = p.x[ok ? a + p.s1 * b + p.s2 * zz : 0];
        return ok ? v : T(0);
      };
      const int I = x + f.s1 * y + f.s2 * z;
      const T e0 = xcv(q[0][1], q[1][1], q[2][1]);
      T s = e0 * f.Dg[I];
      s += (xcv(q[0][0], q[1][1], q[2][1]) * f.L[I] + xcv(q[0][2], q[1][1], q[2][1]) * f.L[I + 1]);
      s += (xcv(q[0][1], q[1][0], q[2][1]) * f.L[f.n + I] + xcv(q[0][1], q[1][2], q[2][1]) * f.L[f.n + I + f.s1]);
      if (D == 3)
        s += (xcv(q[0][1], q[1][1], q[2][0]) * f.L[2 * f.n + I] + xcv(q[0][1], q[1][1], q[2][2]) * f.L[2 * f.n + I + f.s2]);
      const T rn = f.r[I] - w * s;
      f.r[I] = rn;
      f.x[I] = f.x[I] + w * e0;
      f.e[I] = rn * f.iD[I];
    });
    sync(wave);
  };

  // The passes in order, one loop over them: each pass's code is there once (a launch runs it from
  // cold instruction lines).  ls: the first level of the first wave's part (pairs shrink with the
  // level); a pass belongs to the level it starts from on the way down, and ends at on the way up.
  int ls = d.n;
  while (!KEEP && ls > 0 && lev(ls - 1).npair <= WAVE_PAIRS) --ls;
  const int nd = 2 * (d.n - 1), ns = nd + 2 * d.n - 1;
  bool was_wave = false;
#pragma unroll 1
  for (int k = 0; k < ns; ++k) {
    const bool down = k < nd, odd = (down ? k : k - nd) & 1;
    const int l = down ? k >> 1 : d.n - 1 - ((k - nd + 1) >> 1);
    const bool wave = l >= ls;
    if (was_wave && !wave) __syncthreads();
    was_wave = wave;
    if (wave && tid >= 64) continue;
    const int ln = wave ? 6 : lnt;
    if (down) {
      if (!odd) jacobi(l, ln, wave); else restrict_to(l, ln, wave);
    } else {
      if (!odd) smooth(l, ln, wave); else prolong(l, ln, wave);
    }
  }
  if (KEEP) {
    __syncthreads();
    for (int l = 0; l < d.n; ++l) {  // copy back
      const SLev<T> q = lev(l);
      for (int k = tid; k < q.n; k += blockDim.x) {
        d.lv[l].x[k] = q.x[k]; d.lv[l].r[k] = q.r[k]; d.lv[l].e[k] = q.e[k];
      }
    }
  }
}
template <class T, int D, bool KEEP>
__global__ void __launch_bounds__(1024) k_mg_tail_lds(TailDesc<T> d, const T* __restrict__ wp) {
  __shared__ double cg[5][TAIL_CG_MAX];
  k_mg_tail_lds_body<T, D, KEEP>(d, wp, cg);
}

// ---- the same tail for levels of at most one x pair per thread ----
// A pass over such a level is a few dozen dependent instructions per wave; what it costs is their
// latency, the LDS round trips and the barriers (measured on 48x32 and its four coarser levels with
// loops over the pairs: 0.45 us per half sweep of six cells, 5.7 us to copy the levels in and 2.8 us
// to form D and 1/D).  So a thread owns the same pair for a whole visit of a level and keeps its
// coefficients, residual and x in registers over the four half sweeps; the LDS carries only what
// other threads read (ϵ, the residuals a restriction sums, the coarse x); the L, D and 1/D of all
// levels lie in one image in memory, formed when L changes (k_level_tables), so one round of loads
// brings them in.
template <class T>
struct TailFast {
  int n, perdir, exact, nimg;  // levels; image elements
  const T* img;                // L, D, 1/D of every level, as the LDS holds them
  const T* r;                  // the first level's residual
  T* x;                        // the first level's x (ghosts untouched)
  TailLv lv[TAIL_MAX_LEVELS];
};
constexpr int TAIL_FAST_PAIRS = 1024, TAIL_WAVE_PAIRS = 64;
template <class T, int D>
__device__ __forceinline__ void k_mg_tail_fast_body(const TailFast<T>& d, const T* __restrict__ wp,
                                                    double (*cg)[TAIL_CG_MAX]) {
  const int tid = threadIdx.x;
  extern __shared__ __align__(16) unsigned char tail_smem[];
  T* const S = reinterpret_cast<T*>(tail_smem);
  const T w = *wp;
  {  // the image, the first level's r, and zeros where ϵ has its ghosts
    typedef T V4 __attribute__((ext_vector_type(4)));
    const TailLv q = d.lv[0];
    const int n4 = d.nimg >> 2;  // the host pads the image to whole vectors
    const V4* gi = (const V4*)d.img;
    T rv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = tid + k * TAIL_FAST_PAIRS;
      rv[k] = j < q.n ? d.r[j] : T(0);
    }
#pragma unroll 4
    for (int k = tid; k < n4; k += TAIL_FAST_PAIRS) ((V4*)S)[k] = gi[k];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = tid + k * TAIL_FAST_PAIRS;
      if (j < q.n) S[q.oR + j] = rv[k];
    }
    for (int j = tid + 4 * TAIL_FAST_PAIRS; j < q.n; j += TAIL_FAST_PAIRS) S[q.oR + j] = d.r[j];
    for (int l = 0; l < d.n; ++l)
      for (int j = tid; j < d.lv[l].n; j += TAIL_FAST_PAIRS) S[d.lv[l].oE + j] = T(0);
  }
  __syncthreads();
  auto sync = [&](bool wave) {
    if (wave) {
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      __syncthreads();
    }
  };
  // this thread's pair (x, x+1) of a level: its first cell, or none
  struct Own { int x, y, z, I; bool a, b; };
  auto own = [&](const TailLv& q) -> Own {
    Own o;
    o.x = 1 + 2 * (tid & ((1 << q.lx) - 1));
    o.y = 1 + ((tid >> q.lx) & ((1 << q.ly) - 1));
    o.z = D == 3 ? 1 + (tid >> (q.lx + q.ly)) : 0;
    o.a = o.x <= q.N0 - 2 && o.y <= q.N1 - 2 && (D == 3 ? o.z <= q.N2 - 2 : (tid >> (q.lx + q.ly)) == 0);
    o.b = o.a && o.x + 1 <= q.N0 - 2;
    // a thread without a pair stands on the first one and stores nothing
    o.x = o.a ? o.x : 1;
    o.y = o.a ? o.y : 1;
    if (D == 3) o.z = o.a ? o.z : 1;
    o.I = o.x + q.s1 * o.y + q.s2 * o.z;
    return o;
  };
  // the pair's face coefficients: x faces at x, x+1, x+2; y and z faces of both cells, low and high
  struct Coef { T x0, x1, x2, ya, yb, Ya, Yb, za, zb, Za, Zb; };
  auto coef = [&](const TailLv& q, int I) -> Coef {
    const T* L = S + q.oL;
    Coef c = {};
    c.x0 = L[I]; c.x1 = L[I + 1]; c.x2 = L[I + 2];
    c.ya = L[q.n + I]; c.yb = L[q.n + I + 1]; c.Ya = L[q.n + I + q.s1]; c.Yb = L[q.n + I + q.s1 + 1];
    if (D == 3) {
      const T* Z = L + 2 * q.n;
      c.za = Z[I]; c.zb = Z[I + 1]; c.Za = Z[I + q.s2]; c.Zb = Z[I + q.s2 + 1];
    }
    return c;
  };
  // periodic ghosts of ϵ (perBC!, src/core.jl:239-243); threads of the pass only
  auto perbc = [&](const TailLv& q, bool wave) {
    if (!d.perdir) return;
    const int N[3] = {q.N0, q.N1, q.N2};
    for (int k = tid; k < q.n; k += wave ? 64 : TAIL_FAST_PAIRS) {
      const int c[3] = {k % q.N0, (k / q.s1) % q.N1, D == 3 ? k / q.s2 : 0};
      int m[3] = {c[0], c[1], c[2]};
      bool ghost = false;
#pragma unroll
      for (int r = 0; r < D; ++r) {
        if (!((d.perdir >> r) & 1)) continue;
        if (c[r] == 0) { m[r] = N[r] - 2; ghost = true; }
        else if (c[r] == N[r] - 1) { m[r] = 1; ghost = true; }
      }
      if (ghost) S[q.oE + k] = S[q.oE + m[0] + q.s1 * m[1] + q.s2 * m[2]];
    }
    sync(wave);
  };
  // the first level's x = 0 and ϵ = r·iD, as restrict! leaves them on the others
  {
    const TailLv q = d.lv[0];
    const Own o = own(q);
    if (o.a) {
      S[q.oX + o.I] = 0;
      S[q.oE + o.I] = S[q.oR + o.I] * S[q.oI + o.I];
    }
    if (o.b) {
      S[q.oX + o.I + 1] = 0;
      S[q.oE + o.I + 1] = S[q.oR + o.I + 1] * S[q.oI + o.I + 1];
    }
    __syncthreads();
  }
  // Jacobi! (ω = 1) on level l, restrict! to l+1, ϵ = r·iD there
  auto down = [&](int l, bool wave) {
    const TailLv q = d.lv[l], c = d.lv[l + 1];
    perbc(q, wave);
    {
      const Own o = own(q);
      if (o.a) {
        const T* e = S + q.oE + o.I;
        const T em = e[-1], ea = e[0], eb = e[1], ep = e[2];
        const T ma = e[-q.s1], mb = e[1 - q.s1], pa = e[q.s1], pb = e[q.s1 + 1];
        const Coef k = coef(q, o.I);
        const T Da = S[q.oD + o.I], Db = S[q.oD + o.I + 1], ra = S[q.oR + o.I], rb = S[q.oR + o.I + 1];
        T sa = ea * Da, sb = eb * Db;
        sa += (em * k.x0 + eb * k.x1);
        sb += (ea * k.x1 + ep * k.x2);
        sa += (ma * k.ya + pa * k.Ya);
        sb += (mb * k.yb + pb * k.Yb);
        if (D == 3) {
          sa += (e[-q.s2] * k.za + e[q.s2] * k.Za);
          sb += (e[1 - q.s2] * k.zb + e[q.s2 + 1] * k.Zb);
        }
        S[q.oR + o.I] = ra - T(1) * sa;
        S[q.oX + o.I] = T(0) + T(1) * ea;
        if (o.b) {
          S[q.oR + o.I + 1] = rb - T(1) * sb;
          S[q.oX + o.I + 1] = T(0) + T(1) * eb;
        }
      }
    }
    sync(wave);
    {
      const Own o = own(c);
      if (o.a) {
        const bool cx = q.cm & 1, cy = q.cm & 2, cz = D == 3 && (q.cm & 4);
        const int fx = cx ? 2 * o.x - 1 : o.x, fy = cy ? 2 * o.y - 1 : o.y, fz = cz ? 2 * o.z - 1 : o.z;
        const T* r = S + q.oR + fx + q.s1 * fy + q.s2 * fz;
        T sa = 0, sb = 0;
        auto row = [&](const T* p) {  // both cells' children of one fine row, in x order
          if (cx) {
            sa += p[0];
            sa += p[1];
            sb += p[2];
            sb += p[3];
          } else {
            sa += p[0];
            sb += p[1];
          }
        };
        row(r);
        if (cy) row(r + q.s1);
        if (cz) {
          row(r + q.s2);
          if (cy) row(r + q.s2 + q.s1);
        }
        S[c.oR + o.I] = sa;
        S[c.oX + o.I] = 0;
        S[c.oE + o.I] = sa * S[c.oI + o.I];
        if (o.b) {
          S[c.oR + o.I + 1] = sb;
          S[c.oX + o.I + 1] = 0;
          S[c.oE + o.I + 1] = sb * S[c.oI + o.I + 1];
        }
      }
    }
    sync(wave);
  };
  // prolongate! from level l+1 and increment!(l) (not on the coarsest), smooth!(l); x of the first
  // level goes to memory
  auto up = [&](int l, bool wave) {
    const TailLv q = d.lv[l];
    const Own o = own(q);
    T* const e = S + q.oE + o.I;
    const Coef k = coef(q, o.I);
    const T ia = S[q.oI + o.I], ib = S[q.oI + o.I + 1];
    T ra = S[q.oR + o.I], rb = S[q.oR + o.I + 1], xa = S[q.oX + o.I], xb = S[q.oX + o.I + 1];
    if (l < d.n - 1) {
      const TailLv c = d.lv[l + 1];
      const T Da = S[q.oD + o.I], Db = S[q.oD + o.I + 1];
      int qx[4], qy[3], qz[3] = {0, 0, 0};
#pragma unroll
      for (int t = 0; t < 4; ++t) qx[t] = pro_map(o.x - 1 + t, q.N0, d.perdir & 1, q.cm & 1);
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        qy[t] = pro_map(o.y - 1 + t, q.N1, (d.perdir >> 1) & 1, (q.cm >> 1) & 1);
        if (D == 3) qz[t] = pro_map(o.z - 1 + t, q.N2, (d.perdir >> 2) & 1, (q.cm >> 2) & 1);
      }
      const T* X = S + c.oX;
      auto xc = [&](int a, int b, int z) -> T {  // 0 for "no value", whose load goes to cell 0
        const bool ok = a >= 0 && b >= 0 && z >= 0;
        const T v = X[ok ? a + c.s1 * b + c.s2 * z : 0];
        return ok ? v : T(0);
      };
      const T em = xc(qx[0], qy[1], qz[1]), ea = xc(qx[1], qy[1], qz[1]);
      const T eb = xc(qx[2], qy[1], qz[1]), ep = xc(qx[3], qy[1], qz[1]);
      const T ma = xc(qx[1], qy[0], qz[1]), mb = xc(qx[2], qy[0], qz[1]);
      const T pa = xc(qx[1], qy[2], qz[1]), pb = xc(qx[2], qy[2], qz[1]);
      T sa = ea * Da, sb = eb * Db;
      sa += (em * k.x0 + eb * k.x1);
      sb += (ea * k.x1 + ep * k.x2);
      sa += (ma * k.ya + pa * k.Ya);
      sb += (mb * k.yb + pb * k.Yb);
      if (D == 3) {
        sa += (xc(qx[1], qy[1], qz[0]) * k.za + xc(qx[1], qy[1], qz[2]) * k.Za);
        sb += (xc(qx[2], qy[1], qz[0]) * k.zb + xc(qx[2], qy[1], qz[2]) * k.Zb);
      }
      ra = ra - w * sa;
      rb = rb - w * sb;
      xa = xa + w * ea;
      xb = xb + w * eb;
      if (o.a) e[0] = ra * ia;
      if (o.b) e[1] = rb * ib;
      sync(wave);
    }
    perbc(q, wave);
    // half_rangek (src/Poisson.jl:130-132) on the last axis; the sweep of colour `it` updates the
    // cells whose 0-based indices and it + D + 1 sum to an even number
    const int klim = D == 3 ? 2 * (q.N2 / 2) - 2 : 2 * (q.N1 / 2) - 2;
    const bool reach = (D == 3 ? o.z : o.y) <= klim;
    const bool exact = d.exact && l == d.n - 1 && q.n <= TAIL_CG_MAX && !d.perdir;
    if (exact) {
      if (d.exact == 2) {
        if (tid == 0) {
          SLev<T> p;
          p.N0 = q.N0; p.N1 = q.N1; p.N2 = q.N2; p.s1 = q.s1; p.s2 = q.s2; p.n = q.n;
          p.L = S + q.oL; p.r = S + q.oR; p.e = S + q.oE;
          tail_pcg<T, D>(p, cg);
        }
        sync(wave);
      } else {
        // Mixed precision: smooth! of the coarsest level in double: ϵ = r·iD and the four GS-RB half
        // sweeps (src/Poisson.jl:141-148) with ϵ, D and iD held in double, then ϵ rounded to T for
        // increment!.  Same algorithm and order as the T sweeps.  (pcg! here instead moved the
        // constant the Neumann problem leaves free in p away from the reference algorithm's: on a
        // 64x32x32 sphere, p 2.9e-3 and the force 7.5e-4 from the Float64 oracle, against 1e-4 and 5e-6.)
        double* const E = cg[0];
        for (int j = tid; j < q.n; j += wave ? 64 : TAIL_FAST_PAIRS) E[j] = 0;
        sync(wave);
        auto idiag = [&](T l0, T h0, T l1, T h1, T l2, T h2) {
          double sd = 0;
          sd -= ((double)l0 + (double)h0);
          sd -= ((double)l1 + (double)h1);
          if (D == 3) sd -= ((double)l2 + (double)h2);
          return sd == 0.0 ? 0.0 : 1.0 / sd;
        };
        const double da = idiag(k.x0, k.x1, k.ya, k.Ya, k.za, k.Za), db = idiag(k.x1, k.x2, k.yb, k.Yb, k.zb, k.Zb);
        double* const p0 = E + o.I;
        if (o.a) p0[0] = (double)ra * da;
        if (o.b) p0[1] = (double)rb * db;
        sync(wave);
        bool fa = ((o.x + o.y + o.z + 1 + D + 1) & 1) == 0;
#pragma unroll 1
        for (int it = 1; it <= 4; ++it) {
          if ((fa ? o.a : o.b) && reach) {
            double* const p = p0 + (fa ? 0 : 1);
            double sv = (double)(fa ? ra : rb);
            sv -= (p[-1] * (double)(fa ? k.x0 : k.x1) + p[1] * (double)(fa ? k.x1 : k.x2));
            sv -= (p[-q.s1] * (double)(fa ? k.ya : k.yb) + p[q.s1] * (double)(fa ? k.Ya : k.Yb));
            if (D == 3) sv -= (p[-q.s2] * (double)(fa ? k.za : k.zb) + p[q.s2] * (double)(fa ? k.Za : k.Zb));
            p[0] = sv * (fa ? da : db);
          }
          fa = !fa;
          sync(wave);
        }
        if (o.a) e[0] = (T)p0[0];
        if (o.b) e[1] = (T)p0[1];
      }
    } else {
      // sweep 1's cell of the pair: xa when the sum with it = 1 is even
      bool fa = ((o.x + o.y + o.z + 1 + D + 1) & 1) == 0;
#pragma unroll 1
      for (int it = 1; it <= 4; ++it) {
        if (fa ? o.a : o.b) {
          const T* p = e + (fa ? 0 : 1);
          const T xm = p[-1], xp = p[1], ym = p[-q.s1], yp = p[q.s1];
          T s = fa ? ra : rb;
          s -= (xm * (fa ? k.x0 : k.x1) + xp * (fa ? k.x1 : k.x2));
          s -= (ym * (fa ? k.ya : k.yb) + yp * (fa ? k.Ya : k.Yb));
          if (D == 3) s -= (p[-q.s2] * (fa ? k.za : k.zb) + p[q.s2] * (fa ? k.Za : k.Zb));
          if (reach) e[fa ? 0 : 1] = s * (fa ? ia : ib);
        }
        fa = !fa;
        if (it < 4) sync(wave);  // after sweep 4 a thread reads only its own pair's ϵ
      }
    }
    // increment!'s x += ω·ϵ (its r is dead: the next V-cycle's restrict! overwrites it)
    if (l == 0) {
      const int64_t I = o.I;
      if (o.a) d.x[I] = xa + w * e[0];
      if (o.b) d.x[I + 1] = xb + w * e[1];
    } else {
      if (o.a) S[q.oX + o.I] = xa + w * e[0];
      if (o.b) S[q.oX + o.I + 1] = xb + w * e[1];
      sync(wave);
    }
  };
  // one loop over the visits: each one's code is there once (a launch runs it from cold lines)
  bool was_wave = false;
#pragma unroll 1
  for (int k = 0; k < 2 * d.n - 1; ++k) {
    const bool dn = k < d.n - 1;
    const int l = dn ? k : 2 * (d.n - 1) - k;
    const bool wave = d.lv[l].small != 0;
    if (was_wave && !wave) __syncthreads();
    was_wave = wave;
    if (wave && tid >= 64) continue;
    if (dn) down(l, wave); else up(l, wave);
  }
}
template <class T, int D>
__global__ void __launch_bounds__(TAIL_FAST_PAIRS) k_mg_tail_fast(TailFast<T> d, const T* __restrict__ wp) {
  __shared__ double cg[5][TAIL_CG_MAX];
  k_mg_tail_fast_body<T, D>(d, wp, cg);
}

// ---- the up-leg of one level in one launch ----
// prolongate! from level l+1, increment!(l), ϵ = r·iD, the four GS-RB half sweeps and smooth!'s
// increment! of a flow's own solver (src/MultiLevelPoisson.jl:98-100, src/Poisson.jl:100-148); x of
// the level comes out final, r and ϵ stay on the chip (the next V-cycle overwrites them).
//
// As separate launches (one prolongation, four half sweeps, the increment in the next finer
// prolongation) a level below a million cells costs five launches of 3-5 us, each moving a few MB
// that sit in the caches.  Here a block takes a region of 64 x 32 cells (2D) or 16 x 16 x 12 (3D)
// around its output tile: stage s of a cell needs stage s − 1 of its neighbours, so the halo is the
// four half sweeps' (FIN: one more, for the residual), which the blocks recompute.  A thread owns
// x pairs of the region (one in 2D, two in 3D), one cell of which each half sweep updates, and
// keeps their residuals, 1/D and coefficients in registers; the LDS carries ϵ, and before it the
// prolonged coarse values.  Every value is formed by the operations of the separate passes in their
// order, so the results are the same bits; only FIN's Σr² is summed over other tiles.
//
// FIN (the finest level): also r −= ω·Aϵ into rout (the neighbouring blocks still read r), the next
// Jacobi!'s ϵ = r·iD into ej and the block's Σr² into partial.
// Periodic directions: ghosts hold perBC!'s image of the first ϵ for all four half sweeps, as in the
// reference; FIN needs the images of the last and takes no periodic directions.
template <class T>
struct UpArgs {
  Geo gf, gc;
  int cm, perdir;
  LRows<T> L;
  const T* r;
  T* x;
  const T* xc;
  const T* w;
  T* rout;
  T* ej;
  double* partial;
  int ntx, nty;  // output tiles in x and y
};
template <int D, bool FIN>
struct UpTile {
  static constexpr int H = FIN ? 5 : 4;
  static constexpr int LX = D == 3 ? 3 : 5, LY = D == 3 ? 4 : 5;  // log2 of the pairs and rows
  static constexpr int RX = 2 << LX, RY = 1 << LY, RZ = D == 3 ? 12 : 1;
  static constexpr int OX = RX - 2 * H, OY = RY - 2 * H, OZ = D == 3 ? RZ - 2 * H : 1;
  static constexpr int SX = RX + 2, SY = RY + 2, SZ = D == 3 ? RZ + 2 : 1;  // with a ring of one cell
  static constexpr int NI = D == 3 ? 2 : 1, DZ = RZ / NI;                   // pairs per thread, planes apart
  static constexpr int THREADS = (RX / 2) * RY * DZ;
};
template <class T, int D, bool FIN>
constexpr size_t up_lds() {
  using U = UpTile<D, FIN>;
  return sizeof(T) * U::SX * U::SY * U::SZ;
}
// The face coefficients of an x pair (cells 0 and 1): x faces x0, x1, x2; y and z faces low and high
template <class T, int D>
struct PairCoef {
  T x0, x1, x2, yl[2], yh[2], zl[D == 3 ? 2 : 1], zh[D == 3 ? 2 : 1];
  __device__ __forceinline__ T diag(int c) const {
    T s = 0;
    s -= ((c ? x1 : x0) + (c ? x2 : x1));
    s -= (yl[c] + yh[c]);
    if constexpr (D == 3) s -= (zl[c] + zh[c]);
    return s;
  }
  // x(I)·D + Σ_i (x(I−e_i)·L[I,i] + x(I+e_i)·L[I+e_i,i]) at cell c, where p stands (s = x(I)·D)
  __device__ __forceinline__ T mult(int c, T s, const T* p, int sy, int sz) const {
    s += (p[-1] * (c ? x1 : x0) + p[1] * (c ? x2 : x1));
    s += (p[-sy] * yl[c] + p[sy] * yh[c]);
    if constexpr (D == 3) s += (p[-sz] * zl[c] + p[sz] * zh[c]);
    return s;
  }
  // gauss (src/Poisson.jl:116-122) before the product with iD; first: cell 0, where p stands
  __device__ __forceinline__ T gauss(bool first, T s, const T* p, int sy, int sz) const {
    const T xm = p[-1], xp = p[1], ym = p[-sy], yp = p[sy];
    T zm = T(0), zp = T(0);
    if constexpr (D == 3) {
      zm = p[-sz];
      zp = p[sz];
    }
    s -= (xm * (first ? x0 : x1) + xp * (first ? x1 : x2));
    s -= (ym * (first ? yl[0] : yl[1]) + yp * (first ? yh[0] : yh[1]));
    if constexpr (D == 3) s -= (zm * (first ? zl[0] : zl[1]) + zp * (first ? zh[0] : zh[1]));
    return s;
  }
};
// from the two cells' own coefficients; h of cell 0 and l of cell 1 in x are one face, taken from
// cell 0 where it has a value (va)
template <class T, int D>
__device__ __forceinline__ PairCoef<T, D> pair_coef(const LC<T>& a, const LC<T>& b, bool va) {
  PairCoef<T, D> c;
  c.x0 = a.l[0]; c.x1 = va ? a.h[0] : b.l[0]; c.x2 = b.h[0];
  c.yl[0] = a.l[1]; c.yh[0] = a.h[1]; c.yl[1] = b.l[1]; c.yh[1] = b.h[1];
  if constexpr (D == 3) {
    c.zl[0] = a.l[2]; c.zh[0] = a.h[2]; c.zl[1] = b.l[2]; c.zh[1] = b.h[2];
  }
  return c;
}
template <class T, int D, bool FIN>
__device__ __forceinline__ void k_up_body(const UpArgs<T>& a, int lid, int pidx) {
  using U = UpTile<D, FIN>;
  constexpr int H = U::H, NI = U::NI, SX = U::SX, SXY = U::SX * U::SY;
  extern __shared__ __align__(16) unsigned char up_smem[];
  T* const S = reinterpret_cast<T*>(up_smem);  // SXY·SZ values
  const T w = *a.w;
  const int tid = threadIdx.x;
  const int N[3] = {a.gf.N[0], a.gf.N[1], a.gf.N[2]};
  const int tx = lid % a.ntx, t1 = lid / a.ntx, ty = t1 % a.nty, tz = t1 / a.nty;
  // the region's first cell
  const int bx = 1 + tx * U::OX - H, by = 1 + ty * U::OY - H, bz = D == 3 ? 1 + tz * U::OZ - H : 0;
  // the inside cell whose value stands at coordinate c of direction q: itself, the image of a
  // periodic ghost (or of the cell one beyond it), or none (−1)
  auto image = [&](int c, int q) -> int {
    const int n = N[q];
    if (c >= 1 && c <= n - 2) return c;
    if (!((a.perdir >> q) & 1) || c < -1 || c > n) return -1;
    return c < 1 ? c + (n - 2) : c - (n - 2);
  };
  // ---- the prolonged coarse values of the region and one cell around it ----
  {
    constexpr int NS = SXY * U::SZ;
#pragma unroll 4
    for (int k = tid; k < NS; k += U::THREADS) {
      const int cx = image(bx - 1 + k % SX, 0), cy = image(by - 1 + (k / SX) % U::SY, 1);
      const int cz = D == 3 ? image(bz - 1 + k / SXY, 2) : 0;
      const bool ok = cx >= 0 && cy >= 0 && cz >= 0;
      const int qx = (a.cm & 1) ? (cx + 1) >> 1 : cx, qy = (a.cm & 2) ? (cy + 1) >> 1 : cy;
      const int qz = D == 3 ? ((a.cm & 4) ? (cz + 1) >> 1 : cz) : 0;
      const T v = a.xc[ok ? qx + a.gc.s[1] * qy + a.gc.s[2] * qz : 0];
      S[k] = ok ? v : T(0);
    }
  }
  const int lp = tid & ((1 << U::LX) - 1), ly = (tid >> U::LX) & ((1 << U::LY) - 1), lz0 = D == 3 ? tid >> (U::LX + U::LY) : 0;
  const int cx = bx + 2 * lp, cy = by + ly;
  const int s0 = 1 + 2 * lp + SX * (1 + ly);  // LDS index of the pair's first cell in plane −1 (3D) or 0
  const int mxa = image(cx, 0), mxb = image(cx + 1, 0), my = image(cy, 1);
  const int klim = D == 3 ? 2 * (N[2] / 2) - 2 : 2 * (N[1] / 2) - 2;
  const bool ixa = cx >= 1 && cx <= N[0] - 2, ixb = cx + 1 >= 1 && cx + 1 <= N[0] - 2, iy = cy >= 1 && cy <= N[1] - 2;
  T ra[NI], rb[NI], ia[NI], ib[NI], xa[NI], xb[NI];
  PairCoef<T, D> C[NI];
  // a cell without a value takes the first inside cell's coefficients; its ϵ is set to 0 below
  auto coef = [&](int i) -> PairCoef<T, D> {
    const int mz = D == 3 ? image(bz + lz0 + U::DZ * i, 2) : 0;
    const bool row = my >= 0 && mz >= 0;
    const int y = row ? my : 1, z = D == 3 ? (row ? mz : 1) : 0;
    return pair_coef<T, D>(lcell(a.gf, a.L, row && mxa >= 0 ? mxa : 1, y, z),
                           lcell(a.gf, a.L, row && mxb >= 0 ? mxb : 1, y, z), mxa >= 0);
  };
  uint32_t fl = 0;  // per pair: 1, 2 updated by the sweeps; 4, 8 output cells
#pragma unroll
  for (int i = 0; i < NI; ++i) {  // the pairs' own loads, before the barrier
    const int cz = D == 3 ? bz + lz0 + U::DZ * i : 0;
    const int mz = D == 3 ? image(cz, 2) : 0;
    const bool iz = D == 2 || (cz >= 1 && cz <= N[2] - 2);
    const bool row = my >= 0 && mz >= 0;
    const bool reach = (D == 3 ? cz : cy) <= klim;
    const bool oy = ly >= H && ly < H + U::OY && (D == 2 || (lz0 + U::DZ * i >= H && lz0 + U::DZ * i < H + U::OZ));
    const bool in = iy && iz;
    const bool oa = in && ixa && oy && 2 * lp >= H && 2 * lp < H + U::OX;
    const bool ob = in && ixb && oy && 2 * lp + 1 >= H && 2 * lp + 1 < H + U::OX;
    fl |= (uint32_t)((in && ixa && reach ? 1 : 0) | (in && ixb && reach ? 2 : 0) | (oa ? 4 : 0) | (ob ? 8 : 0)) << (4 * i);
    const int64_t rowI = row ? a.gf.s[1] * my + a.gf.s[2] * mz : 0;
    const bool va = row && mxa >= 0, vb = row && mxb >= 0;
    ra[i] = va ? a.r[rowI + mxa] : T(0);
    rb[i] = vb ? a.r[rowI + mxb] : T(0);
    xa[i] = oa ? a.x[rowI + mxa] : T(0);
    xb[i] = ob ? a.x[rowI + mxb] : T(0);
    C[i] = coef(i);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NI; ++i) {  // increment! with the prolonged values, ϵ = r·iD
    const T* p = S + s0 + (D == 3 ? SXY * (1 + lz0 + U::DZ * i) : 0);
    const PairCoef<T, D>& c = C[i];
    const T e0 = p[0], e1 = p[1];
    const T Da = c.diag(0), Db = c.diag(1);
    ra[i] = ra[i] - w * c.mult(0, e0 * Da, p, SX, SXY);
    rb[i] = rb[i] - w * c.mult(1, e1 * Db, p + 1, SX, SXY);
    xa[i] = xa[i] + w * e0;
    xb[i] = xb[i] + w * e1;
    ia[i] = inv_diag(Da);
    ib[i] = inv_diag(Db);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NI; ++i) {  // ghosts and cells beyond hold 0; periodic ghosts their image's ϵ
    const int cz = D == 3 ? bz + lz0 + U::DZ * i : 0;
    const bool row = my >= 0 && (D == 2 || image(cz, 2) >= 0);
    T* p = S + s0 + (D == 3 ? SXY * (1 + lz0 + U::DZ * i) : 0);
    p[0] = row && mxa >= 0 ? ra[i] * ia[i] : T(0);
    p[1] = row && mxb >= 0 ? rb[i] * ib[i] : T(0);
  }
  __syncthreads();
#pragma unroll 1
  for (int it = 1; it <= 4; ++it) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int cz = D == 3 ? bz + lz0 + U::DZ * i : 0;
      const bool fa = ((cx + cy + cz + it + D + 1) & 1) == 0;  // the pair's cell of this sweep's colour
      if ((fl >> (4 * i + (fa ? 0 : 1))) & 1) {
        T* p = S + s0 + (D == 3 ? SXY * (1 + lz0 + U::DZ * i) : 0) + (fa ? 0 : 1);
        const T s = C[i].gauss(fa, fa ? ra[i] : rb[i], p, SX, SXY);
        p[0] = s * (fa ? ia[i] : ib[i]);
      }
    }
    if (it < 4 || FIN) __syncthreads();
  }
  double acc = 0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {  // smooth!'s increment!
    const int cz = D == 3 ? bz + lz0 + U::DZ * i : 0;
    const bool oa = (fl >> (4 * i)) & 4, ob = (fl >> (4 * i)) & 8;
    const T* p = S + s0 + (D == 3 ? SXY * (1 + lz0 + U::DZ * i) : 0);
    const int64_t I = cx + a.gf.s[1] * cy + a.gf.s[2] * cz;
    const T e0 = p[0], e1 = p[1];
    if (oa) a.x[I] = xa[i] + w * e0;
    if (ob) a.x[I + 1] = xb[i] + w * e1;
    if (FIN) {
      const PairCoef<T, D>& c = C[i];
      const T na = ra[i] - w * c.mult(0, e0 * c.diag(0), p, SX, SXY);
      const T nb2 = rb[i] - w * c.mult(1, e1 * c.diag(1), p + 1, SX, SXY);
      if (oa) {
        a.rout[I] = na;
        a.ej[I] = na * ia[i];
        acc += (double)na * (double)na;
      }
      if (ob) {
        a.rout[I + 1] = nb2;
        a.ej[I + 1] = nb2 * ib[i];
        acc += (double)nb2 * (double)nb2;
      }
    }
  }
  if (FIN) {
    const double t = block_sum(acc);
    if (tid == 0) a.partial[pidx] = t;
  }
}
template <class T, int D, bool FIN>
__global__ void __launch_bounds__((UpTile<D, FIN>::THREADS)) k_up(UpArgs<T> a) {
  k_up_body<T, D, FIN>(a, xcd_tile_id(), (int)blockIdx.x);
}

}  // namespace wl
