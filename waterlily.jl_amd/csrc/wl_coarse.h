// The coarse end of the V-cycle, where a pass over a level costs its latency and not its bytes:
// the single-workgroup tail (k_mg_tail_fast, and its general form k_mg_tail_lds).
//
// Included by wl_kernels.h after the per-cell pieces it uses (LRows, lcell, pro_map, TailDesc).
#pragma once

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
//  - a thread owns x pairs: every half sweep updates one cell of each pair and no lane idles, and a
//    level's pairs are dealt to the threads by shifts chosen from its own extents;
//  - levels of at most 128 pairs run in the first wave alone, two pairs to a lane at most: the LDS
//    serves a wave in order, so their passes need no barrier (the other waves wait at one);
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
    pair_loop(q, lnt, [&](int x, int y, int z) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        if (x + o > q.N0 - 2) continue;
        const int I = x + o + q.s1 * y + q.s2 * z;
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
      }
    });
  }
  __syncthreads();

  // Jacobi!'s increment! (ω = 1): a cell reads ϵ, which no thread writes, and updates its own r and x
  auto jacobi = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l);
    perbc(f, f.e, ln, wave);
    pair_loop(f, ln, [&](int x, int y, int z) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        if (x + o > f.N0 - 2) continue;
        const int I = x + o + f.s1 * y + f.s2 * z;
        f.r[I] = f.r[I] - T(1) * smult(f, f.e, I);
        f.x[I] = f.x[I] + T(1) * f.e[I];
      }
    });
    sync(wave);
  };
  // restrict! to level l+1, fill!(x, 0) and ϵ = r·iD there: children summed in z, y, x order
  auto restrict_to = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l), c = lev(l + 1);
    pair_loop(c, ln, [&](int x, int y, int z) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        if (x + o > c.N0 - 2) continue;
        const int cc[3] = {x + o, y, z};
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
        const int Ic = x + o + c.s1 * y + c.s2 * z;
        c.r[Ic] = s;
        c.x[Ic] = 0;
        c.e[Ic] = s * c.iD[Ic];
      }
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
      pair_loop(p, ln, [&](int x, int y, int z) {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          if (x + o > p.N0 - 2) continue;
          const int I = x + o + p.s1 * y + p.s2 * z;
          if (KEEP) {
            p.r[I] = p.r[I] - w * smult(p, p.e, I);
            p.x[I] = p.x[I] + w * p.e[I];
          } else {
            xinc(I);
          }
        }
      });
      sync(wave);
    }
  };
  // prolongate! from level l+1, increment!(l) and ϵ = r·iD for the smooth! that follows
  auto prolong = [&](int l, int ln, bool wave) {
    const SLev<T> f = lev(l), p = lev(l + 1);
    const int N[3] = {f.N0, f.N1, f.N2};
    pair_loop(f, ln, [&](int x, int y, int z) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        if (x + o > f.N0 - 2) continue;
        const int c[3] = {x + o, y, z};
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
        const int I = x + o + f.s1 * y + f.s2 * z;
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
      }
    });
    sync(wave);
  };

  // The passes in order, one loop over them: each pass's code is there once (a launch runs it from
  // cold instruction lines).  ls: the first level of the first wave's part (pairs shrink with the
  // level); a pass belongs to the level it starts from on the way down, and ends at on the way up.
  int ls = d.n;
  while (ls > 0 && lev(ls - 1).npair <= WAVE_PAIRS) --ls;
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
// levels lie in one image in memory, formed when L changes (k_tail_image), so one round of loads
// brings them in.
struct TailLv {           // one level; built on the host, read with scalar loads
  int N0, N1, N2;
  int s1, s2, n, cm;
  int lx, ly;             // log2 of the threads along x (pairs) and y
  int oL, oD, oI;         // LDS element offsets: L (D arrays of n), D, 1/D ...
  int oR, oX, oE;         // ... r, x, ϵ
  int small;              // run by the first wave alone
};
template <class T>
struct TailFast {
  int n, perdir, exact, nimg;  // levels; image elements
  const T* img;                // L, D, 1/D of every level, as the LDS holds them
  const T* r;                  // the first level's residual
  T* x;                        // the first level's x (ghosts untouched)
  TailLv lv[TAIL_MAX_LEVELS];
};
constexpr int TAIL_FAST_PAIRS = 1024, TAIL_WAVE_PAIRS = 64;
// L, D and 1/D of one level into the image: D and 1/D on inside as set_diag! forms them
// (src/Poisson.jl:43-46), 0 on ghosts
template <class T>
__global__ void __launch_bounds__(256) k_tail_image(Geo g, const T* __restrict__ L, T* __restrict__ img) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= g.n) return;
  for (int i = 0; i < g.D; ++i) img[k + i * g.n] = L[k + i * g.n];
  const int c[3] = {(int)(k % g.N[0]), (int)((k / g.N[0]) % g.N[1]), (int)(k / g.s[2])};
  bool in = true;
  for (int q = 0; q < g.D; ++q) in &= c[q] >= 1 && c[q] <= g.N[q] - 2;
  const T Dg = in ? diag_at<T>(g, L, k) : T(0);
  img[k + g.D * g.n] = Dg;
  img[k + (g.D + 1) * g.n] = in ? inv_diag(Dg) : T(0);
}
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

}  // namespace wl
