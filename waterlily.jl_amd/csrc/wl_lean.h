// The V-cycle passes of a large 3D level that keep Jacobi!'s and the prolongation's results on the
// chip (a flow's own solver without periodic directions, levels coarsened in every direction, x
// pairs per lane as in k_gs_half2).
//
// The plain passes store, per level and V-cycle, the Jacobi ϵ, r and x after Jacobi!, r, x and ϵ
// after the prolongation, and r and x after smooth!: 24.7 values per cell with the four half sweeps,
// in passes that run at the memory's rate.  Most of it can be formed again from the residual r₀ the
// V-cycle starts from (ϵ_J = r₀·iD, seven values) and the coarse x, which is an eighth of the level:
//   k_lean_restrict    reads r₀, writes the coarse r                                 1.1 values
//   k_lean_prolong     reads r₀ and the coarse x, writes r₂ = r₀ − Aϵ_J − ω·Ae_c       2.25
//   k_lean_gs_first    reads r₂ (whose r₂·iD is the ϵ the sweep starts from), writes one colour  1.5
//   k_lean_gs × 3      one colour of ϵ read and written each, r₂'s lines               6
//   k_lean_increment   reads r₀, r₂, ϵ, x and the coarse x; writes x and r           6.25
// 17.1 values.  x of a coarser level is written by the prolongation (ϵ_J + ω·e_c), of the finest by
// the increment alone.  Each value is formed by the plain passes' operations in their order; only Σr² is
// summed over other tiles.
//
// Bound by memory: FP32 512x256x256 with a sphere, us per launch, plain -> lean: restriction 227 -> 75,
// prolongation 190 -> 131, half sweep 81 -> 76, increment 208 -> 210 (it has taken over x's part of the
// others), the projection's residual, which no longer writes ϵ and a mean-free source, 314 -> 211; the
// step 7592 -> 6258.
//
// Away from bodies a level's coefficients are its constants, 0 on wall faces.  Where that holds for a
// wave's 128 cells of a row, the cells beside them and the four neighbour rows (k_seg_*, one flag per
// row and 128 cells), D and 1/D are constants too, by the walls the row lies at, and nothing is loaded
// for them; elsewhere the wave reads L and 1/D (iD, formed with the flags).  The choice is uniform in
// a wave, one branch per plane.  (With flags for whole rows, walls excluded, 9% of the rows read L and
// took a third of the time: 90 us per half sweep at 512x256x256 against 57 without them.)
// Ghosts of r₀, r₂, x and ϵ are 0.
//
// Included by wl_kernels.h after the pair kernels.
#pragma once

namespace wl {

constexpr int SEG_PAIRS = 64;  // pairs of a row per flag: a wave's
inline int lean_nseg(const Geo& g) { return ((g.N[0] - 2) / 2 + SEG_PAIRS - 1) / SEG_PAIRS; }
template <class T>
struct LeanL {
  const T* L;
  const T* iD;
  const uint8_t* fast;  // flags (k_seg_fast); nullptr: every wave reads L and iD
  int nseg;
  T c0, c1, c2;         // the uniform face coefficients
  // 1/D of a uniform cell: [at a y wall][at a z wall], in the middle of x and beside an x wall
  T im[2][2], iw[2][2];
};
// 1/D formed on the host by diag_at's and inv_diag's operations
template <class T>
inline LeanL<T> lean_l(const T* L, const T* iD, const uint8_t* fast, int nseg, const T* c) {
  LeanL<T> a{L, iD, fast, nseg, c[0], c[1], c[2], {{T(0), T(0)}, {T(0), T(0)}}, {{T(0), T(0)}, {T(0), T(0)}}};
  for (int xw = 0; xw < 2; ++xw)
    for (int yw = 0; yw < 2; ++yw)
      for (int zw = 0; zw < 2; ++zw) {
        T s = 0;
        s -= (xw ? c[0] : c[0] + c[0]);
        s -= (yw ? c[1] : c[1] + c[1]);
        s = s - (zw ? c[2] : c[2] + c[2]);
        (xw ? a.iw : a.im)[yw][zw] = s == T(0) ? s : T(1) / s;
      }
  return a;
}
// Flags.  Pass 1, one wave per row and segment: bit i: component i has its constant (0 on wall faces)
// over the segment's cells and those beside them, the x faces one further; and 1/D of its cells (k_diag's)
template <class T>
__global__ void __launch_bounds__(256) k_seg_bits(Geo g, const T* __restrict__ L, T c0, T c1, T c2, int nseg,
                                                  uint8_t* __restrict__ bits, T* __restrict__ iD) {
  const int64_t w = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (w >= (int64_t)g.N[1] * g.N[2] * nseg) return;  // uniform over the wavefront
  const int seg = (int)(w % nseg);
  const int64_t row = w / nseg;
  const int y = (int)(row % g.N[1]), z = (int)(row / g.N[1]);
  const int x0 = 2 * SEG_PAIRS * seg, x1 = min(x0 + 2 * SEG_PAIRS + 1, g.N[0] - 1);  // the cells beside included
  const int64_t base = at(g, 0, y, z);
  const T e1 = (y == 1 || y == g.N[1] - 1) ? T(0) : c1, e2 = (z == 1 || z == g.N[2] - 1) ? T(0) : c2;
  const bool inside = y >= 1 && y <= g.N[1] - 2 && z >= 1 && z <= g.N[2] - 2;
  const int64_t dy = inside ? g.s[1] : 0, dz = inside ? g.s[2] : 0;
  const T *L0 = L + base, *L1 = L0 + g.n, *L2 = L1 + g.n;
  bool a0 = true, a1 = true, a2 = true;
#pragma unroll
  for (int k = 0; k < 3; ++k) {  // no branch before the loads: a cell beyond repeats the last one
    const int x = x0 + lane + 64 * k;
    const int xf = min(max(x, 1), min(x1 + 1, g.N[0] - 1)), xc = min(max(x, 1), min(x1, g.N[0] - 2));
    const T f = L0[xf], xl = L0[xc], xh = L0[xc + 1];
    const T yl = L1[xc], yh = L1[xc + dy], zl = L2[xc], zh = L2[xc + dz];
    a0 &= same_bits(f, (xf == 1 || xf == g.N[0] - 1) ? T(0) : c0);
    a1 &= same_bits(yl, e1);
    a2 &= same_bits(zl, e2);
    T s = 0;  // diag_at's order
    s -= (xl + xh);
    s -= (yl + yh);
    s -= (zl + zh);
    if (inside && x > x0 && x < x1) iD[base + x] = inv_diag(s);
  }
  const bool b0 = __all(a0), b1 = __all(a1), b2 = __all(a2);
  if (lane == 0) bits[w] = (uint8_t)(b0 | (b1 << 1) | (b2 << 2));
}
// Pass 2: every face of the segment's cells (an inside row).  Pass 3: that of the row and of its four
// neighbours (ghost rows hold 0 and need no coefficient), and the level's row flags (LRows: a row whose
// y and z faces are no walls).
// Pass 1 is bound by its read of L: 159 us at 512x256x256, for 143 + 139 + 198 of a pass without 1/D,
// k_diag and k_level_tables; a measure! and update! there 1325 -> 998 us.
__global__ void __launch_bounds__(256) k_seg_uniform(Geo g, int nseg, const uint8_t* __restrict__ bits,
                                                     uint8_t* __restrict__ uni) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (int64_t)g.N[1] * g.N[2] * nseg) return;
  const int64_t row = k / nseg, sy = nseg, sz = (int64_t)g.N[1] * nseg;
  const int y = (int)(row % g.N[1]), z = (int)(row / g.N[1]);
  bool f = y >= 1 && y <= g.N[1] - 2 && z >= 1 && z <= g.N[2] - 2;
  if (f) f = bits[k] == 7 && (bits[k + sy] & 2) && (bits[k + sz] & 4);
  uni[k] = f ? 1 : 0;
}
__global__ void __launch_bounds__(256) k_seg_fast(Geo g, int nseg, const uint8_t* __restrict__ uni,
                                                  uint8_t* __restrict__ fast, uint8_t* __restrict__ rows) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= (int64_t)g.N[1] * g.N[2] * nseg) return;
  const int64_t row = k / nseg, sy = nseg, sz = (int64_t)g.N[1] * nseg;
  const int y = (int)(row % g.N[1]), z = (int)(row / g.N[1]);
  bool f = y >= 1 && y <= g.N[1] - 2 && z >= 1 && z <= g.N[2] - 2;
  if (f)
    f = uni[k] && (y == 1 || uni[k - sy]) && (y == g.N[1] - 2 || uni[k + sy]) && (z == 1 || uni[k - sz]) &&
        (z == g.N[2] - 2 || uni[k + sz]);
  fast[k] = f ? 1 : 0;
  if (k == row * nseg) {
    bool r = y >= 2 && y <= g.N[1] - 3 && z >= 2 && z <= g.N[2] - 3;
    for (int s = 0; s < nseg; ++s) r = r && uni[k + s];
    rows[row] = r ? 1 : 0;
  }
}
// the flags of row y and a segment over planes zlo + lane (lanes below nz)
template <class T>
__device__ __forceinline__ uint32_t lean_flags(const Geo& g, const LeanL<T>& A, int seg, int y, int zlo, int nz, int lane) {
  return (lane < nz && A.fast != nullptr && A.fast[(y + (int64_t)g.N[1] * (zlo + lane)) * A.nseg + seg] != 0) ? 1u : 0u;
}
// A wave's loads and stores: a base that is uniform in the wave (a row of a plane, in scalar registers)
// and one 32-bit byte offset per lane, the same for every row of a field, so stepping to the next
// plane costs scalar adds only (WL_KEEP_OFFSET keeps the compiler from widening the offset to 64 bits
// outside the loop, which would cost an addition per load).  Planes come in pairs (odd, even), written
// out, and every load of the planes ahead is issued whatever the plane (on a tile's last plane it reads
// one already read): behind a branch the wait for the current plane's values became a wait for all.
template <class T>
__device__ __forceinline__ T ldo(const T* base, uint32_t b) {
  return *(const T*)((const char*)base + b);
}
template <class T>
__device__ __forceinline__ P2<T> ldo2(const T* base, uint32_t b) {
  return ld2((const T*)((const char*)base + b));
}
template <class T>
__device__ __forceinline__ void sto2(T* base, uint32_t b, T x, T y) {
  st2((T*)((char*)base + b), x, y);
}
#define WL_KEEP_OFFSET(o) asm volatile("" : "+v"(o))
// Slabs of zc planes go round-robin to the XCDs, each walking its slab's tiles in order: a body's rows,
// which read their coefficients, lie in few neighbouring slabs and would keep two or three XCDs busy
// alone if each had one contiguous range (xcd_tile_id): half sweep 84 -> 77 us, prolongation 152 -> 130
// at 512x256x256.  A last part of fewer than 8 slabs keeps the launch's order.
__device__ __forceinline__ int lean_tile(const ZT& t) {
  const int per = t.nbx * t.nby, slabs = (int)gridDim.x / per, b = (int)blockIdx.x;
  const int j = b >> 3;
  return b < (slabs & ~7) * per ? ((j / per) * 8 + (b & 7)) * per + j % per : b;
}
// a tile's row for this wave: y uniform
__device__ __forceinline__ PairCell lean_cell(const ZT& t) {
  PairCell c;
  const int lid = lean_tile(t);
  const int tx = lid % t.nbx, r1 = lid / t.nbx, ty = r1 % t.nby, tz = r1 / t.nby;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  c.p = t.b.lo[0] + tx * t.sx + (int)threadIdx.x;
  c.y = t.b.lo[1] + ty * t.sy + wv;
  c.z0 = t.b.lo[2] + tz * t.zc;
  c.z1 = c.z0 + t.zc - 1 < t.b.hi[2] ? c.z0 + t.zc - 1 : t.b.hi[2];
  c.vx = c.p <= t.b.hi[0];
  c.xa = 1 + 2 * (c.vx ? c.p : t.b.hi[0]);
  c.edge_r = threadIdx.x == 63 || c.p >= t.b.hi[0];
  return c;
}
template <bool B>
struct FlagC {
  static constexpr bool value = B;
};
// The coefficients, D and 1/D of a pair's cells in row y of plane z: FAST the constants
template <class T>
struct PairLD {
  T xa, xm, xb;                              // x faces: low of a, between, high of b
  T ya, yb, Ya, Yb, za, zb, Za, Zb;          // y and z faces, low and high
  T Da, Db;
  // x(I)·D + Σ_i (x(I−e_i)·L[I,i] + x(I+e_i)·L[I+e_i,i]) of both cells (src/Poisson.jl:70-76)
  __device__ __forceinline__ T ma(T l, const P2<T>& v, const P2<T>& ym, const P2<T>& yp, const P2<T>& zm, const P2<T>& zp) const {
    T s = v.a * Da;
    s += (l * xa + v.b * xm);
    s += (ym.a * ya + yp.a * Ya);
    s += (zm.a * za + zp.a * Za);
    return s;
  }
  __device__ __forceinline__ T mb(T r, const P2<T>& v, const P2<T>& ym, const P2<T>& yp, const P2<T>& zm, const P2<T>& zp) const {
    T s = v.b * Db;
    s += (v.a * xm + r * xb);
    s += (ym.b * yb + yp.b * Yb);
    s += (zm.b * zb + zp.b * Zb);
    return s;
  }
};
// A plane's form: coefficients from memory, or the constants with the z walls tested, or those of a
// plane two away from the z walls
enum LeanMode { LEAN_MEM = 0, LEAN_WALL = 1, LEAN_MID = 2 };
template <int M>
struct ModeC {
  static constexpr int value = M;
};
// The constants of a wave's row (y) and of its neighbour rows, for this lane's pair: the x faces at its
// ends, the row's y faces, −(x faces) − (y faces) as diag_at sums them, and 1/D per row [own, y−1, y+1]
// in the middle of z
template <class T>
struct PairU {
  bool lw, hw;
  T xa, xb, yl, yh, sa, sb;
  int yw[3];  // at a y wall: own row, row y−1, row y+1
  T ia[3], ib[3];
  __device__ __forceinline__ T id(const LeanL<T>& A, int row, int zw, bool b) const {
    return (b ? hw : lw) ? A.iw[yw[row]][zw] : A.im[yw[row]][zw];
  }
};
template <class T>
__device__ __forceinline__ PairU<T> pair_u(const Geo& g, const LeanL<T>& A, int xa, int y) {
  PairU<T> u;
  u.lw = xa == 1;
  u.hw = xa + 1 == g.N[0] - 2;
  u.xa = u.lw ? T(0) : A.c0;
  u.xb = u.hw ? T(0) : A.c0;
  u.yl = y == 1 ? T(0) : A.c1;
  u.yh = y == g.N[1] - 2 ? T(0) : A.c1;
  T s = 0;
  s -= (u.xa + A.c0);
  u.sa = s - (u.yl + u.yh);
  s = 0;
  s -= (A.c0 + u.xb);
  u.sb = s - (u.yl + u.yh);
  u.yw[0] = y == 1 || y == g.N[1] - 2;
  u.yw[1] = y == 2;
  u.yw[2] = y == g.N[1] - 3;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    u.ia[k] = u.id(A, k, 0, false);
    u.ib[k] = u.id(A, k, 0, true);
  }
  return u;
}
__device__ __forceinline__ bool at_zwall(const Geo& g, int z) { return z == 1 || z == g.N[2] - 2; }
// R: the row's element offset in a field, o: the lane's byte offset of xa
template <int M, class T>
__device__ __forceinline__ PairLD<T> pair_ld(const Geo& g, const LeanL<T>& A, int64_t R, uint32_t o, const PairU<T>& u, int z) {
  PairLD<T> c;
  if constexpr (M != LEAN_MEM) {
    c.xa = u.xa;
    c.xm = A.c0;
    c.xb = u.xb;
    c.ya = c.yb = u.yl;
    c.Ya = c.Yb = u.yh;
    c.za = c.zb = (M == LEAN_WALL && z == 1) ? T(0) : A.c2;
    c.Za = c.Zb = (M == LEAN_WALL && z == g.N[2] - 2) ? T(0) : A.c2;
    c.Da = u.sa - (c.za + c.Za);
    c.Db = u.sb - (c.zb + c.Zb);
  } else {
    const T* L = A.L + R;
    const P2<T> x = ldo2(L, o), y = ldo2(L + g.n, o), Y = ldo2(L + g.n + g.s[1], o);
    const P2<T> zl = ldo2(L + 2 * g.n, o), Z = ldo2(L + 2 * g.n + g.s[2], o);
    c.xa = x.a; c.xm = x.b; c.xb = ldo(L + 2, o);
    c.ya = y.a; c.yb = y.b; c.Ya = Y.a; c.Yb = Y.b;
    c.za = zl.a; c.zb = zl.b; c.Za = Z.a; c.Zb = Z.b;
    T s = 0;  // diag_at's order
    s -= (c.xa + c.xm);
    s -= (c.ya + c.Ya);
    c.Da = s - (c.za + c.Za);
    s = 0;
    s -= (c.xm + c.xb);
    s -= (c.yb + c.Yb);
    c.Db = s - (c.zb + c.Zb);
  }
  return c;
}
// 1/D of the pair in the row at R: row 0 own, 1: y−1, 2: y+1, in plane z
template <int M, class T>
__device__ __forceinline__ P2<T> pair_id(const Geo& g, const LeanL<T>& A, int64_t R, uint32_t o, const PairU<T>& u, int row, int z) {
  if constexpr (M == LEAN_MEM) return ldo2(A.iD + R, o);
  else if constexpr (M == LEAN_WALL) return at_zwall(g, z) ? P2<T>{u.id(A, row, 1, false), u.id(A, row, 1, true)} : P2<T>{u.ia[row], u.ib[row]};
  else return P2<T>{u.ia[row], u.ib[row]};
}
template <int M, class T>
__device__ __forceinline__ P2<T> eps_j(const Geo& g, const LeanL<T>& A, const P2<T>& v, int64_t R, uint32_t o, const PairU<T>& u,
                                       int row, int z) {
  const P2<T> d = pair_id<M>(g, A, R, o, u, row, z);
  return P2<T>{v.a * d.a, v.b * d.b};
}
// the cell beside a pair (offset k from xa) in the own row, x even on its left, odd on its right: never
// x = 1 or N0 − 2 (a ghost holds 0)
template <int M, class T>
__device__ __forceinline__ T eps_side(const Geo& g, const LeanL<T>& A, T v, int64_t R, uint32_t o, int k, const PairU<T>& u, int z) {
  if constexpr (M == LEAN_MEM) return v * ldo(A.iD + R + k, o);
  else return v * A.im[u.yw[0]][(M == LEAN_WALL && at_zwall(g, z)) ? 1 : 0];
}
// f with the plane's form
template <class F>
__device__ __forceinline__ void lean_mode(const Geo& g, bool fast, int z, F&& f) {
  if (!fast) f(ModeC<LEAN_MEM>{});
  else if (z <= 2 || z >= g.N[2] - 3) f(ModeC<LEAN_WALL>{});
  else f(ModeC<LEAN_MID>{});
}

// ---- Jacobi! + restrict! (src/MultiLevelPoisson.jl:92-94,13-19) from r₀ alone ----
// Lanes as in k_inc_restrict2: lane l of a wave's halves owns the x children of coarse cell l & 31 in
// fine rows 2Q−1 (lanes 0..31) and 2Q (32..63), so each half is the other's inner y neighbour.  CE:
// also the coarse x = 0 and ϵ = r·iD (a coarse level run by the plain passes).
template <class T, bool CE>
__global__ void __launch_bounds__(256) k_lean_restrict(Geo gf, Geo gc, ZT t, LeanL<T> A, const T* __restrict__ r,
                                                       LRows<T> Lc, T* __restrict__ rc, T* __restrict__ xc,
                                                       T* __restrict__ ec, Gate gate) {
  if (gate.closed()) return;
  int cx, cy, z0, z1;
  zt_cell_id(t, lean_tile(t), cx, cy, z0, z1);  // the tile is 32 coarse cells wide
  const int lane = threadIdx.x, half = lane >> 5;
  cx = cx - lane + (lane & 31);
  if (cy > t.b.hi[1]) return;  // a whole wave (one coarse row)
  const bool vx = cx <= t.b.hi[0];
  const int q = vx ? cx : t.b.hi[0];
  const int xa = 2 * q - 1;
  const bool lead = vx && half == 0;
  const int64_t s1 = gf.s[1], s2 = gf.s[2];
  const int cyu = __builtin_amdgcn_readfirstlane(cy);
  const int f0 = 2 * z0 - 1, f1 = 2 * z1;
  // both rows' flags, lane j holding plane f0 + j (a tile has at most 64 fine planes)
  const int seg = __builtin_amdgcn_readfirstlane((2 * (cx - (lane & 31)) - 1) / (2 * SEG_PAIRS));
  const uint32_t fl = lean_flags(gf, A, seg, 2 * cyu - 1, f0, f1 - f0 + 1, lane) & lean_flags(gf, A, seg, 2 * cyu, f0, f1 - f0 + 1, lane);
  const uint32_t flc = (lane < z1 - z0 + 1 && row_uniform(gc, Lc, cyu, z0 + lane)) ? 1u : 0u;
  const PairU<T> u = pair_u(gf, A, xa, 2 * cyu - 1 + half);
  // lane offsets of the own row and of the outer y neighbour, from the row below the pair of rows
  uint32_t o = (uint32_t)((xa + (half ? 2 : 1) * s1) * (int64_t)sizeof(T));
  uint32_t oo = (uint32_t)((xa + (half ? 3 : 0) * s1) * (int64_t)sizeof(T));
  int64_t R = s1 * (2 * cyu - 2) + s2 * f0;  // that row in the current plane
  P2<T> vm = ldo2(r + R - s2, o), v0 = ldo2(r + R, o), vp = ldo2(r + R + s2, o), ov = ldo2(r + R, oo);
  T lv = ldo(r + R - 1, o), rv = ldo(r + R + 2, o);
  T s = 0;
  auto step = [&](int fz) {
    WL_KEEP_OFFSET(o);
    WL_KEEP_OFFSET(oo);
    const T* pn = r + R + (fz < f1 ? s2 : 0);
    const P2<T> vn = ldo2(pn + (fz < f1 ? s2 : 0), o), on = ldo2(pn, oo);
    const T ln = ldo(pn - 1, o), rn = ldo(pn + 2, o);
    T ra, rb;
    lean_mode(gf, __builtin_amdgcn_readlane(fl, fz - f0) != 0u, fz, [&](auto mc) {
      constexpr int M = decltype(mc)::value;
      const P2<T> e0 = eps_j<M>(gf, A, v0, R, o, u, 0, fz), em = eps_j<M>(gf, A, vm, R - s2, o, u, 0, fz - 1);
      const P2<T> ep = eps_j<M>(gf, A, vp, R + s2, o, u, 0, fz + 1);
      P2<T> od;
      if constexpr (M == LEAN_MEM) {
        od = ldo2(A.iD + R, oo);
      } else {
        const P2<T> d1 = pair_id<M>(gf, A, R, oo, u, 1, fz), d2 = pair_id<M>(gf, A, R, oo, u, 2, fz);
        od = P2<T>{half ? d2.a : d1.a, half ? d2.b : d1.b};
      }
      const P2<T> eo{ov.a * od.a, ov.b * od.b};
      const T ja = __shfl_xor(e0.a, 32, 64), jb = __shfl_xor(e0.b, 32, 64);  // the wave's other row
      const P2<T> ym{half ? ja : eo.a, half ? jb : eo.b}, yp{half ? eo.a : ja, half ? eo.b : jb};
      const T xl = eps_side<M>(gf, A, lv, R, o, -1, u, fz), xr = eps_side<M>(gf, A, rv, R, o, 2, u, fz);
      const PairLD<T> c = pair_ld<M>(gf, A, R, o, u, fz);
      ra = v0.a - T(1) * c.ma(xl, e0, ym, yp, em, ep);
      rb = v0.b - T(1) * c.mb(xr, e0, ym, yp, em, ep);
    });
    // children summed in z, y, x order
    const T a1 = __shfl_down(ra, 32, 64), b1 = __shfl_down(rb, 32, 64);
    s += ra;
    s += rb;
    s += a1;
    s += b1;
    vm = v0;
    v0 = vp;
    vp = vn;
    ov = on;
    lv = ln;
    rv = rn;
    R += s2;
  };
#pragma unroll 1
  for (int kc = z0; kc <= z1; ++kc) {
    s = 0;
    step(2 * kc - 1);
    step(2 * kc);
    if (lead) {
      const int64_t Ic = at(gc, cx, cyu, kc);
      rc[Ic] = s;
      if (CE) {
        const bool uc = __builtin_amdgcn_readlane(flc, kc - z0) != 0u;
        xc[Ic] = 0;
        ec[Ic] = s * inv_diag(diag_at<T>(gc, lcell_row(gc, Lc, cx, cyu, kc, uc), Ic));
      }
    }
  }
}

// The coarse x (CINC: x + ω·ϵ, its last increment!, ϵ colour-split with SPLITC) of cells qx + k in a
// coarse row; 0 on ghosts
template <class T, bool CINC, bool SPLITC>
struct CoarseX {
  const T* xc;
  const T* ec;
  SplitG sg;
  int64_t c1, c2;
  int N1;
  T w;
  uint32_t o;   // the lane's byte offset of qx
  uint32_t qx;
  __device__ __forceinline__ T at(int k, int qy, int qz) const {
    const int64_t R = c1 * qy + c2 * qz;
    T v = ldo(xc + R + k, o);
    if (CINC) {
      if constexpr (SPLITC) {
        const int64_t S = (int64_t)sg.Q * (qy + (int64_t)N1 * qz);
        const uint32_t q = qx + (uint32_t)k;
        const T* e0 = ec + S;
        const T* e1 = e0 + sg.H;
        const uint32_t b = ((q + 1) >> 1) * (uint32_t)sizeof(T);
        // the two colours alternate along the row
        const uint32_t odd = (q + (uint32_t)(qy + qz)) & 1u;
        v = v + w * (odd ? ldo(e1, b) : ldo(e0, b));
      } else {
        v = v + w * ldo(ec + R + k, o);
      }
    }
    return v;
  }
};

// ---- prolongate! + increment!(ω) after Jacobi! (src/MultiLevelPoisson.jl:92,98-100) from r₀ ----
// r₂ = (r₀ − Aϵ_J) − ω·Ae_c; XW: also x = ϵ_J + ω·e_c (a coarser level, whose x was 0).
// A coarse cell covers two fine rows and planes, so of a cell's y and z neighbours one lies under the
// same coarse cell: a lane reads the next coarse plane's values (own, beside in x and y) once per
// two planes.
template <class T, bool CINC, bool SPLITC, bool XW>
__global__ void __launch_bounds__(256) k_lean_prolong(Geo g, Geo gc, ZT t, LeanL<T> A, const T* __restrict__ r,
                                                      T* __restrict__ r2, T* __restrict__ x,
                                                      const T* __restrict__ xc, const T* __restrict__ ec,
                                                      SplitG sgc, const T* __restrict__ wp) {
  const T w = *wp;
  const PairCell c = lean_cell(t);
  if (c.y > t.b.hi[1]) return;
  const int lane = threadIdx.x, y = c.y;
  const int64_t s1 = g.s[1], s2 = g.s[2];
  const bool yodd = y & 1;
  const uint32_t fl = lean_flags(g, A, __builtin_amdgcn_readfirstlane(c.p) / SEG_PAIRS, y, c.z0, c.z1 - c.z0 + 1, lane);
  const PairU<T> u = pair_u(g, A, c.xa, y);
  const int qx = (c.xa + 1) >> 1, qy = (y + 1) >> 1, qn = yodd ? qy - 1 : qy + 1;
  CoarseX<T, CINC, SPLITC> X{xc, ec, sgc, gc.s[1], gc.s[2], gc.N[1], w, (uint32_t)(qx * (int)sizeof(T)), (uint32_t)qx};
  uint32_t o = (uint32_t)(c.xa * (int)sizeof(T));
  int64_t R = s1 * y + s2 * c.z0;
  P2<T> vm = ldo2(r + R - s2, o), v0 = ldo2(r + R, o), vp = ldo2(r + R + s2, o);
  P2<T> ymv = ldo2(r + R - s1, o), ypv = ldo2(r + R + s1, o);
  T lv = ldo(r + R - 1, o), rv = ldo(r + R + 2, o);
  int qz = (c.z0 + 1) >> 1;  // z0 is odd: the first plane of a coarse cell
  T Cm = X.at(0, qy, qz - 1), C0 = X.at(0, qy, qz), Cp = T(0);
  T Cy = X.at(0, qn, qz), Cl = X.at(-1, qy, qz), Cr = X.at(1, qy, qz);
  auto step = [&](int z, auto oc) {
    constexpr bool odd = decltype(oc)::value;
    WL_KEEP_OFFSET(o);
    const T* pn = r + R + (z < c.z1 ? s2 : 0);
    const P2<T> vn = ldo2(pn + (z < c.z1 ? s2 : 0), o), ymn = ldo2(pn - s1, o), ypn = ldo2(pn + s1, o);
    const T ln = ldo(pn - 1, o), rn = ldo(pn + 2, o);
    T Cyn = T(0), Cln = T(0), Crn = T(0);
    if constexpr (odd) {
      Cp = X.at(0, qy, qz + 1);  // needed from the coarse cell's second plane on
    } else {
      const int qa = z < c.z1 ? qz + 1 : qz;
      Cyn = X.at(0, qn, qa);
      Cln = X.at(-1, qy, qa);
      Crn = X.at(1, qy, qa);
    }
    const T cym = yodd ? Cy : C0, cyp = yodd ? C0 : Cy;
    lean_mode(g, __builtin_amdgcn_readlane(fl, z - c.z0) != 0u, z, [&](auto mc) {
      constexpr int M = decltype(mc)::value;
      const P2<T> e0 = eps_j<M>(g, A, v0, R, o, u, 0, z), em = eps_j<M>(g, A, vm, R - s2, o, u, 0, z - 1);
      const P2<T> ep = eps_j<M>(g, A, vp, R + s2, o, u, 0, z + 1);
      const P2<T> ym = eps_j<M>(g, A, ymv, R - s1, o, u, 1, z), yp = eps_j<M>(g, A, ypv, R + s1, o, u, 2, z);
      const T xl = eps_side<M>(g, A, lv, R, o, -1, u, z), xr = eps_side<M>(g, A, rv, R, o, 2, u, z);
      const PairLD<T> k = pair_ld<M>(g, A, R, o, u, z);
      T ra = v0.a - T(1) * k.ma(xl, e0, ym, yp, em, ep);
      T rb = v0.b - T(1) * k.mb(xr, e0, ym, yp, em, ep);
      const T czm = odd ? Cm : C0, czp = odd ? C0 : Cp;
      const P2<T> q{C0, C0}, qm{cym, cym}, qp{cyp, cyp}, zm{czm, czm}, zp{czp, czp};
      ra = ra - w * k.ma(Cl, q, qm, qp, zm, zp);
      rb = rb - w * k.mb(Cr, q, qm, qp, zm, zp);
      if (c.vx) {
        sto2(r2 + R, o, ra, rb);
        if (XW) sto2(x + R, o, (T(0) + T(1) * e0.a) + w * C0, (T(0) + T(1) * e0.b) + w * C0);
      }
    });
    vm = v0;
    v0 = vp;
    vp = vn;
    ymv = ymn;
    ypv = ypn;
    lv = ln;
    rv = rn;
    R += s2;
    if constexpr (!odd) {  // the next plane lies in the next coarse one
      ++qz;
      Cm = C0;
      C0 = Cp;
      Cy = Cyn;
      Cl = Cln;
      Cr = Crn;
    }
  };
#pragma unroll 1
  for (int z = c.z0; z < c.z1; z += 2) {
    WL_KEEP_OFFSET(X.o);
    WL_KEEP_OFFSET(X.qx);
    step(z, FlagC<true>{});
    step(z + 1, FlagC<false>{});
  }
}

// ---- the first GS-RB half sweep (src/Poisson.jl:141-148) from r₂ ----
// ϵ = r₂·iD of the colour it reads is formed from r₂; the colour it updates is stored colour-split for
// k_lean_gs, which then needs no initial ϵ: sweep 2 overwrites the other colour unread.
template <class T>
__global__ void __launch_bounds__(256) k_lean_gs_first(Geo g, SplitG sg, ZT t, LeanL<T> A, const T* __restrict__ r2,
                                                       T* __restrict__ e) {
  constexpr int K = 1;  // the colour of sweep 1 in 3D: (it + D + 1) mod 2
  const PairCell c = lean_cell(t);
  if (c.y > t.b.hi[1]) return;
  const int lane = threadIdx.x, y = c.y;
  const int64_t s1 = g.s[1], s2 = g.s[2], t2 = (int64_t)sg.Q * g.N[1];
  const uint32_t fl = lean_flags(g, A, __builtin_amdgcn_readfirstlane(c.p) / SEG_PAIRS, y, c.z0, c.z1 - c.z0 + 1, lane);
  const PairU<T> u = pair_u(g, A, c.xa, y);
  uint32_t o = (uint32_t)(c.xa * (int)sizeof(T)), oj = (uint32_t)(((c.xa + 1) >> 1) * (int)sizeof(T));
  int64_t R = s1 * y + s2 * c.z0;
  T* E = e + (K ? sg.H : 0) + (int64_t)sg.Q * y + t2 * c.z0;
  P2<T> vm = ldo2(r2 + R - s2, o), v0 = ldo2(r2 + R, o), vp = ldo2(r2 + R + s2, o);
  auto run = [&](auto hc) {  // H0: the updated cell of the pair in the tile's first plane
    constexpr int H0 = decltype(hc)::value ? 1 : 0;
    T ymv = ldo(r2 + R - s1 + H0, o), ypv = ldo(r2 + R + s1 + H0, o), sv = ldo(r2 + R + (H0 ? 2 : -1), o);
    auto step = [&](int z, auto hh) {
      constexpr int h = decltype(hh)::value ? 1 : 0;
      WL_KEEP_OFFSET(o);
      WL_KEEP_OFFSET(oj);
      // the planes ahead (the other cell of the pair is updated in the next one)
      const T* pn = r2 + R + (z < c.z1 ? s2 : 0);
      const P2<T> vn = ldo2(pn + (z < c.z1 ? s2 : 0), o);
      const T ymn = ldo(pn - s1 + (1 - h), o), ypn = ldo(pn + s1 + (1 - h), o), sn = ldo(pn + (h ? -1 : 2), o);
      T nv;
      lean_mode(g, __builtin_amdgcn_readlane(fl, z - c.z0) != 0u, z, [&](auto mc) {
        constexpr int M = decltype(mc)::value;
        const P2<T> d = pair_id<M>(g, A, R, o, u, 0, z);
        const T xs = eps_side<M>(g, A, sv, R, o, h ? 2 : -1, u, z);
        const T own = h ? d.b : d.a;
        const T xi = h ? v0.a * d.a : v0.b * d.b;
        auto nb = [&](T v, int64_t S, int row, int zz) -> T {
          const P2<T> e = pair_id<M>(g, A, S, o, u, row, zz);
          return v * (h ? e.b : e.a);
        };
        const T ym = nb(ymv, R - s1, 1, z), yp = nb(ypv, R + s1, 2, z);
        const T zm = nb(h ? vm.b : vm.a, R - s2, 0, z - 1), zp = nb(h ? vp.b : vp.a, R + s2, 0, z + 1);
        const PairLD<T> k = pair_ld<M>(g, A, R, o, u, z);
        T s = h ? v0.b : v0.a;
        s -= ((h ? xi : xs) * (h ? k.xm : k.xa) + (h ? xs : xi) * (h ? k.xb : k.xm));
        s -= (ym * (h ? k.yb : k.ya) + yp * (h ? k.Yb : k.Ya));
        s -= (zm * (h ? k.zb : k.za) + zp * (h ? k.Zb : k.Za));
        nv = s * own;
      });
      if (c.vx) *(T*)((char*)E + oj) = nv;
      vm = v0;
      v0 = vp;
      vp = vn;
      ymv = ymn;
      ypv = ypn;
      sv = sn;
      R += s2;
      E += t2;
    };
#pragma unroll 1
    for (int z = c.z0; z < c.z1; z += 2) {
      step(z, FlagC<H0 == 1>{});
      step(z + 1, FlagC<H0 == 0>{});
    }
  };
  if (((1 + y + c.z0) & 1) == K) run(FlagC<false>{}); else run(FlagC<true>{});
}

// ---- the other half sweeps: k_gs_half_s with the constants and the loads ahead ----
template <class T>
__global__ void __launch_bounds__(256) k_lean_gs(Geo g, SplitG sg, ZT t, LeanL<T> A, const T* __restrict__ r2,
                                                 T* __restrict__ e, int it) {
  const PairCell c = lean_cell(t);
  if (c.y > t.b.hi[1]) return;
  const int lane = threadIdx.x, y = c.y;
  const int K = it & 1;  // the colour this sweep updates: (it + D + 1) mod 2
  const int64_t s1 = g.s[1], s2 = g.s[2], t1 = sg.Q, t2 = (int64_t)sg.Q * g.N[1];
  const uint32_t fl = lean_flags(g, A, __builtin_amdgcn_readfirstlane(c.p) / SEG_PAIRS, y, c.z0, c.z1 - c.z0 + 1, lane);
  const PairU<T> u = pair_u(g, A, c.xa, y);
  uint32_t o = (uint32_t)(c.xa * (int)sizeof(T)), oj = (uint32_t)(((c.xa + 1) >> 1) * (int)sizeof(T));
  int64_t R = s1 * y + s2 * c.z0;
  const int64_t S = t1 * y + t2 * c.z0;
  const T* __restrict__ O = e + (K ? 0 : sg.H) + S;  // ϵ of the other colour (read only)
  T* __restrict__ E = e + (K ? sg.H : 0) + S;        // ϵ of this colour (written only)
  T om = ldo(O - t2, oj), o0 = ldo(O, oj), op = ldo(O + t2, oj), ym = ldo(O - t1, oj), yp = ldo(O + t1, oj);
  auto run = [&](auto hc) {  // H0: the updated cell of the pair in the tile's first plane
    constexpr int H0 = decltype(hc)::value ? 1 : 0;
    T xo = ldo(O + (H0 ? 1 : -1), oj), rr = ldo(r2 + R + H0, o);
    auto step = [&](int z, auto hh) {
      constexpr int h = decltype(hh)::value ? 1 : 0;
      WL_KEEP_OFFSET(o);
      WL_KEEP_OFFSET(oj);
      const int64_t d = z < c.z1 ? t2 : 0;
      const T* On = O + d;
      const T on = ldo(On + d, oj), rn = ldo(r2 + R + (z < c.z1 ? s2 : 0) + (1 - h), o);
      const T ymn = ldo(On - t1, oj), ypn = ldo(On + t1, oj), xn = ldo(On + (h ? -1 : 1), oj);
      T nv;
      lean_mode(g, __builtin_amdgcn_readlane(fl, z - c.z0) != 0u, z, [&](auto mc) {
        constexpr int M = decltype(mc)::value;
        const PairLD<T> k = pair_ld<M>(g, A, R, o, u, z);
        T s = rr;
        s -= ((h ? o0 : xo) * (h ? k.xm : k.xa) + (h ? xo : o0) * (h ? k.xb : k.xm));
        s -= (ym * (h ? k.yb : k.ya) + yp * (h ? k.Yb : k.Ya));
        s -= (om * (h ? k.zb : k.za) + op * (h ? k.Zb : k.Za));
        if constexpr (M == LEAN_MEM) {
          nv = s * ldo(A.iD + R + h, o);
        } else {
          const P2<T> d = pair_id<M>(g, A, R, o, u, 0, z);
          nv = s * (h ? d.b : d.a);
        }
      });
      if (c.vx) *(T*)((char*)E + oj) = nv;
      om = o0;
      o0 = op;
      op = on;
      ym = ymn;
      yp = ypn;
      xo = xn;
      rr = rn;
      R += s2;
      O += t2;
      E += t2;
    };
#pragma unroll 1
    for (int z = c.z0; z < c.z1; z += 2) {
      step(z, FlagC<H0 == 1>{});
      step(z + 1, FlagC<H0 == 0>{});
    }
  };
  if (((1 + y + c.z0) & 1) == K) run(FlagC<false>{}); else run(FlagC<true>{});
}

// ---- smooth!'s increment! of the finest level with the Jacobi! and prolongation increments of x ----
// x = ((xin·scale + ϵ_J) + ω·e_c) + ω·ϵ (xin: the level's x, or in a projection's first V-cycle p,
// with scale = dt), r = r₂ − ω·Aϵ over r₀ (read by its own lane before), and the block's Σr².
template <class T, bool CINC, bool SPLITC>
__global__ void __launch_bounds__(256) k_lean_increment(Geo g, Geo gc, ZT t, LeanL<T> A, T* r,
                                                        const T* __restrict__ r2, const T* xin, T scale,
                                                        T* x, const T* __restrict__ e, SplitG sg,
                                                        const T* __restrict__ xc, const T* __restrict__ ec,
                                                        SplitG sgc, const T* __restrict__ wp,
                                                        double* __restrict__ partial) {
  const T w = *wp;
  const PairCell c = lean_cell(t);
  double acc = 0;
  if (c.y <= t.b.hi[1]) {
    const int lane = threadIdx.x, y = c.y;
    const int64_t s1 = g.s[1], s2 = g.s[2], t1 = sg.Q, t2 = (int64_t)sg.Q * g.N[1];
    const uint32_t fl = lean_flags(g, A, __builtin_amdgcn_readfirstlane(c.p) / SEG_PAIRS, y, c.z0, c.z1 - c.z0 + 1, lane);
    const PairU<T> u = pair_u(g, A, c.xa, y);
    const int qx = (c.xa + 1) >> 1, qy = (y + 1) >> 1;
    CoarseX<T, CINC, SPLITC> X{xc, ec, sgc, gc.s[1], gc.s[2], gc.N[1], w, (uint32_t)(qx * (int)sizeof(T)), (uint32_t)qx};
    uint32_t o = (uint32_t)(c.xa * (int)sizeof(T)), oj = (uint32_t)(qx * (int)sizeof(T));
    int64_t R = s1 * y + s2 * c.z0, S = t1 * y + t2 * c.z0;
    auto run = [&](auto pc) {  // P0: (y + z) mod 2 in the tile's first plane
      constexpr int P0 = decltype(pc)::value ? 1 : 0;
      // the pair's ϵ in a row of parity par: xa (odd) has colour 1 − par
      const T* const e0s = e;
      const T* const e1s = e + sg.H;
      auto ldE = [&](int64_t q, int par) -> P2<T> {
        return P2<T>{ldo((par ? e0s : e1s) + q, oj), ldo((par ? e1s : e0s) + q, oj)};
      };
      auto left = [&](int64_t q, int par) -> T { return ldo((par ? e1s : e0s) + q - 1, oj); };
      auto right = [&](int64_t q, int par) -> T { return ldo((par ? e0s : e1s) + q + 1, oj); };
      P2<T> em = ldE(S - t2, 1 - P0), e0 = ldE(S, P0), ep = ldE(S + t2, 1 - P0);
      P2<T> ym = ldE(S - t1, 1 - P0), yp = ldE(S + t1, 1 - P0);
      T xl = left(S, P0), xr = right(S, P0);
      P2<T> rr = ldo2(r2 + R, o), r0 = ldo2((const T*)r + R, o), xx = ldo2(xin + R, o);
      int qz = (c.z0 + 1) >> 1;  // z0 is odd: the first plane of a coarse cell
      T C0 = X.at(0, qy, qz), Cn = T(0);
      auto step = [&](int z, auto pp, auto oc) {
        constexpr int par = decltype(pp)::value ? 1 : 0;
        constexpr bool odd = decltype(oc)::value;
        WL_KEEP_OFFSET(o);
        WL_KEEP_OFFSET(oj);
        const bool more = z < c.z1;
        const int64_t Rn = R + (more ? s2 : 0), Sn = S + (more ? t2 : 0);
        const P2<T> en = ldE(Sn + (more ? t2 : 0), par), rrn = ldo2(r2 + Rn, o), r0n = ldo2((const T*)r + Rn, o);
        const P2<T> xxn = ldo2(xin + Rn, o), ymn = ldE(Sn - t1, par), ypn = ldE(Sn + t1, par);
        const T xln = left(Sn, 1 - par), xrn = right(Sn, 1 - par);
        if constexpr (!odd) Cn = X.at(0, qy, more ? qz + 1 : qz);
        T ra, rb;
        P2<T> d;
        lean_mode(g, __builtin_amdgcn_readlane(fl, z - c.z0) != 0u, z, [&](auto mc) {
          constexpr int M = decltype(mc)::value;
          const PairLD<T> k = pair_ld<M>(g, A, R, o, u, z);
          d = pair_id<M>(g, A, R, o, u, 0, z);
          ra = rr.a - w * k.ma(xl, e0, ym, yp, em, ep);
          rb = rr.b - w * k.mb(xr, e0, ym, yp, em, ep);
        });
        const T xa = ((xx.a * scale + T(1) * (r0.a * d.a)) + w * C0) + w * e0.a;
        const T xb = ((xx.b * scale + T(1) * (r0.b * d.b)) + w * C0) + w * e0.b;
        if (c.vx) {
          sto2(r + R, o, ra, rb);
          sto2(x + R, o, xa, xb);
          acc += (double)ra * (double)ra;
          acc += (double)rb * (double)rb;
        }
        em = e0;
        e0 = ep;
        ep = en;
        ym = ymn;
        yp = ypn;
        xl = xln;
        xr = xrn;
        rr = rrn;
        r0 = r0n;
        xx = xxn;
        R += s2;
        S += t2;
        if constexpr (!odd) {
          C0 = Cn;
          ++qz;
        }
      };
#pragma unroll 1
      for (int z = c.z0; z < c.z1; z += 2) {
        WL_KEEP_OFFSET(X.o);
        WL_KEEP_OFFSET(X.qx);
        step(z, FlagC<P0 == 1>{}, FlagC<true>{});
        step(z + 1, FlagC<P0 == 0>{}, FlagC<false>{});
      }
    };
    if ((y + c.z0) & 1) run(FlagC<true>{}); else run(FlagC<false>{});
  }
  const double tt = block_sum(acc);
  if (threadIdx.x == 0 && threadIdx.y == 0) partial[blockIdx.x] = tt;
}

}  // namespace wl
