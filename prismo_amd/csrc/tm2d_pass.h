// Several textbook Yee steps of a 2-D TM grid (Ez, Hx, Hy) per launch: a
// workgroup holds a tile of the grid in registers, steps it `ns` times and
// writes the part of it that its halo still covers.
//
// One step per launch moves every field through the caches once per step and
// pays a launch and a chain of row loads each time: a 540 x 290 FP64 grid took
// 11.6 us a step with its sources and samples, of which its 157 k cells need
// well under 1; a 2000 x 1500 FP32 one 26.6 us.  A pass of 8 steps reads the
// state once, with a halo of 8 cells, and writes it once: 2.0 us and 4.9 us a
// step.  What is left is latency (a pass of the small grid waits for its loads,
// 16 barriers and the source table) and, on large grids, the vector ALU:
// 13 instructions a cell and step, halo cells included, 20 in a CPML layer.
//
// Tile: 8 waves stacked in y, each 64 columns (one per lane) by R rows in
// registers; 8 cells on each side are halo (a step's E depends on fields one
// cell away in every direction), so 48 columns and 8 R - 16 rows are written.
// x neighbours come from the neighbouring lanes (DPP), y neighbours from the
// lane's own registers, and one row per wave boundary through LDS.  8 waves of
// few rows, not 4 of many: a step is one long dependent chain per wave, and the
// second wave on a SIMD fills its gaps (540 x 290, 8 steps: 4 waves of 8 rows
// 20 us, 8 of 4 16.6).  8 steps, not 4: the loads, stores and the launch cost a
// pass of the small grid as much as 6 steps (11.7 us for 4 steps, 16.6 for 8);
// on the large grid 28.5 us for 4 steps and 40 for 8.
//
// Sources are added after every step, samples taken after the sources.  Halo
// cells get their sources too (they are recomputed from the same inputs by the
// tile that owns them).  CPML memory of both field halves is read from one set
// and written to another, as the fields are.
//
// The arithmetic of a cell does not depend on where in a tile it lies: nothing
// is contracted but the multiply-adds written here.
#pragma once
#include "pm_internal.h"

namespace pm {

constexpr int kTmS = 8;                 // steps per pass (halo width)
constexpr int kTmW = 8;                 // waves per workgroup
// columns and rows a tile with a halo of S cells writes
__host__ __device__ constexpr int tm_cols(int S) { return 64 - 2 * S; }
__host__ __device__ constexpr int tm_rows(int R, int S = kTmS) { return kTmW * R - 2 * S; }
constexpr int kTmCols = tm_cols(kTmS);

template <int CTRL>
__device__ __forceinline__ int tm_dpp32(int fill, int v) {
  return __builtin_amdgcn_update_dpp(fill, v, CTRL, 0xf, 0xf, true);
}
// The neighbouring lane's value: wave_shr:1 (0x138) from the lane below,
// wave_shl:1 (0x130) from the lane above; 0 at the wave's end (bound control, so
// the move folds into the subtraction that uses it).
template <int CTRL, typename T>
__device__ __forceinline__ T tm_lane(T v) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, tm_dpp32<CTRL>(0, __builtin_bit_cast(int, v)));
  } else {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)tm_dpp32<CTRL>(0, (int)(unsigned)u);
    const unsigned hi = (unsigned)tm_dpp32<CTRL>(0, (int)(unsigned)(u >> 32));
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  }
}

__device__ __forceinline__ float tm_fma(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double tm_fma(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

// Lane l's value (l a constant), for every lane.
template <typename T>
__device__ __forceinline__ T tm_bcast(T v, int l) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
  } else {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  }
}

// f[r] of rows j0 .. j1 - 1 (the wave's first row: jb) to x[(row - j0) stride], for
// lanes with `in`.  A wave whose rows are all wanted, the usual case of a line
// along y, or none, makes no test per row: with one, the tiles that sample took
// twice as long as the others.
template <typename T, int R>
__device__ __forceinline__ void tm_put(gptr<T> x, int stride, bool in, int j0, int j1, int jb,
                                       const T (&f)[R]) {
  const int a = j0 - jb, b = j1 - jb;  // uniform
  if (a >= R || b <= 0) return;
  x -= (int64_t)a * stride;
  if (a <= 0 && b >= R) {
    if (in) {
#pragma unroll
      for (int r = 0; r < R; ++r) x[r * stride] = f[r];
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r >= a && r < b && in) x[r * stride] = f[r];
}

// f[r] += v[r] on rows j0 .. j1 - 1, for lanes with `in`.
template <typename T, int R, class V>
__device__ __forceinline__ void tm_add(const V& v, bool in, int j0, int j1, int jb, T (&f)[R]) {
  const int a = j0 - jb, b = j1 - jb;
  if (a <= 0 && b >= R) {
#pragma unroll
    for (int r = 0; r < R; ++r) f[r] = in ? f[r] + v(r) : f[r];
    return;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) f[r] = in && r >= a && r < b ? f[r] + v(r) : f[r];
}

// One grid as a pass sees it (uniform): offsets are 32-bit elements.
struct TmGrid {
  int nx, ny;
  uint32_t sy;
  int px0, px1, py0, py1;          // CPML layers
  const void *ez, *hx, *hy;        // read
  void *ez_o, *hx_o, *hy_o;        // written
  const void *ca, *cb;
  // CPML memory [H of x, H of y, E of x, E of y]: Hy, Hx, Ez, Ez terms.  x
  // layers: slab index (or column) + xst * row; y layers: column + yst * slab
  // index (or row)
  const void* ps[4];
  void* ps_o[4];
  uint32_t xst, yst;
  bool full;                       // CPML memory arrays span the grid
  double idx, idy, db, cb_scale;
};

// Per-lane x profiles (outside the layers be = ce = bh = ch = 0, ike = ikh = 1).
template <typename T>
struct TmXProf {
  T be, ce, ike, bh, ch, ikh;
};

template <typename T, int R>
struct TmShared {
  // Ez of each wave's last row (behind a row of zeros), Hx of each wave's first
  // row (before one)
  T e[kTmW + 1][64], h[kTmW + 1][64];
  // y profiles of the rows, E (be ce ike -) and H (bh ch ikh -): 16-byte reads
  alignas(16) T y[kTmW * R][2][4];
};

// ns (at most S) steps of the tile (x0, y0: first column and row it writes) by
// this wave.
// yp(k, j): y profile k (be ce ike bh ch ikh) at row j, for one j per lane.
// io.first() and io.second() issue their own loads before and behind the fields';
// io.sources(s, ...), io.samples(s, ...) act on the registers after step s.  With
// IO::kStatus, returns bit 31 set when an Ez value this lane wrote is Inf or NaN
// (a value that was stays so: it is looked at after the last step).  With
// IO::kPackedE, where g.full, the E set that is read or the one that is written
// holds the layers alone (io.packed(false), io.packed(true)).
template <typename T, int CK, int R, int S, bool XP, bool YP, class YProf, class IO>
__device__ __forceinline__ uint32_t tm_pass(const TmGrid& g, const TmXProf<T>& xp, bool xpml,
                                            const YProf& yp, IO& io, int ns, int x0, int y0,
                                            int w, TmShared<T, R>& sh) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int nx = g.nx, ny = g.ny;
  const int i = x0 - S + lane;        // this lane's column
  const int jb = y0 - S + w * R;      // this wave's first row
  // (without XP every column of the tile is inside the grid, without YP every row)
  const bool lin = !XP || (i >= 0 && i < nx);        // the column exists
  const bool le_ok = !XP || (i >= 0 && i < nx - 1);  // and holds Ez
  const int ic = XP ? min(max(i, 0), nx - 1) : i;
  const T idx = (T)g.idx, idy = (T)g.idy, db = (T)g.db;

  T ez[R], hx[R], hy[R], cb[R], ca[CK == PM_COEFF_CACB ? R : 1];
  T qhx[XP ? R : 1], qex[XP ? R : 1];  // x layers: Hy and Ez terms
  T qhy[YP ? R : 1], qey[YP ? R : 1];  // y layers: Hx and Ez terms
  // (lanes outside the layers read position 0 of a row)
  const uint32_t xslab = (uint32_t)(i < g.px0 ? i : g.px0 + (i - (nx - g.px1)));
  const uint32_t xo = !xpml ? 0u : g.full ? (uint32_t)ic : xslab;
  auto yrow = [&](int j) {  // y layers: row of the memory array
    if (g.full) return (uint32_t)j;
    return (uint32_t)(j < g.py0 ? j : g.py0 + (j - (ny - g.py1)));
  };
  // where IO::kPackedE: positions in the E set that is read (out false) or written
  auto xe = [&](bool out, uint32_t row) {
    return io.packed(out) ? xslab + (uint32_t)(g.px0 + g.px1) * row : xo + g.xst * row;
  };
  auto ye = [&](bool out, int j) {
    const int gap = io.packed(out) ? ny - g.py0 - g.py1 : 0;
    return (uint32_t)(j < g.py0 ? j : j - gap);
  };
  auto ypml = [&](int j) { return j >= 0 && j < ny && (j < g.py0 || j >= ny - g.py1); };
  io.first();
  // every load up front, from clamped positions (cells beyond the grid are 0)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = jb + r, jc = YP ? min(max(j, 0), ny - 1) : j;
    const bool ok = lin && (!YP || (j >= 0 && j < ny));
    const uint32_t o = (uint32_t)jc * g.sy + (uint32_t)ic;
    const T e = ((gptr<const T>)g.ez)[o], a = ((gptr<const T>)g.hx)[o],
            b = ((gptr<const T>)g.hy)[o];
    ez[r] = ok ? e : (T)0;
    hx[r] = ok && le_ok ? a : (T)0;
    hy[r] = ok && (!YP || j < ny - 1) ? b : (T)0;
    if constexpr (CK == PM_COEFF_CB_F16)
      cb[r] = (T)g.cb_scale * (T)((gptr<const _Float16>)g.cb)[o];
    else
      cb[r] = ((gptr<const T>)g.cb)[o];
    if constexpr (CK == PM_COEFF_CACB) ca[r] = ((gptr<const T>)g.ca)[o];
    // positions without Ez hold 0 and stay so
    if (!(ok && le_ok) || (YP && j >= ny - 1)) {
      ez[r] = cb[r] = (T)0;
      if constexpr (CK == PM_COEFF_CACB) ca[r] = (T)0;
    }
    if constexpr (XP) {
      const uint32_t q = xpml ? xo + g.xst * (uint32_t)jc : 0u;
      uint32_t qe = q;
      if constexpr (IO::kPackedE) qe = xpml ? xe(false, (uint32_t)jc) : 0u;
      const T h = ((gptr<const T>)g.ps[0])[q], f = ((gptr<const T>)g.ps[2])[qe];
      qhx[r] = ok && xpml ? h : (T)0;
      qex[r] = ok && xpml ? f : (T)0;
    }
    if constexpr (YP) {
      const bool in = ypml(j);
      const uint32_t q = in ? (uint32_t)ic + g.yst * yrow(j) : 0u;
      uint32_t qe = q;
      if constexpr (IO::kPackedE) qe = in ? (uint32_t)ic + g.yst * ye(false, j) : 0u;
      const T h = ((gptr<const T>)g.ps[1])[q], f = ((gptr<const T>)g.ps[3])[qe];
      qhy[r] = ok && in ? h : (T)0;
      qey[r] = ok && in ? f : (T)0;
    }
  }
  // y profiles of the wave's rows to LDS: read back there as broadcasts (scalar
  // loads in the row loop cost a tile in the y layers 10 us).  A wave reads only
  // what it wrote.
  if constexpr (YP) {
    if (lane < R) {
      const int j = jb + lane;
      const bool in = ypml(j);
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        sh.y[w * R + lane][k / 3][k % 3] = in ? yp(k, j) : (T)(k % 3 == 2 ? 1 : 0);
      }
    }
  }
  if (w == 0) sh.e[0][lane] = (T)0;
  if (w == kTmW - 1) sh.h[kTmW][lane] = (T)0;
  io.second(ns);
  uint32_t bad = 0;
  for (int s = 0; s < ns; ++s) {
    // the row number is made opaque per step: the tests of the sources and samples
    // on it are one scalar compare each, but hoisted out of the loop they would
    // hold a mask per row in SGPRs and spill
    int js = jb;
    asm volatile("" : "+s"(js));
    // H: backward differences of E
    sh.e[w + 1][lane] = ez[R - 1];
    __syncthreads();
    T below = sh.e[w][lane];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // (outside the layers the profiles leave a difference as it is, so every
      // variant of this code gives a cell the same bits)
      T d1 = (ez[r] - below) * idy;
      T d2 = (ez[r] - tm_lane<0x138>(ez[r])) * idx;
      if constexpr (YP) {
        const T* y = sh.y[w * R + r][1];
        qhy[r] = tm_fma(y[0], qhy[r], y[1] * d1);
        d1 = tm_fma(d1, y[2], qhy[r]);
      }
      if constexpr (XP) {
        qhx[r] = tm_fma(xp.bh, qhx[r], xp.ch * d2);
        d2 = tm_fma(d2, xp.ikh, qhx[r]);
      }
      hx[r] = tm_fma(-db, d1, hx[r]);
      hy[r] = tm_fma(db, d2, hy[r]);
      below = ez[r];
    }
    // E: forward differences of H
    sh.h[w][lane] = hx[0];
    __syncthreads();
    const T above = sh.h[w + 1][lane];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T e1 = (tm_lane<0x130>(hy[r]) - hy[r]) * idx;
      T e2 = ((r + 1 < R ? hx[r + 1 < R ? r + 1 : 0] : above) - hx[r]) * idy;
      if constexpr (XP) {
        qex[r] = tm_fma(xp.be, qex[r], xp.ce * e1);
        e1 = tm_fma(e1, xp.ike, qex[r]);
      }
      if constexpr (YP) {
        const T* y = sh.y[w * R + r][0];
        qey[r] = tm_fma(y[0], qey[r], y[1] * e2);
        e2 = tm_fma(e2, y[2], qey[r]);
      }
      const T c = e1 - e2;
      T v;
      if constexpr (CK == PM_COEFF_CACB)
        v = tm_fma(cb[r], c, ca[r] * ez[r]);
      else
        v = tm_fma(cb[r], c, ez[r]);
      ez[r] = v;
    }
    io.sources(s, i, js, ez, hx, hy);
    io.samples(s, i, js, ez, hx, hy);
  }
  const bool mine = lane >= S && lane < 64 - S && lin;
  if (!mine) return 0;
  if (S % R == 0 && (w * R < S || w * R >= kTmW * R - S)) return 0;  // all halo
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int t = w * R + r, j = jb + r;
    if (S % R != 0 && (t < S || t >= kTmW * R - S)) continue;  // uniform
    if (YP && j >= ny) continue;
    const uint32_t o = (uint32_t)j * g.sy + (uint32_t)i;
    // positions past a component's extent stay 0 in memory (next to an Inf or NaN
    // their zero coefficient does not keep them so)
    const bool ly_ok = !YP || j < ny - 1;
    const T e = le_ok && ly_ok ? ez[r] : (T)0;
    if constexpr (IO::kStatus) {
      if constexpr (sizeof(T) == 4)
        bad |= (__builtin_bit_cast(uint32_t, e) & 0x7f800000u) + 0x00800000u;
      else
        bad |= ((uint32_t)(__builtin_bit_cast(uint64_t, e) >> 32) & 0x7ff00000u) + 0x00100000u;
    }
    ((gptr<T>)g.ez_o)[o] = e;
    ((gptr<T>)g.hx_o)[o] = le_ok ? hx[r] : (T)0;
    ((gptr<T>)g.hy_o)[o] = ly_ok ? hy[r] : (T)0;
    if constexpr (XP) {
      if (xpml) {
        const uint32_t q = xo + g.xst * (uint32_t)j;
        uint32_t qe = q;
        if constexpr (IO::kPackedE) qe = xe(true, (uint32_t)j);
        ((gptr<T>)g.ps_o[0])[q] = qhx[r];
        ((gptr<T>)g.ps_o[2])[qe] = qex[r];
      }
    }
    if constexpr (YP) {
      if (ypml(j)) {
        const uint32_t q = (uint32_t)i + g.yst * yrow(j);
        uint32_t qe = q;
        if constexpr (IO::kPackedE) qe = (uint32_t)i + g.yst * ye(true, j);
        ((gptr<T>)g.ps_o[1])[q] = qhy[r];
        ((gptr<T>)g.ps_o[3])[qe] = qey[r];
      }
    }
  }
  return bad;
}

// The pass with the CPML and edge code the tile needs (uniform over the
// workgroup): XP for tiles that reach an x layer or the grid's first or last
// column, YP the same in y (an axis without layers then reads element 0 of
// some array, unused, and stores nothing).
template <typename T, int CK, int R, int S = kTmS, class YProf, class IO>
__device__ __forceinline__ uint32_t tm_tile(const TmGrid& g, const TmXProf<T>& xp, bool xpml,
                                            const YProf& yp, IO& io, int ns, int x0, int y0,
                                            int w, TmShared<T, R>& sh) {
  const bool hasx = x0 - S < g.px0 || x0 - S + 64 > g.nx - max(g.px1, 1);
  const bool hasy = y0 - S < g.py0 || y0 - S + kTmW * R > g.ny - max(g.py1, 1);
  if (hasx && hasy)
    return tm_pass<T, CK, R, S, true, true>(g, xp, xpml, yp, io, ns, x0, y0, w, sh);
  if (hasx) return tm_pass<T, CK, R, S, true, false>(g, xp, xpml, yp, io, ns, x0, y0, w, sh);
  if (hasy) return tm_pass<T, CK, R, S, false, true>(g, xp, xpml, yp, io, ns, x0, y0, w, sh);
  return tm_pass<T, CK, R, S, false, false>(g, xp, xpml, yp, io, ns, x0, y0, w, sh);
}

// Workgroup order: groups of 64 of which XCD x takes 8 neighbours, so tiles
// that share halo cells share an L2.
__device__ __forceinline__ int tm_order(int b, int n) {
  return b < (n & ~63) ? (b & ~63) + (b & 7) * 8 + ((b >> 3) & 7) : b;
}

// Rows per wave.  8 rows spend less on the halo (44 % of a tile, 4 rows 62 %),
// 4 rows make more workgroups: FP32 takes 8 once those fill every compute unit
// twice (400 steps of 1400 x 1000: 2.37 ms with 8, 2.56 with 4; 1000 x 800: 2.23
// and 2.11; 150 x 100: 2.21 and 1.78).  FP64 keeps 4: 8 rows take 227 registers,
// one workgroup per compute unit (2000 x 1500: 4.57 and 4.60, 1400 x 1000: 3.36
// and 3.09, 540 x 290: 1.99 and 1.70).
inline int tm_pick_rows(double cells, int esz, int n_cu) {
  return esz == 4 && cells >= 2.0 * n_cu * kTmCols * tm_rows(8) ? 8 : 4;
}

}  // namespace pm
