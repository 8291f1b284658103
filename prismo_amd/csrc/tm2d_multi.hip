// Several 2-D TM steps per launch of one simulation (tm2d_pass.h): its sources
// and monitor samples inside, so a run of steps is a launch per 8 steps.
#include "tm2d_pass.h"

namespace pm {
namespace {

template <typename T>
struct SimY {
  gptr<const T> p[6];
  __device__ __forceinline__ T operator()(int k, int j) const { return p[k][j]; }
};

struct SimProf {
  const void* x[6];  // be ce ike bh ch ikh
  const void* y[6];
};

// Source and sample tables of a launch: table row of the first step, sample
// row of the first step (a launch never crosses the end of the sample ring).
struct SimIoArgs {
  const KSrc* src;
  const KSbox* sbox;
  int n_src, n_sbox, ncols;
  int64_t row, xrow;
  const int64_t* clock;
  void* X;
};

// The tables are in device memory.  Lane t keeps source box t and lane
// kMaxSrc + t sample box t, lane l also the values of source l / 4 at steps
// l % 4, l % 4 + 4; all of it is loaded beside the fields, and a box is read back with
// lane broadcasts.  (Read where they are used, a tile with a source waited for
// its table entry, its box and its value one after the other in every step.)
// Boxes that do not meet the tile are masked out; most tiles have none.
template <typename T>
struct SimIo {
  static constexpr bool kStatus = false, kPackedE = false;
  __device__ __forceinline__ static constexpr bool packed(bool) { return false; }
  static_assert(kMaxSrc * 4 <= 64 && kMaxSrc + kMaxSbox <= 64 && kTmS % 4 == 0, "lanes");
  const SimIoArgs& a;
  int x0, y0, rows;  // what the tile writes: columns x0 .., rows y0 ..
  int comp, kind, i0, i1, j0, j1;  // this lane's box (kind: a sample box's column)
  double value[kTmS / 4], prof, div;  // (prof: the address's bits)
  gptr<const double> table;
  unsigned smask, bmask;

  __device__ __forceinline__ void first() {
    const int lane = threadIdx.x & 63;
    const int t = min(lane, a.n_src - 1), u = min(max(lane - kMaxSrc, 0), a.n_sbox - 1);
    const bool is_src = lane < a.n_src, is_box = lane >= kMaxSrc && lane - kMaxSrc < a.n_sbox;
    comp = kind = i0 = i1 = j0 = j1 = 0;
    prof = div = 0.0;
    table = nullptr;
#pragma unroll
    for (int v = 0; v < kTmS / 4; ++v) value[v] = 0.0;
    if (a.n_src > 0) {
      const gptr<const KSrc> q = (gptr<const KSrc>)a.src + t;
      if (is_src) {
        comp = q->comp;
        kind = q->kind;
        i0 = q->i0;
        i1 = q->k0 < q->k1 ? q->i1 : q->i0;
        j0 = q->j0;
        j1 = q->j1;
        prof = __builtin_bit_cast(double, (uint64_t)q->profile);
        div = q->divisor;
      }
      table = (gptr<const double>)((gptr<const KSrc>)a.src + min(lane / 4, a.n_src - 1))->table;
    }
    if (is_box) {
      const gptr<const KSbox> q = (gptr<const KSbox>)a.sbox + u;
      comp = q->comp;
      kind = q->col0;
      i0 = q->i0;
      i1 = q->k0 < q->k1 ? q->i1 : q->i0;
      j0 = q->j0;
      j1 = q->j1;
    }
  }

  __device__ __forceinline__ void second(int ns) {
    const int lane = threadIdx.x & 63;
    const bool is_src = lane < a.n_src, is_box = lane >= kMaxSrc && lane - kMaxSrc < a.n_sbox;
    if (a.n_src > 0) {
      const int64_t row = a.row + (a.clock ? *a.clock : 0);
#pragma unroll
      for (int v = 0; v < kTmS / 4; ++v) value[v] = table[row + min(4 * v + lane % 4, ns - 1)];
    }
    // sources act on the halo too, samples on what the tile writes
    const int h = is_src ? kTmS : 0;
    const bool hit = (is_src || is_box) && i0 < x0 + kTmCols + h && i1 > x0 - h && i0 < i1 &&
                     j0 < y0 + rows + h && j1 > y0 - h && j0 < j1;
    const unsigned long long m = __ballot(hit);
    smask = (unsigned)(m & ((1u << kMaxSrc) - 1));
    bmask = (unsigned)(m >> kMaxSrc);
  }

  __device__ __forceinline__ int of(int v, int l) const { return __builtin_amdgcn_readlane(v, l); }

  template <int R>
  __device__ __forceinline__ void add(int t, int s, int i, int jb, T (&f)[R]) const {
    const int b0 = of(i0, t), b1 = of(i1, t), c0 = of(j0, t), c1 = of(j1, t);
    double v = tm_bcast(value[0], t * 4 + (s & 3));
#pragma unroll
    for (int k = 1; k < kTmS / 4; ++k) v = s / 4 == k ? tm_bcast(value[k], t * 4 + (s & 3)) : v;
    const bool in = i >= b0 && i < b1;
    if (c0 >= jb + R || c1 <= jb) return;  // uniform
    if (of(kind, t) == 0) {
      const T u = (T)v;
      tm_add([&](int) { return u; }, in, c0, c1, jb, f);
      return;
    }
    // the profile's values of all rows from clamped positions, without a
    // branch between them: one wait for the loads, not one per row
    const gptr<const double> p =
        (gptr<const double>)__builtin_bit_cast(uint64_t, tm_bcast(prof, t));
    const double d = tm_bcast(div, t);
    const int ni = b1 - b0, ic = min(max(i, b0), b1 - 1) - b0;
    double u[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      u[r] = p[(int64_t)(min(max(jb + r, c0), c1 - 1) - c0) * ni + ic];
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = v * u[r];
    if (d != 0.0) {
#pragma unroll
      for (int r = 0; r < R; ++r) u[r] = u[r] / d;
    }
    tm_add([&](int r) { return (T)u[r]; }, in, c0, c1, jb, f);
  }

  template <int R>
  __device__ __forceinline__ void sources(int s, int i, int jb, T (&ez)[R], T (&hx)[R],
                                          T (&hy)[R]) const {
    for (unsigned m = smask; m; m &= m - 1) {
      const int t = __builtin_ctz(m), c = of(comp, t);
      if (c == PM_EZ) add(t, s, i, jb, ez);
      else if (c == PM_HX) add(t, s, i, jb, hx);
      else add(t, s, i, jb, hy);
    }
  }

  template <int R>
  __device__ __forceinline__ void put(int t, int s, int i, int jb, const T (&f)[R]) const {
    const int b0 = of(i0, t), b1 = of(i1, t), c0 = of(j0, t), c1 = of(j1, t), ni = b1 - b0;
    const bool in = i >= max(b0, x0) && i < min(b1, x0 + kTmCols);
    const gptr<T> X = (gptr<T>)a.X + (a.xrow + s) * (int64_t)a.ncols + of(kind, t) + (i - b0);
    const int p0 = max(c0, y0), p1 = min(c1, y0 + rows);  // rows the tile writes
    tm_put(X + (int64_t)(p0 - c0) * ni, ni, in, p0, p1, jb, f);
  }

  template <int R>
  __device__ __forceinline__ void samples(int s, int i, int jb, const T (&ez)[R],
                                          const T (&hx)[R], const T (&hy)[R]) const {
    for (unsigned m = bmask; m; m &= m - 1) {
      const int t = kMaxSrc + __builtin_ctz(m), c = of(comp, t);
      if (c == PM_EZ) put(t, s, i, jb, ez);
      else if (c == PM_HX) put(t, s, i, jb, hx);
      else put(t, s, i, jb, hy);
    }
  }
};

template <typename T, int CK, int R>
__global__ __launch_bounds__(64 * kTmW, 4) void k_tm2d_multi(const TmGrid g, const SimProf pr,
                                                             const SimIoArgs io, int ns,
                                                             int nstrip) {
  __shared__ TmShared<T, R> sh;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int b = tm_order(blockIdx.x, gridDim.x);
  const int x0 = (b % nstrip) * kTmCols, y0 = (b / nstrip) * tm_rows(R);
  const int i = x0 - kTmS + lane;
  const bool xpml = i >= 0 && i < g.nx && (i < g.px0 || i >= g.nx - g.px1);
  TmXProf<T> xp{(T)0, (T)0, (T)1, (T)0, (T)0, (T)1};
  if (xpml) {
    xp.be = ((gptr<const T>)pr.x[0])[i];
    xp.ce = ((gptr<const T>)pr.x[1])[i];
    xp.ike = ((gptr<const T>)pr.x[2])[i];
    xp.bh = ((gptr<const T>)pr.x[3])[i];
    xp.ch = ((gptr<const T>)pr.x[4])[i];
    xp.ikh = ((gptr<const T>)pr.x[5])[i];
  }
  SimY<T> yp;
#pragma unroll
  for (int k = 0; k < 6; ++k) yp.p[k] = (gptr<const T>)pr.y[k];
  SimIo<T> o{io, x0, y0, tm_rows(R)};
  (void)tm_tile<T, CK, R>(g, xp, xpml, yp, o, ns, x0, y0, w, sh);
}

template <typename T, int CK, int R>
int launch_rows(const TmGrid& g, const SimProf& pr, const SimIoArgs& io, int ns,
                 hipStream_t s) {
  const int nstrip = (g.nx + kTmCols - 1) / kTmCols;
  const int ntile = (g.ny + tm_rows(R) - 1) / tm_rows(R);
  hipLaunchKernelGGL((k_tm2d_multi<T, CK, R>), dim3(nstrip * ntile), dim3(64 * kTmW), 0, s, g,
                     pr, io, ns, nstrip);
  return 0;
}

template <typename T, int CK>
int launch_ck(const TmGrid& g, const SimProf& pr, const SimIoArgs& io, int ns, int R,
              hipStream_t s) {
  if constexpr (sizeof(T) == 4) {
    if (R == 8) return launch_rows<T, CK, 8>(g, pr, io, ns, s);
  }
  return launch_rows<T, CK, 4>(g, pr, io, ns, s);
}

}  // namespace

int launch_tm2d_multi(const KGrid& g, int precision, int ck, const Tm2dBufs& b, const KAux* src,
                      const KAux* smp, int64_t step, const int64_t* clock, int ns, int n_cu,
                      hipStream_t s) {
  if (g.ndim != 2 || g.n_ade || ns < 1 || ns > kTmS) return -1;
  if (precision == PM_FP64 ? ck == PM_COEFF_CB_F16 || ck == PM_COEFF_FULL : ck == PM_COEFF_FULL)
    return -1;
  TmGrid t{};
  t.nx = g.nx;
  t.ny = g.ny;
  t.sy = (uint32_t)g.sy;
  t.px0 = g.pml[0];
  t.px1 = g.pml[1];
  t.py0 = g.pml[2];
  t.py1 = g.pml[3];
  t.ez = b.Ei;
  t.hx = b.Hi[0];
  t.hy = b.Hi[1];
  t.ez_o = b.Eo;
  t.hx_o = b.Ho[0];
  t.hy_o = b.Ho[1];
  t.ca = g.ca[2];
  t.cb = g.cb[2];
  for (int q = 0; q < 2; ++q) {
    // an axis without CPML: element 0 of Ez, read and not used
    t.ps[q] = b.psh_in[q] ? b.psh_in[q] : b.Ei;
    t.ps_o[q] = b.psh_out[q];
    t.ps[2 + q] = b.pse_in[q] ? b.pse_in[q] : b.Ei;
    t.ps_o[2 + q] = b.pse_out[q];
  }
  t.xst = (uint32_t)(g.pml[0] + g.pml[1]);
  t.yst = (uint32_t)g.nx;
  t.full = false;
  t.idx = g.idx;
  t.idy = g.idy;
  t.db = g.db_const;
  t.cb_scale = g.cb_scale;
  SimProf pr{};
  for (int a = 0; a < 2; ++a) {
    const void** d = a == 0 ? pr.x : pr.y;
    d[0] = g.pml_be[a];
    d[1] = g.pml_ce[a];
    d[2] = g.pml_ike[a];
    d[3] = g.pml_bh[a];
    d[4] = g.pml_ch[a];
    d[5] = g.pml_ikh[a];
  }
  SimIoArgs io{};
  if (src) {
    io.src = src->src_dev;
    io.n_src = src->n_src;
    io.row = step - src->table_step0;
  }
  if (smp) {
    io.sbox = smp->sbox_dev;
    io.n_sbox = smp->n_sbox;
    io.ncols = smp->ncols;
    io.xrow = step % smp->sample_T;
    io.X = smp->X;
  }
  io.clock = clock;
  const int R = tm_pick_rows((double)g.nx * g.ny, precision == PM_FP64 ? 8 : 4, n_cu);
  if (precision == PM_FP64)
    return ck == PM_COEFF_CACB ? launch_ck<double, PM_COEFF_CACB>(t, pr, io, ns, R, s)
                               : launch_ck<double, PM_COEFF_CB>(t, pr, io, ns, R, s);
  if (ck == PM_COEFF_CACB) return launch_ck<float, PM_COEFF_CACB>(t, pr, io, ns, R, s);
  if (ck == PM_COEFF_CB_F16) return launch_ck<float, PM_COEFF_CB_F16>(t, pr, io, ns, R, s);
  return launch_ck<float, PM_COEFF_CB>(t, pr, io, ns, R, s);
}

int tm2d_multi_steps() { return kTmS; }

}  // namespace pm
