// Batched 2-D TM stepping of many uneven grids (include/pmbatch.h).
//
// One launch advances every design by up to eight steps: a workgroup takes one
// tile of one design (tm2d_pass.h), and a table gives it the design and the
// tile.  One step per launch moved 300 MB a step for 64 coupler grids of
// 9.8 M cells together: 68 us at 4.5 TB/s, the rate of a large copy, so only
// fewer passes over the state could make it faster; eight steps a pass take 148
// us, 18 a step, two thirds of which the vector ALU is busy (a third of the tiles
// of a coupler touch a CPML layer).  Reads come from field set `par`, writes go
// to set par ^ 1, so neighbouring tiles never see a half-updated value; the CPML
// memory of both field halves is ping-ponged for the same reason.  The plan has
// one E-side set, which spans the grid; the second, in the workspace, holds the
// layers alone (28 k values, not 334 k, for 540 x 290 cells with 16 layers a
// side), and calls begin and end with the state in the plan's.  Sources are added
// after the E update, samples are taken after the sources, as
// src/prismo/core/simulation.py:147-164 orders them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/pmbatch.h"
#include "tm2d_pass.h"

namespace pm {
namespace {

struct KWork {
  int d, x0, y0;
};

// A design and the second set of its E-side CPML memory: x layers (pml[0] +
// pml[1] values per row), y layers (pml[2] + pml[3] rows of sy).
struct KDesign {
  pm_batch_design d;
  void* psi_ex1;
  void* psi_ey1;
};

struct KBatch {
  const KDesign* des;
  const KWork* work;
  const KWork* work1;  // of one step
  int ncols, sample_T;
  int64_t* clock;
  int32_t* status;  // per design: bit 0 set once an Ez value was not finite
  int xcd;          // 1: XCD-grouped workgroup order, 0: launch order
  double idx, idy;
  const double* tab_e;
  const double* tab_h;
  int64_t table_step0;
  void* X;
};

template <typename T>
struct BatchY {
  gptr<const T> p;  // 8 values per row
  __device__ __forceinline__ T operator()(int k, int j) const { return p[8 * j + k]; }
};

// Sources (one Ez and one Hy line) and sample lines of a tile.  Lane l holds
// line l and the source values of step l of the pass: loaded beside the fields,
// read back with lane broadcasts.  Lines that do not meet the tile are masked
// out; most tiles have none.
template <typename T, int S>
struct BatchIo {
  static constexpr bool kStatus = true, kPackedE = true;
  static_assert(PM_BATCH_MAX_LINES <= 64 && kTmS <= 64, "one lane per entry");
  const KBatch& k;
  const pm_batch_design& D;
  int64_t step;      // of the pass's first step
  int x0, y0, rows;  // what the tile writes: columns x0 .., rows y0 ..
  int pe;            // the E-side memory set read
  int comp, col, li, j0, j1;  // this lane's line
  T ve, vh;
  int se_i, se0, se1, sh_i, sh0, sh1;
  bool hit_e, hit_h;
  unsigned mask;
  gptr<T> X;

  __device__ __forceinline__ bool packed(bool out) const { return (pe != 0) != (S > 1 && out); }

  __device__ __forceinline__ void first() {
    const int lane = threadIdx.x & 63;
    comp = col = li = j0 = j1 = 0;
    if (lane < D.n_lines) {
      const gptr<const pm_batch_line> L = (gptr<const pm_batch_line>)D.line + lane;
      comp = L->comp;
      li = L->i;
      j0 = L->j0;
      j1 = L->j1;
      col = L->col;
    }
    se_i = D.src_e[0];
    se0 = D.src_e[1];
    se1 = D.src_e[2];
    sh_i = D.src_h[0];
    sh0 = D.src_h[1];
    sh1 = D.src_h[2];
    X = (gptr<T>)k.X + (step % k.sample_T) * (int64_t)k.ncols;
  }

  // sources act on the halo too, samples on what the tile writes
  __device__ __forceinline__ bool meets(int i, int a, int b, int h) const {
    return i >= x0 - h && i < x0 + tm_cols(S) + h && a < y0 + rows + h && b > y0 - h && a < b;
  }

  __device__ __forceinline__ void second(int ns) {
    const int lane = threadIdx.x & 63;
    const int64_t row = step - k.table_step0 + min(lane, ns - 1);
    ve = (T)((gptr<const double>)k.tab_e)[row];
    vh = (T)((gptr<const double>)k.tab_h)[row];
    hit_e = meets(se_i, se0, se1, S);
    hit_h = meets(sh_i, sh0, sh1, S);
    mask = (unsigned)__ballot(meets(li, j0, j1, 0));
  }

  template <int R>
  __device__ __forceinline__ void sources(int s, int i, int jb, T (&ez)[R], T (&hx)[R],
                                          T (&hy)[R]) const {
    if (hit_e) {
      const T v = tm_bcast(ve, s);
      tm_add([&](int) { return v; }, i == se_i, se0, se1, jb, ez);
    }
    if (hit_h) {
      const T v = tm_bcast(vh, s);
      tm_add([&](int) { return v; }, i == sh_i, sh0, sh1, jb, hy);
    }
  }

  __device__ __forceinline__ int of(int v, int l) const { return __builtin_amdgcn_readlane(v, l); }

  template <int R>
  __device__ __forceinline__ void put(int t, int s, int i, int jb, const T (&f)[R]) const {
    const int c0 = of(j0, t), c1 = of(j1, t);
    const int p0 = max(c0, y0), p1 = min(c1, y0 + rows);  // rows the tile writes
    const gptr<T> x = X + s * (int64_t)k.ncols + of(col, t) + (p0 - c0);
    tm_put(x, 1, i == of(li, t), p0, p1, jb, f);
  }

  template <int R>
  __device__ __forceinline__ void samples(int s, int i, int jb, const T (&ez)[R],
                                          const T (&hx)[R], const T (&hy)[R]) const {
    for (unsigned m = mask; m; m &= m - 1) {
      const int t = __builtin_ctz(m), c = of(comp, t);
      if (c == 0) put(t, s, i, jb, ez);
      else if (c == 1) put(t, s, i, jb, hx);
      else put(t, s, i, jb, hy);
    }
  }
};

// S = 8: up to eight steps; S = 1: one step, whose tiles have a halo of one cell
// (62 columns by 30 rows written of 64 by 32, not 48 by 16) and whose E-side
// memory is updated in place: its neighbour may have written a halo cell's value
// before the tile reads it, but that goes into the halo cell's E alone, which a
// single step does not use.  par: field set read, pe: E-side memory set read.  Calls of one step (32 designs of 532 x 332 cells):
// with S = 8 46 us FP32, 131 FP64; with S = 1 33 and 82 (one step per launch and
// no halo: 42 and 84).
template <typename T, int CK, int R, int S>
__global__ __launch_bounds__(64 * kTmW, 4) void k_batch_tm(const KBatch k, int64_t step_arg,
                                                           int use_clock, int s_rel, int ns,
                                                           int par, int pe) {
  __shared__ TmShared<T, R> sh;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int b = k.xcd ? tm_order(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const KWork wk = (S > 1 ? k.work : k.work1)[b];
  const KDesign& KD = k.des[wk.d];
  const pm_batch_design& D = KD.d;
  const int x0 = wk.x0, y0 = wk.y0;
  const int nx = D.nx;
  TmGrid g;
  g.nx = nx;
  g.ny = D.ny;
  g.sy = g.xst = g.yst = (uint32_t)D.sy;
  g.px0 = D.pml[0];
  g.px1 = D.pml[1];
  g.py0 = D.pml[2];
  g.py1 = D.pml[3];
  g.ez = D.ez[par];
  g.hx = D.hx[par];
  g.hy = D.hy[par];
  g.ez_o = D.ez[par ^ 1];
  g.hx_o = D.hx[par ^ 1];
  g.hy_o = D.hy[par ^ 1];
  g.ca = nullptr;
  g.cb = D.cb;
  g.ps[0] = D.psi_hy[par];
  g.ps[1] = D.psi_hx[par];
  g.ps[2] = pe ? KD.psi_ex1 : D.psi_ex;
  g.ps[3] = pe ? KD.psi_ey1 : D.psi_ey;
  g.ps_o[0] = D.psi_hy[par ^ 1];
  g.ps_o[1] = D.psi_hx[par ^ 1];
  const bool second = (pe != 0) != (S > 1);
  g.ps_o[2] = second ? KD.psi_ex1 : D.psi_ex;
  g.ps_o[3] = second ? KD.psi_ey1 : D.psi_ey;
  g.full = true;
  g.idx = k.idx;
  g.idy = k.idy;
  g.db = D.db;
  g.cb_scale = D.cb_scale;
  const gptr<const T> prof = (gptr<const T>)D.prof;
  const int i = x0 - S + lane;
  const bool xpml = i >= 0 && i < nx && (i < g.px0 || i >= nx - g.px1);
  TmXProf<T> xp{(T)0, (T)0, (T)1, (T)0, (T)0, (T)1};
  if (xpml) {
    xp.be = prof[i];
    xp.ce = prof[nx + i];
    xp.ike = prof[2 * nx + i];
    xp.bh = prof[3 * nx + i];
    xp.ch = prof[4 * nx + i];
    xp.ikh = prof[5 * nx + i];
  }
  const BatchY<T> yp{prof + 6 * (int64_t)nx};
  BatchIo<T, S> io{k, D, use_clock ? *k.clock + s_rel : step_arg, x0, y0, tm_rows(R, S), pe};
  const uint32_t bad = tm_tile<T, CK, R, S>(g, xp, xpml, yp, io, ns, x0, y0, w, sh);
  // a diverged design is flagged by the lanes that saw it (rare)
  if (bad >> 31) atomicOr(k.status + wk.d, 1);
}

// The layers of every design (blockIdx.y) from the plan's E-side CPML memory to the
// workspace's (pack) or back: at the ends of a call whose state is in set 1.
template <typename T>
__global__ __launch_bounds__(256) void k_batch_psi(const KDesign* des, int pack) {
  const KDesign& KD = des[blockIdx.y];
  const pm_batch_design& D = KD.d;
  const int sx = D.pml[0] + D.pml[1], sl = D.pml[2] + D.pml[3];
  const int64_t n = (int64_t)sx * D.ny, m = n + (int64_t)sl * D.nx;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < m;
       e += (int64_t)gridDim.x * 256) {
    T *full, *layers;
    if (e < n) {
      const int s = (int)(e % sx);
      full = (T*)D.psi_ex + e / sx * D.sy + (s < D.pml[0] ? s : D.nx - sx + s);
      layers = (T*)KD.psi_ex1 + e;
    } else {
      const int s = (int)((e - n) / D.nx), i = (int)((e - n) % D.nx);
      full = (T*)D.psi_ey + (int64_t)(s < D.pml[2] ? s : D.ny - sl + s) * D.sy + i;
      layers = (T*)KD.psi_ey1 + (int64_t)s * D.sy + i;
    }
    if (pack) *layers = *full;
    else *full = *layers;
  }
}

__global__ void k_clock_set(int64_t* clock, int64_t v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *clock = v;
}

__global__ void k_clock_add(int64_t* clock, int64_t v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *clock += v;
}

}  // namespace
}  // namespace pm

using namespace pm;

struct pm_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  bool configured = false;
  pm_batch_plan plan{};
  std::vector<pm_batch_design> des;
  std::vector<KWork> work, work1;  // tiles of up to eight steps, of one
  int rows = 4;                    // rows per wave of a tile
  KBatch kb{};
  KDft dft{};
  int64_t step = 0;   // absolute index of the next step
  int parity = 0;     // field set that holds the state
  int pe = 0;         // E-side memory set
  int64_t pend0 = 0;  // first step of the pending sample block
  int pend_n = 0;
  hipGraphExec_t graph[4] = {};  // per starting sets: parity + 2 pe
  int n_cu = 256;
  int xcd = 1;  // workgroup order (pm_batch_set_tuning)
  bool timing = false;
  int64_t timed_steps = 0;  // steps in spans[0]
  std::vector<std::pair<hipEvent_t, hipEvent_t>> spans[3];
  std::string err;
};

namespace {

int bfail(pm_batch* b, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  if (b) b->err = buf;
  return code;
}

int bhip(pm_batch* b, hipError_t e, const char* what) {
  if (e == hipSuccess) return 0;
  return bfail(b, (int)e, "%s: %s", what, hipGetErrorString(e));
}

struct BSpan {
  pm_batch* b;
  int which;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  BSpan(pm_batch* bb, int w) : b(bb), which(w) {
    if (b->timing && hipEventCreateWithFlags(&e0, hipEventDisableSystemFence) == hipSuccess &&
        hipEventCreateWithFlags(&e1, hipEventDisableSystemFence) == hipSuccess)
      (void)hipEventRecord(e0, b->stream);
  }
  ~BSpan() {
    if (e0 && e1) {
      (void)hipEventRecord(e1, b->stream);
      b->spans[which].push_back({e0, e1});
    }
  }
};

int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// Workspace: the step clock at offset 0, then the design table, the tile
// lists, one status word per design and the second E-side CPML memory.
struct Layout {
  int64_t des, work, work1, status, psi, total;
};

void build_work(const pm_batch_plan& p, int rows, int halo, std::vector<KWork>& work) {
  work.clear();
  for (int d = 0; d < p.n_design; ++d) {
    const pm_batch_design& D = p.design[d];
    for (int y0 = 0; y0 < D.ny; y0 += tm_rows(rows, halo))
      for (int x0 = 0; x0 < D.nx; x0 += tm_cols(halo)) work.push_back(KWork{d, x0, y0});
  }
}

// Second E-side CPML memory of the x (axis 0) or y layers of a design; without
// layers one value is still read.
int64_t psi_bytes(const pm_batch_plan& p, const pm_batch_design& D, int axis) {
  const int64_t n = (int64_t)(D.pml[2 * axis] + D.pml[2 * axis + 1]) * (axis ? D.sy : D.ny);
  return align256(std::max<int64_t>(n, 1) * (p.precision == PM_FP64 ? 8 : 4));
}

// (sized for the shortest tiles, whichever the device gets)
Layout layout(const pm_batch_plan& p) {
  std::vector<KWork> w, w1;
  build_work(p, 4, kTmS, w);
  build_work(p, 4, 1, w1);
  Layout l{};
  l.des = 256;
  l.work = align256(l.des + (int64_t)sizeof(KDesign) * p.n_design);
  l.work1 = align256(l.work + (int64_t)(sizeof(KWork) * w.size()));
  l.status = align256(l.work1 + (int64_t)(sizeof(KWork) * w1.size()));
  l.psi = align256(l.status + (int64_t)sizeof(int32_t) * p.n_design);
  l.total = l.psi;
  for (int d = 0; d < p.n_design; ++d)
    l.total += psi_bytes(p, p.design[d], 0) + psi_bytes(p, p.design[d], 1);
  return l;
}

int validate(pm_batch* b, const pm_batch_plan& p) {
  if (p.abi_version != PM_ABI_VERSION) return bfail(b, PM_EINVAL, "ABI version mismatch");
  if (p.precision != PM_FP64 && p.precision != PM_FP32)
    return bfail(b, PM_EINVAL, "precision must be PM_FP64 or PM_FP32");
  if (p.coeff_kind != PM_COEFF_CB && p.coeff_kind != PM_COEFF_CB_F16)
    return bfail(b, PM_EINVAL, "coeff_kind must be CB or CB_F16");
  if (p.n_design < 1 || !p.design) return bfail(b, PM_EINVAL, "no designs");
  if (!(p.dx > 0) || !(p.dy > 0) || !(p.dt > 0)) return bfail(b, PM_EINVAL, "bad dx/dy/dt");
  if (p.chunk < 2) return bfail(b, PM_EINVAL, "chunk must be >= 2");
  if (p.sample_T < 1 || p.ncols < 0 || !p.X) return bfail(b, PM_EINVAL, "bad sample ring");
  if (!p.src_e_table || !p.src_h_table || p.table_len < 1)
    return bfail(b, PM_EINVAL, "source tables required");
  if (p.nfreq < 0) return bfail(b, PM_EINVAL, "bad nfreq");
  if (p.nfreq > 0) {
    if (!p.W_re || !p.W_im || !p.dft.acc_re || !p.dft.acc_im)
      return bfail(b, PM_EINVAL, "spectra need W tables and accumulators");
    if (p.dft.col0 < 0 || p.dft.col1 > p.ncols || p.dft.col0 >= p.dft.col1 ||
        p.dft.f0 < 0 || p.dft.f1 > p.nfreq || p.dft.f0 >= p.dft.f1)
      return bfail(b, PM_EINVAL, "DFT group outside the sample columns / frequencies");
    if (p.precision == PM_FP32 && (!p.dft.cmp_re || !p.dft.cmp_im))
      return bfail(b, PM_EINVAL, "FP32 spectra need compensation arrays");
  }
  for (int d = 0; d < p.n_design; ++d) {
    const pm_batch_design& D = p.design[d];
    if (D.nx < 2 || D.ny < 2 || D.sy < D.nx) return bfail(b, PM_EINVAL, "design %d: bad size", d);
    // the kernel addresses a design's arrays with 32-bit byte offsets
    if ((int64_t)D.ny * D.sy * (p.precision == PM_FP64 ? 8 : 4) >= (int64_t)1 << 32)
      return bfail(b, PM_EINVAL, "design %d: %d x %lld cells exceed 32-bit offsets", d, D.ny,
                   (long long)D.sy);
    for (int s = 0; s < 2; ++s)
      if (!D.ez[s] || !D.hx[s] || !D.hy[s] || !D.psi_hx[s] || !D.psi_hy[s])
        return bfail(b, PM_EINVAL, "design %d: missing field or CPML arrays", d);
    if (!D.psi_ex || !D.psi_ey || !D.cb || !D.prof)
      return bfail(b, PM_EINVAL, "design %d: missing arrays", d);
    if (D.pml[0] < 0 || D.pml[1] < 0 || D.pml[2] < 0 || D.pml[3] < 0 ||
        D.pml[0] + D.pml[1] > D.nx || D.pml[2] + D.pml[3] > D.ny)
      return bfail(b, PM_EINVAL, "design %d: bad CPML layers", d);
    if (D.n_lines < 0 || D.n_lines > PM_BATCH_MAX_LINES)
      return bfail(b, PM_EINVAL, "design %d: too many sample lines", d);
    for (int l = 0; l < D.n_lines; ++l) {
      const pm_batch_line& L = D.line[l];
      if (L.comp < 0 || L.comp > 2 || L.i < 0 || L.i >= D.nx || L.j0 < 0 || L.j1 > D.ny ||
          L.j0 > L.j1 || L.col < 0 || L.col + (L.j1 - L.j0) > p.ncols)
        return bfail(b, PM_EINVAL, "design %d: bad sample line %d", d, l);
    }
    // Ez exists on (nx-1) x (ny-1), Hy on nx x (ny-1)
    if (D.src_e[1] < 0 || D.src_e[1] > D.src_e[2] ||
        (D.src_e[2] > D.src_e[1] && (D.src_e[0] < 0 || D.src_e[0] >= D.nx - 1 ||
                                     D.src_e[2] > D.ny - 1)))
      return bfail(b, PM_EINVAL, "design %d: Ez source line outside Ez", d);
    if (D.src_h[1] < 0 || D.src_h[1] > D.src_h[2] ||
        (D.src_h[2] > D.src_h[1] && (D.src_h[0] < 0 || D.src_h[0] >= D.nx ||
                                     D.src_h[2] > D.ny - 1)))
      return bfail(b, PM_EINVAL, "design %d: Hy source line outside Hy", d);
  }
  return 0;
}

template <typename T, int CK>
void launch_ck(pm_batch* b, int64_t step_arg, int use_clock, int s_rel, int ns, int par, int pe) {
  const dim3 nt(64 * kTmW), nb((unsigned)(ns == 1 ? b->work1 : b->work).size());
  if (ns == 1) {
    hipLaunchKernelGGL((k_batch_tm<T, CK, 4, 1>), nb, nt, 0, b->stream, b->kb, step_arg,
                       use_clock, s_rel, ns, par, pe);
    return;
  }
  if constexpr (sizeof(T) == 4) {
    if (b->rows == 8) {
      hipLaunchKernelGGL((k_batch_tm<T, CK, 8, kTmS>), nb, nt, 0, b->stream, b->kb, step_arg,
                         use_clock, s_rel, ns, par, pe);
      return;
    }
  }
  hipLaunchKernelGGL((k_batch_tm<T, CK, 4, kTmS>), nb, nt, 0, b->stream, b->kb, step_arg,
                     use_clock, s_rel, ns, par, pe);
}

// ns steps from field set `par` into the other, and, more than one, from E-side
// memory set `pe` into the other; both are advanced.
int launch_steps(pm_batch* b, int64_t step, int use_clock, int s_rel, int ns, int* par, int* pe) {
  const bool f16 = b->plan.coeff_kind == PM_COEFF_CB_F16;
  if (b->plan.precision == PM_FP64) {
    if (f16) launch_ck<double, PM_COEFF_CB_F16>(b, step, use_clock, s_rel, ns, *par, *pe);
    else launch_ck<double, PM_COEFF_CB>(b, step, use_clock, s_rel, ns, *par, *pe);
  } else {
    if (f16) launch_ck<float, PM_COEFF_CB_F16>(b, step, use_clock, s_rel, ns, *par, *pe);
    else launch_ck<float, PM_COEFF_CB>(b, step, use_clock, s_rel, ns, *par, *pe);
  }
  *par ^= 1;
  if (ns > 1) *pe ^= 1;
  return bhip(b, hipGetLastError(), "batch step launch");
}

// With the E-side CPML memory's state in set 1: from the plan's arrays into the
// workspace (before steps, pack) or back (after them).
int move_psi(pm_batch* b, bool pack) {
  if (b->pe == 0) return 0;
  int64_t most = 0;
  for (const pm_batch_design& D : b->des)
    most = std::max(most, (int64_t)(D.pml[0] + D.pml[1]) * D.ny +
                              (int64_t)(D.pml[2] + D.pml[3]) * D.nx);
  if (most == 0) return 0;
  const unsigned nb = (unsigned)std::min<int64_t>((most + 255) / 256, 256);
  for (size_t d0 = 0; d0 < b->des.size(); d0 += 65535) {
    const dim3 grid(nb, (unsigned)std::min<size_t>(b->des.size() - d0, 65535));
    if (b->plan.precision == PM_FP64)
      hipLaunchKernelGGL(k_batch_psi<double>, grid, dim3(256), 0, b->stream, b->kb.des + d0,
                         pack ? 1 : 0);
    else
      hipLaunchKernelGGL(k_batch_psi<float>, grid, dim3(256), 0, b->stream, b->kb.des + d0,
                         pack ? 1 : 0);
  }
  return bhip(b, hipGetLastError(), "batch CPML memory launch");
}

int flush_block(pm_batch* b, int64_t first, int rows, const int64_t* wclock) {
  const pm_batch_plan& p = b->plan;
  if (p.nfreq == 0 || rows == 0) return 0;
  const int esz = p.precision == PM_FP64 ? 8 : 4;
  const char* X0 = (const char*)p.X + (first % p.sample_T) * (int64_t)p.ncols * esz;
  const int64_t wcol = wclock ? p.table_step0 : first - p.table_step0;
  launch_dft(b->dft, X0, p.ncols, p.W_re, p.W_im, p.table_len, wcol, rows, p.precision,
             b->stream, wclock);
  return bhip(b, hipGetLastError(), "batch DFT launch");
}

int capture(pm_batch* b, int slot) {
  int par = slot & 1, pe = slot >> 1;
  const pm_batch_plan& p = b->plan;
  hipGraph_t g = nullptr;
  int r = bhip(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal),
               "begin capture");
  if (r) return r;
  for (int s = 0; s < p.sample_T && !r; s += kTmS)
    r = launch_steps(b, 0, 1, s, std::min(kTmS, p.sample_T - s), &par, &pe);
  if (!r) r = flush_block(b, 0, p.sample_T, b->kb.clock);
  if (!r) {
    hipLaunchKernelGGL(k_clock_add, dim3(1), dim3(64), 0, b->stream, b->kb.clock,
                       (int64_t)p.sample_T);
    r = bhip(b, hipGetLastError(), "clock launch");
  }
  hipError_t e = hipStreamEndCapture(b->stream, &g);
  if (r) {
    if (g) (void)hipGraphDestroy(g);
    return r;
  }
  r = bhip(b, e, "end capture");
  if (r) return r;
  r = bhip(b, hipGraphInstantiate(&b->graph[slot], g, nullptr, nullptr, 0), "instantiate");
  (void)hipGraphDestroy(g);
  return r;
}

void drop_graphs(pm_batch* b) {
  for (auto& g : b->graph)
    if (g) {
      (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
}

}  // namespace

extern "C" {

int pm_batch_create(int device, void* stream, pm_batch** out) {
  if (!out) return PM_EINVAL;
  *out = nullptr;
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) return (int)e;
  if (device < 0 || device >= n) return PM_EINVAL;
  e = hipSetDevice(device);
  if (e != hipSuccess) return (int)e;
  pm_batch* b = new pm_batch();
  b->device = device;
  int cu = 0;
  if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
      cu > 0)
    b->n_cu = cu;
  b->stream = (hipStream_t)stream;
  *out = b;
  return 0;
}

int pm_batch_destroy(pm_batch* b) {
  if (!b) return PM_EINVAL;
  (void)hipSetDevice(b->device);
  drop_graphs(b);
  for (auto& v : b->spans)
    for (auto& ab : v) {
      (void)hipEventDestroy(ab.first);
      (void)hipEventDestroy(ab.second);
    }
  delete b;
  return 0;
}

const char* pm_batch_last_error(pm_batch* b) { return b ? b->err.c_str() : "null handle"; }

int pm_batch_workspace_bytes(const pm_batch_plan* p, int64_t* bytes) {
  if (!p || !bytes || p->n_design < 1 || !p->design || p->chunk < 2) return PM_EINVAL;
  *bytes = layout(*p).total;
  return 0;
}

int pm_batch_configure(pm_batch* b, const pm_batch_plan* p) {
  if (!b || !p) return PM_EINVAL;
  (void)hipSetDevice(b->device);
  b->configured = false;
  drop_graphs(b);
  int r = validate(b, *p);
  if (r) return r;
  const Layout l = layout(*p);
  if (!p->work || p->work_bytes < l.total)
    return bfail(b, PM_EINVAL, "workspace of %lld bytes required", (long long)l.total);
  double cells = 0;
  for (int d = 0; d < p->n_design; ++d) cells += (double)p->design[d].nx * p->design[d].ny;
  b->rows = tm_pick_rows(cells, p->precision == PM_FP64 ? 8 : 4, b->n_cu);
  std::vector<KWork> work, work1;
  build_work(*p, b->rows, kTmS, work);
  build_work(*p, 4, 1, work1);
  b->plan = *p;
  b->des.assign(p->design, p->design + p->n_design);
  b->plan.design = b->des.data();
  b->work = std::move(work);
  b->work1 = std::move(work1);
  char* ws = (char*)p->work;
  std::vector<KDesign> kd(b->des.size());
  char* psi = ws + l.psi;
  for (size_t d = 0; d < kd.size(); ++d) {
    const int64_t n = psi_bytes(*p, b->des[d], 0);
    kd[d] = KDesign{b->des[d], psi, psi + n};
    psi += n + psi_bytes(*p, b->des[d], 1);
  }
  KBatch& k = b->kb;
  k.clock = (int64_t*)ws;
  k.des = (const KDesign*)(ws + l.des);
  k.work = (const KWork*)(ws + l.work);
  k.work1 = (const KWork*)(ws + l.work1);
  k.status = (int32_t*)(ws + l.status);
  k.xcd = b->xcd;
  k.ncols = p->ncols;
  k.sample_T = p->sample_T;
  k.idx = 1.0 / p->dx;
  k.idy = 1.0 / p->dy;
  k.tab_e = p->src_e_table;
  k.tab_h = p->src_h_table;
  k.table_step0 = p->table_step0;
  k.X = p->X;
  b->dft = KDft{p->dft.col0, p->dft.col1, p->dft.f0, p->dft.f1, p->dft.acc_re,
                p->dft.acc_im, p->dft.cmp_re, p->dft.cmp_im};
  r = bhip(b, hipMemcpyAsync((void*)k.des, kd.data(), sizeof(KDesign) * kd.size(),
                             hipMemcpyHostToDevice, b->stream), "design table upload");
  if (!r)
    r = bhip(b, hipMemcpyAsync((void*)k.work, b->work.data(), sizeof(KWork) * b->work.size(),
                               hipMemcpyHostToDevice, b->stream), "tile list upload");
  if (!r)
    r = bhip(b, hipMemcpyAsync((void*)k.work1, b->work1.data(), sizeof(KWork) * b->work1.size(),
                               hipMemcpyHostToDevice, b->stream), "tile list upload");
  // status words start clear (an upload, not a memset: nothing here is
  // captured, but the same holds for every buffer a graph reads)
  const std::vector<int32_t> zeros((size_t)p->n_design, 0);
  if (!r)
    r = bhip(b, hipMemcpyAsync(k.status, zeros.data(), sizeof(int32_t) * zeros.size(),
                               hipMemcpyHostToDevice, b->stream), "status upload");
  // the uploads read pageable host memory: finish them
  if (!r) r = bhip(b, hipStreamSynchronize(b->stream), "upload sync");
  if (r) return r;
  b->step = p->table_step0;
  b->parity = b->pe = 0;
  b->pend0 = b->step;
  b->pend_n = 0;
  b->configured = true;
  return 0;
}

int pm_batch_run(pm_batch* b, int32_t nsteps, uint32_t flags) {
  if (!b) return PM_EINVAL;
  if (!b->configured) return bfail(b, PM_ENOPLAN, "pm_batch_run before pm_batch_configure");
  if (nsteps < 0) return bfail(b, PM_EINVAL, "nsteps < 0");
  const pm_batch_plan& p = b->plan;
  if (b->step + nsteps > p.table_step0 + p.table_len)
    return bfail(b, PM_ERANGE, "source/phasor tables end at step %lld",
                 (long long)(p.table_step0 + p.table_len));
  (void)hipSetDevice(b->device);
  const int T = p.sample_T;
  const bool graphs = (flags & PM_RUN_GRAPH) && (T % 2 == 0);
  if ((flags & PM_RUN_GRAPH) && !graphs)
    return bfail(b, PM_EINVAL, "graph replay needs an even sample_T");
  if (graphs && b->stream == nullptr)
    return bfail(b, PM_EINVAL, "graph replay needs a non-default stream");
  int64_t left = nsteps;
  bool clock_ok = false;
  if (left > 0) {
    const int r = move_psi(b, true);
    if (r) return r;
  }
  while (left > 0) {
    if (graphs && b->step % T == 0 && b->pend_n == 0 && left >= T) {
      int r = 0;
      const int slot = b->parity + 2 * b->pe;
      if (!b->graph[slot]) r = capture(b, slot);
      if (r) return r;
      if (!clock_ok) {
        hipLaunchKernelGGL(k_clock_set, dim3(1), dim3(64), 0, b->stream, b->kb.clock, b->step);
        r = bhip(b, hipGetLastError(), "clock launch");
        if (r) return r;
        clock_ok = true;
      }
      {
        BSpan sp(b, 2);
        r = bhip(b, hipGraphLaunch(b->graph[slot], b->stream), "graph launch");
      }
      if (r) return r;
      // (T is even: no launch of the block holds one step)
      const int odd = ((T + kTmS - 1) / kTmS) & 1;
      b->parity ^= odd;
      b->pe ^= odd;
      b->step += T;
      b->pend0 = b->step;
      left -= T;
      continue;
    }
    clock_ok = false;
    // a launch does not cross the end of a sample block
    const int m = (int)std::min<int64_t>({kTmS, left, T - b->step % T});
    int r;
    {
      BSpan sp(b, 0);
      r = launch_steps(b, b->step, 0, 0, m, &b->parity, &b->pe);
    }
    if (r) return r;
    if (b->timing) b->timed_steps += m;
    if (b->pend_n == 0) b->pend0 = b->step;
    b->pend_n += m;
    b->step += m;
    left -= m;
    if (b->step % T == 0) {
      BSpan sp(b, 1);
      r = flush_block(b, b->pend0, b->pend_n, nullptr);
      if (r) return r;
      b->pend_n = 0;
      b->pend0 = b->step;
    }
  }
  return nsteps > 0 ? move_psi(b, false) : 0;
}

int pm_batch_flush(pm_batch* b) {
  if (!b) return PM_EINVAL;
  if (!b->configured) return bfail(b, PM_ENOPLAN, "pm_batch_flush before configure");
  (void)hipSetDevice(b->device);
  int r = flush_block(b, b->pend0, b->pend_n, nullptr);
  if (r) return r;
  b->pend_n = 0;
  b->pend0 = b->step;
  return 0;
}

int pm_batch_parity(pm_batch* b) { return b ? b->parity : PM_EINVAL; }
int64_t pm_batch_steps(pm_batch* b) { return b ? b->step - b->plan.table_step0 : PM_EINVAL; }

int pm_batch_sync(pm_batch* b) {
  if (!b) return PM_EINVAL;
  (void)hipSetDevice(b->device);
  return bhip(b, hipStreamSynchronize(b->stream), "sync");
}

int pm_batch_set_tuning(pm_batch* b, int waves, int xcd_order) {
  if (!b) return PM_EINVAL;
  if (waves != 1 && waves != 2 && waves != 4 && waves != 8)
    return bfail(b, PM_EINVAL, "waves per workgroup must be 1, 2, 4 or 8");
  if (xcd_order != 0 && xcd_order != 1) return bfail(b, PM_EINVAL, "xcd_order must be 0 or 1");
  (void)hipSetDevice(b->device);
  // a captured graph holds the old workgroup order
  drop_graphs(b);
  b->xcd = b->kb.xcd = xcd_order;
  return 0;
}

int pm_batch_design_status(pm_batch* b, int32_t* out, int32_t n) {
  if (!b || !out) return PM_EINVAL;
  if (!b->configured) return bfail(b, PM_ENOPLAN, "pm_batch_design_status before configure");
  if (n != b->plan.n_design)
    return bfail(b, PM_EINVAL, "status of %d designs asked, the plan has %d", n,
                 b->plan.n_design);
  (void)hipSetDevice(b->device);
  int r = bhip(b, hipStreamSynchronize(b->stream), "status sync");
  if (!r)
    r = bhip(b, hipMemcpyAsync(out, b->kb.status, sizeof(int32_t) * (size_t)n,
                               hipMemcpyDeviceToHost, b->stream), "status download");
  if (!r) r = bhip(b, hipStreamSynchronize(b->stream), "status sync");
  return r;
}

int pm_batch_set_timing(pm_batch* b, int enable) {
  if (!b) return PM_EINVAL;
  b->timing = enable != 0;
  b->timed_steps = 0;
  for (auto& v : b->spans) {
    for (auto& ab : v) {
      (void)hipEventDestroy(ab.first);
      (void)hipEventDestroy(ab.second);
    }
    v.clear();
  }
  return 0;
}

int pm_batch_get_timing(pm_batch* b, int which, double* avg_ms, int64_t* count) {
  if (!b || which < 0 || which > 2 || !avg_ms || !count) return PM_EINVAL;
  (void)hipSetDevice(b->device);
  double tot = 0;
  int64_t n = 0;
  for (auto& ab : b->spans[which]) {
    float ms = 0;
    if (hipEventSynchronize(ab.second) != hipSuccess) continue;
    if (hipEventElapsedTime(&ms, ab.first, ab.second) == hipSuccess) {
      tot += ms;
      ++n;
    }
  }
  // a launch holds several steps: class 0 counts those
  if (which == 0 && n) n = b->timed_steps;
  *avg_ms = n ? tot / n : 0.0;
  *count = n;
  return 0;
}

}  // extern "C"
