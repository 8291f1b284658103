// Surrogate MLP kernels (include/pmmlp.h): a BF16 MFMA GEMM with fused
// bias / GELU / GELU-derivative epilogues, the bias-gradient column sum,
// the weighted MSE loss and gradient, and Adam.
//
// GEMM tiling: a workgroup of 4 waves owns a 64 x 64 block of C; each wave a
// 32 x 32 quarter as 2 x 2 V_MFMA_F32_16X16X32_BF16 tiles.  K goes in blocks
// of 128: the workgroup stages A (64 x 128) and B (128 x 64) in LDS as BF16,
// both k-contiguous per row/column, so each lane reads its 8-element operand
// with one 16-byte LDS load, and runs 4 MFMA K-steps of 32 on the block.
// The next block's global loads are issued into registers before those
// MFMAs, so a GEMM of K <= 256 (every surrogate layer) waits for memory
// about once instead of once per K-step.  The global loads walk the
// unit-stride side of each operand, whichever it is (forward: X rows and W
// rows; input gradient: W columns; weight gradient: dY and X columns over
// the batch).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/pmmlp.h"
#include "../../include/pmfdtd.h"

namespace pm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 64, kBN = 64, kBK = 128, kPad = 8;
constexpr int kStage = kBM * kBK / 256;  // elements of A (and of B) per thread per block

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ unsigned short to_bf16(float x) {
  unsigned u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float gelu(float z) {
  return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
}

// d gelu / dz = Phi(z) + z phi(z)
__device__ __forceinline__ float dgelu(float z) {
  const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

// Operand strides per problem of a batch (blockIdx.z), 0 for a single GEMM.
struct GemmBatch {
  int64_t a, b, c, bias, z;
};

struct GemmLds {
  unsigned short a[kBM][kBK + kPad];
  unsigned short b[kBN][kBK + kPad];
};

// The 64 x 64 block of C at (m0, n0), by the 256 threads of a workgroup.
__device__ __forceinline__ void gemm_tile(int mode, int M, int N, int K,
                                          const float* __restrict__ A, int64_t lam, int64_t lak,
                                          const float* __restrict__ B, int64_t lbk, int64_t lbn,
                                          float* __restrict__ C, int64_t ldc,
                                          const float* __restrict__ bias, float* __restrict__ Z,
                                          int m0, int n0, GemmLds& lds) {
  auto& sa = lds.a;
  auto& sb = lds.b;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;
  const int li = lane & 15, lq = lane >> 4;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0, 0, 0, 0};

  const bool a_kfast = lak == 1;
  const bool b_kfast = lbk == 1;
  // element e of this thread's share of a block: (row, k) of A and (n, k) of
  // B, along the unit-stride axis of each
  auto a_rc = [&](int e, int& r, int& c) {
    const int f = tid + 256 * e;
    if (a_kfast) {
      r = f / kBK;
      c = f % kBK;
    } else {
      r = f % kBM;
      c = f / kBM;
    }
  };
  auto b_rc = [&](int e, int& r, int& c) {
    const int f = tid + 256 * e;
    if (b_kfast) {
      r = f / kBK;
      c = f % kBK;
    } else {
      r = f % kBN;
      c = f / kBN;
    }
  };
  float ra[kStage], rb[kStage];
  auto gload = [&](int k0) {
#pragma unroll
    for (int e = 0; e < kStage; ++e) {
      int r, c;
      a_rc(e, r, c);
      const int m = m0 + r, k = k0 + c;
      ra[e] = (m < M && k < K) ? A[(int64_t)m * lam + (int64_t)k * lak] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < kStage; ++e) {
      int r, c;
      b_rc(e, r, c);
      const int n = n0 + r, k = k0 + c;
      rb[e] = (n < N && k < K) ? B[(int64_t)k * lbk + (int64_t)n * lbn] : 0.0f;
    }
  };
  gload(0);
  for (int k0 = 0; k0 < K; k0 += kBK) {
#pragma unroll
    for (int e = 0; e < kStage; ++e) {
      int r, c;
      a_rc(e, r, c);
      sa[r][c] = to_bf16(ra[e]);
      b_rc(e, r, c);
      sb[r][c] = to_bf16(rb[e]);
    }
    __syncthreads();
    if (k0 + kBK < K) gload(k0 + kBK);  // in flight during this block's MFMAs
#pragma unroll
    for (int kk = 0; kk < kBK; kk += 32) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const unsigned short* p = &sa[wm + 16 * a + li][kk + 8 * lq];
        av[a] = *(const bf16x8*)p;
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const unsigned short* p = &sb[wn + 16 * b + li][kk + 8 * lq];
        bv[b] = *(const bf16x8*)p;
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
    }
    __syncthreads();
  }
  // epilogue: lane holds rows 4 lq + r, column li of each 16 x 16 tile
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * a + 4 * lq + r;
        const int n = n0 + wn + 16 * b + li;
        if (m >= M || n >= N) continue;
        float v = acc[a][b][r];
        const int64_t o = (int64_t)m * ldc + n;
        if (mode == PM_MLP_LINEAR) {
          C[o] = bias ? v + bias[n] : v;
        } else if (mode == PM_MLP_GELU) {
          const float z = bias ? v + bias[n] : v;
          Z[o] = z;
          C[o] = gelu(z);
        } else if (mode == PM_MLP_DGELU) {
          C[o] = v * dgelu(Z[o]);
        } else {
          C[o] = v;
        }
      }
}

__global__ __launch_bounds__(256) void k_gemm(int mode, int M, int N, int K,
                                              const float* __restrict__ A, int64_t lam,
                                              int64_t lak, const float* __restrict__ B,
                                              int64_t lbk, int64_t lbn, float* __restrict__ C,
                                              int64_t ldc, const float* __restrict__ bias,
                                              float* __restrict__ Z, GemmBatch bs) {
  __shared__ GemmLds lds;
  const int64_t q = blockIdx.z;
  gemm_tile(mode, M, N, K, A + q * bs.a, lam, lak, B + q * bs.b, lbk, lbn, C + q * bs.c, ldc,
            bias ? bias + q * bs.bias : nullptr, Z ? Z + q * bs.z : nullptr, blockIdx.y * kBM,
            blockIdx.x * kBN, lds);
}

// one workgroup per 64 columns; 4 waves split the rows, then combine in LDS
__device__ __forceinline__ void colsum_tile(int M, int N, const float* __restrict__ A,
                                            int64_t lda, float* __restrict__ out, int c0,
                                            float (&part)[4][64]) {
  const int c = c0 + (threadIdx.x & 63);
  const int w = threadIdx.x >> 6;
  float s = 0.0f;
  if (c < N)
    for (int m = w; m < M; m += 4) s += A[(int64_t)m * lda + c];
  part[w][threadIdx.x & 63] = s;
  __syncthreads();
  if (w == 0 && c < N)
    out[c] = (part[0][threadIdx.x] + part[1][threadIdx.x]) +
             (part[2][threadIdx.x] + part[3][threadIdx.x]);
}

__global__ __launch_bounds__(256) void k_colsum(int M, int N, const float* __restrict__ A,
                                                int64_t lda, float* __restrict__ out,
                                                int64_t sa, int64_t so) {
  __shared__ float part[4][64];
  const int64_t q = blockIdx.y;  // problem of a batch
  colsum_tile(M, N, A + q * sa, lda, out + q * so, blockIdx.x * 64, part);
}

__global__ __launch_bounds__(256) void k_mse(int M, int N, const float* __restrict__ Y,
                                             const float* __restrict__ T,
                                             const float* __restrict__ w,
                                             float* __restrict__ dY, float* loss, int64_t sy) {
  __shared__ float red[256];
  {
    const int64_t q = blockIdx.y;  // problem of a batch: Y, T, dY at q sy, loss[q]
    Y += q * sy;
    T += q * sy;
    dY += q * sy;
    loss += q;
  }
  const int64_t total = (int64_t)M * N;
  const float scale = 1.0f / (float)total;
  float s = 0.0f;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * 256) {
    const int n = (int)(e % N);
    const float wt = w ? w[n] : 1.0f;
    const float d = Y[e] - T[e];
    s += wt * d * d;
    dY[e] = 2.0f * wt * d * scale;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0] * scale);
}

__global__ __launch_bounds__(256) void k_adam(int64_t n, float* __restrict__ p,
                                              const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v,
                                              float lr, float b1, float b2, float eps, float wd,
                                              float c1, float c2) {
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * 256) {
    const float gi = g[e];
    const float mi = b1 * m[e] + (1.0f - b1) * gi;
    const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
    m[e] = mi;
    v[e] = vi;
    const float mh = mi / c1, vh = vi / c2;
    p[e] -= lr * (mh / (sqrtf(vh) + eps) + wd * p[e]);
  }
}

// ------------------------------------------------------- whole networks
// A layer-by-layer pass moves every activation through memory between
// launches of 64 x 64 tiles: on 65 536 rows of a 4 x 256 network 86 us a
// layer, on a training batch of 256 rows 24 us a launch with 64 workgroups
// (a sixteenth of the chip) waiting for memory.  Here a workgroup takes BM
// rows through all layers, the activations staying in LDS as the BF16 values
// the next product would round them to anyway (the same products in the same
// order: the sums are bitwise those of gemm_tile).  What it reads per layer is
// the weights alone, packed as BF16 in operand order (one 16-byte load per
// lane, tile and K-step, no guard), from L2.
//
// 8 waves as WR x WC; a wave owns RT row tiles and NT column tiles of 16,
// column tiles interleaved over the waves (tile t WC + wc).

constexpr int kNetL = 12;      // layers
constexpr int kNetWidth = 512; // widest layer

// A network of L layers of widths n[0] .. n[L], parameters flat per member:
// all weights (row-major [out][in]), then all biases.
struct NetDesc {
  int L;
  int n[kNetL + 1];
  int64_t woff[kNetL], boff[kNetL];  // in the member's flat parameters
  int64_t poff[kNetL], qoff[kNetL];  // packed weights, packed transposed weights
  int64_t aoff[kNetL];               // rows times this: hidden layer k's values
  int64_t goff[kNetL];               // rows times this: layer k's output gradient
  int64_t nW, nP;                    // weights, parameters
  int64_t nfwd, npack;               // packed elements without / with the transposes
  int64_t nhid, ngrad;               // values per row over hidden / all layers
  // training workspace, widths padded to 16: pre-activations (zpad values a
  // row, layer k from zpo[k]), inputs, gradients
  int64_t zpad, apad, gpad;
  int64_t zpo[kNetL], apo[kNetL], gpo[kNetL];
  int kp;                            // LDS row: widest padded operand + 8
};

__host__ __device__ constexpr int up32(int n) { return (n + 31) & ~31; }
__host__ __device__ constexpr int up16(int n) { return (n + 15) & ~15; }

// Operand order: tile of 16 columns (n) x 32 k: lane l holds column l % 16,
// k = 8 (l / 16) .. + 7.
__device__ __forceinline__ int64_t pack_at(int n, int k, int K) {
  const int kt = up32(K) / 32;
  const int lane = (n & 15) + 16 * ((k >> 3) & 3);
  return (((int64_t)(n >> 4) * kt + (k >> 5)) * 64 + lane) * 8 + (k & 7);
}

// The packed copies of parameter e (a weight); transposed ones where the
// backward pass takes them (not of the first layer).
__device__ __forceinline__ void pack_weight(const NetDesc& d, unsigned short* pk, int64_t e,
                                            float v, bool trans) {
  int k = 0;
  while (k + 1 < d.L && e >= d.woff[k + 1]) ++k;
  const int fi = d.n[k];
  const int r = (int)(e - d.woff[k]);
  const int o = r / fi, i = r - o * fi;
  const unsigned short b = to_bf16(v);
  pk[d.poff[k] + pack_at(o, i, fi)] = b;
  if (trans && k > 0) pk[d.qoff[k] + pack_at(i, o, d.n[k + 1])] = b;
}

__global__ __launch_bounds__(256) void k_net_pack(const NetDesc d, const float* __restrict__ P,
                                                  int64_t ps, unsigned short* __restrict__ pk,
                                                  int64_t ks, int trans) {
  const int64_t q = blockIdx.y;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < d.nW;
       e += (int64_t)gridDim.x * 256)
    pack_weight(d, pk + q * ks, e, P[q * ps + e], trans != 0);
}

extern __shared__ unsigned short net_lds[];

__device__ __forceinline__ bf16x4 to_bf16x4(f32x4 v) { return __builtin_convertvector(v, bf16x4); }

// The wave's weight tiles of PD K-steps, in flight ahead of the products that
// take them: a K-step's loads wait for L2 or the Infinity Cache (the weights
// were just written by other XCDs), 1 to 2 us against 0.1 us of MFMA.
template <int NT, int WC, int PD>
struct NetTiles {
  bf16x8 b[PD][NT];
  __device__ __forceinline__ static bf16x8 at(const unsigned short* pk, int wc, int t, int ntiles,
                                              int kt, int s) {
    // tiles past the layer's width repeat the last one (unused)
    const int nt = min(t * WC + wc, ntiles - 1);
    const unsigned short* base = pk + ((int64_t)nt * kt + s) * 512;  // uniform
    return *(const bf16x8*)(base + 8 * (threadIdx.x & 63));
  }
  __device__ __forceinline__ void fill(const unsigned short* pk, int wc, int N, int K) {
    const int kt = up32(K) / 32, ntiles = up16(N) / 16;
#pragma unroll
    for (int p = 0; p < PD; ++p)
#pragma unroll
      for (int t = 0; t < NT; ++t) b[p][t] = at(pk, wc, t, ntiles, kt, min(p, kt - 1));
  }
};

// acc = W A over K (padded to 32) for this wave's tiles: weights from the packed
// buffer (first K-steps already in w), activations from LDS rows.  The weights
// are the row operand, so a lane holds 4 consecutive columns (16 tile + 4 lq + e)
// of one activation row (row0 + 16 r + li): one 8-byte LDS store and one 16-byte
// memory store where the other order takes four of each.
template <int RT, int NT, int WC, int PD>
__device__ __forceinline__ void net_gemm(const unsigned short* sA, int kp, int row0, int wc, int N,
                                         int K, const unsigned short* __restrict__ pk,
                                         NetTiles<NT, WC, PD>& w, f32x4 (&acc)[RT][NT]) {
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int kt = up32(K) / 32, ntiles = up16(N) / 16;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][t] = f32x4{0, 0, 0, 0};
  const unsigned short* ap = sA + (row0 + li) * kp + 8 * lq;
  for (int s0 = 0; s0 < kt; s0 += PD) {
#pragma unroll
    for (int p = 0; p < PD; ++p) {
      const int s = s0 + p;
      if (s < kt) {
        bf16x8 wv[NT], av[RT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          wv[t] = w.b[p][t];
          // this slot's next K-step, or, when the layer fits the slots, the
          // matrix the slots serve next
          if (s + PD < kt) w.b[p][t] = w.at(pk, wc, t, ntiles, kt, s + PD);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) av[r] = *(const bf16x8*)(ap + 16 * r * kp + 32 * s);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[t], av[r], acc[r][t], 0, 0, 0);
      }
    }
  }
}

// Values n .. n+3 of a row of N (beyond N the last one: the caller does not use
// them).
__device__ __forceinline__ f32x4 load4(const float* p, int n, int N) {
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = p[min(n + e, N - 1)];
  return v;
}

// All biases of a member into LDS behind the activation rows: read from memory
// in the epilogue they would wait for the next layer's weights, issued before
// them (vector loads return in order).
__device__ __forceinline__ float* net_biases(unsigned short* sA, int rows, const NetDesc& d,
                                             const float* __restrict__ Pq) {
  float* sb = (float*)(sA + rows * d.kp);
  for (int f = threadIdx.x; f < (int)d.ngrad; f += blockDim.x) sb[f] = Pq[d.nW + f];
  return sb;
}

// The same stored; vec: rows are 16-byte aligned.
__device__ __forceinline__ void store4(float* p, int n, int N, bool vec, f32x4 v) {
  if (vec) {
    if (n < N) *(f32x4*)(p + n) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) p[n + e] = v[e];
}

// Rows m0 .. of src (row stride ld, through idx when given) into LDS as BF16,
// zero beyond the rows and beyond column n up to a multiple of 32.
__device__ __forceinline__ void net_stage(unsigned short* sA, int kp, int bm, int m0, int M,
                                          int n, const float* __restrict__ src, int64_t ld,
                                          const int64_t* __restrict__ idx) {
  const int np = up32(n);
  for (int f = threadIdx.x; f < bm * np; f += blockDim.x) {
    const int r = f / np, c = f - r * np;
    float v = 0.0f;
    if (m0 + r < M && c < n) {
      const int64_t row = idx ? idx[m0 + r] : m0 + r;
      v = src[row * ld + c];
    }
    sA[r * kp + c] = to_bf16(v);
  }
}

// Y = network(X) for rows of every member (blockIdx.y); hidden activations and
// pre-activations kept in acts / zs (member stride as_, layer k at M aoff[k])
// when given.
//
// Two workgroups of the tall shape share a CU (128 VGPRs): one's products run
// beside the other's epilogue.
template <int RT, int NT, int WR, int WC, int PD>
__global__ __launch_bounds__(64 * WR * WC, RT == 4 && NT == 4 ? 4 : 1) void k_net_forward(
    const NetDesc d, int M, const float* __restrict__ P, int64_t ps,
    const unsigned short* __restrict__ pk, int64_t ks, const float* __restrict__ X, int64_t xs,
    float* __restrict__ Y, int64_t ys, float* __restrict__ acts, float* __restrict__ zs,
    int64_t as_) {
  constexpr int BM = 16 * RT * WR;
  unsigned short* sA = net_lds;
  const int64_t q = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wv / WC, wc = wv % WC;
  const int m0 = blockIdx.x * BM, row0 = wr * 16 * RT;
  const float* Pq = P + q * ps;
  const unsigned short* pq = pk + q * ks;
  Y += q * ys;
  const bool yvec = d.n[d.L] % 4 == 0 && ((uintptr_t)Y & 15) == 0;
  NetTiles<NT, WC, PD> w;
  w.fill(pq + d.poff[0], wc, d.n[1], d.n[0]);
  net_stage(sA, d.kp, BM, m0, M, d.n[0], X + q * xs, d.n[0], nullptr);
  const float* sb = net_biases(sA, BM, d, Pq);
  __syncthreads();
  for (int k = 0; k < d.L; ++k) {
    const int K = d.n[k], N = d.n[k + 1];
    f32x4 acc[RT][NT];
    net_gemm<RT, NT, WC, PD>(sA, d.kp, row0, wc, N, K, pq + d.poff[k], w, acc);
    const bool last = k + 1 == d.L;
    // the next layer's first weights come in during the epilogue
    if (!last) w.fill(pq + d.poff[k + 1], wc, d.n[k + 2], N);
    __syncthreads();  // every wave has read its operands: the rows are replaced
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = 16 * (t * WC + wc) + 4 * lq;
      if (16 * (t * WC + wc) >= up32(N)) continue;
      const f32x4 bias = load4(sb + d.goff[k], n, N);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const int row = row0 + 16 * r + li, m = m0 + row;
        const f32x4 z = acc[r][t] + bias;
        if (last) {
          if (m < M) store4(Y + (int64_t)m * N, n, N, yvec, z);
          continue;
        }
        f32x4 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = n + e < N ? gelu(z[e]) : 0.0f;
        *(bf16x4*)(sA + row * d.kp + n) = to_bf16x4(a);
        if (zs && m < M) {
          const int64_t o = q * as_ + (int64_t)M * d.aoff[k] + (int64_t)m * N;
          store4(zs + o, n, N, false, z);
          store4(acts + o, n, N, false, a);
        }
      }
    }
    __syncthreads();
  }
}

// Workspace of one training minibatch (rows padded to B32, a multiple of 32):
// pre-activations (row stride up16), the layers' inputs and output gradients as
// BF16 in the operand order of the weight gradients (K = row), and each
// 16-row block's column sums of the gradients.
struct NetWork {
  float* zs;
  unsigned short* a;
  unsigned short* g;
  float* part;
};

__host__ __device__ inline int64_t net_work_floats(const NetDesc& d, int B32) {
  return B32 * (d.zpad + d.apad / 2 + d.gpad / 2) + (B32 / 16) * d.ngrad;
}

__device__ __forceinline__ NetWork net_work(const NetDesc& d, float* work, int64_t q, int B32) {
  float* p = work + q * ((net_work_floats(d, B32) + 3) & ~3ll);
  NetWork w;
  w.zs = p;
  p += B32 * d.zpad;
  w.a = (unsigned short*)p;
  p += B32 * (d.apad / 2);
  w.g = (unsigned short*)p;
  p += B32 * (d.gpad / 2);
  w.part = p;
  return w;
}

// The 16 LDS rows (block m0) of width N as operand tiles with K = row.
__device__ __forceinline__ void net_rows_out(const unsigned short* sA, int kp, int N, int m0,
                                             int B32, unsigned short* __restrict__ dst) {
  const int kt = B32 / 32;
  for (int f = threadIdx.x; f < 2 * up16(N); f += blockDim.x) {
    const int n = f >> 1, h = f & 1;
    typedef unsigned short us8 __attribute__((ext_vector_type(8)));
    us8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = sA[(8 * h + e) * kp + n];
    const int lane = (n & 15) + 16 * (((m0 >> 3) & 3) + h);
    *(us8*)(dst + (((int64_t)(n >> 4) * kt + (m0 >> 5)) * 64 + lane) * 8) = v;
  }
}

// One training minibatch of every member (blockIdx.y), 16 rows per workgroup:
// forward, the weighted squared error's gradient and loss, and the gradient
// carried back to the first hidden layer.  Rows are gathered through idx; rows
// from B to B32 have zero gradients.
template <int NT, int PD>
__global__ __launch_bounds__(512) void k_net_train(
    const NetDesc d, int B, int B32, const float* __restrict__ P, int64_t ps,
    const unsigned short* __restrict__ pk, int64_t ks, const float* __restrict__ X,
    const float* __restrict__ T, const int64_t* __restrict__ idx, int64_t is,
    const float* __restrict__ wcol, float* __restrict__ work, float* __restrict__ loss) {
  constexpr int WC = 8;
  unsigned short* sA = net_lds;
  __shared__ float red[8];
  const int64_t q = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int wc = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.x * 16, m = m0 + li;
  const float* Pq = P + q * ps;
  const unsigned short* pq = pk + q * ks;
  idx += q * is;
  const NetWork W = net_work(d, work, q, B32);
  float* part = W.part + (int64_t)blockIdx.x * d.ngrad;
  NetTiles<NT, WC, PD> w;
  w.fill(pq + d.poff[0], wc, d.n[1], d.n[0]);
  net_stage(sA, d.kp, 16, m0, B, d.n[0], X, d.n[0], idx);
  const float* sb = net_biases(sA, 16, d, Pq);
  const int64_t trow = m < B ? idx[m] : 0;
  __syncthreads();
  net_rows_out(sA, d.kp, d.n[0], m0, B32, W.a + (int64_t)B32 * d.apo[0]);
  const int NL = d.n[d.L];
  const float scale = 1.0f / (float)((int64_t)B * NL);
  float s = 0.0f;
  // column sums over the block's rows (the 16 lanes of a quarter wave)
  auto rows16 = [&](f32x4 v) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 1; h < 16; h *= 2)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += __shfl_xor(v[e], h);
    return v;
  };
  for (int k = 0; k < d.L; ++k) {
    const int K = d.n[k], N = d.n[k + 1];
    f32x4 acc[1][NT];
    net_gemm<1, NT, WC, PD>(sA, d.kp, 0, wc, N, K, pq + d.poff[k], w, acc);
    const bool last = k + 1 == d.L;
    // targets ahead of the weights that the backward pass starts with
    f32x4 y[NT], wt[NT];
    if (last) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = min(16 * (t * WC + wc) + 4 * lq, N - 1);
        y[t] = load4(T + trow * NL, n, N);
        wt[t] = wcol ? load4(wcol, n, N) : f32x4{1, 1, 1, 1};
      }
    }
    if (!last) w.fill(pq + d.poff[k + 1], wc, d.n[k + 2], N);
    else if (k > 0) w.fill(pq + d.qoff[k], wc, d.n[k], N);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = 16 * (t * WC + wc) + 4 * lq;
      if (16 * (t * WC + wc) >= up32(N)) continue;
      const f32x4 z = acc[0][t] + load4(sb + d.goff[k], n, N);
      f32x4 v = {0, 0, 0, 0};
      if (last) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= N || m >= B) continue;
          const float dd = z[e] - y[t][e];
          s += wt[t][e] * dd * dd;
          v[e] = 2.0f * wt[t][e] * dd * scale;
        }
        const f32x4 sum = rows16(v);
        if (li == 0) store4(part + d.goff[k], n, N, false, sum);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = n + e < N ? gelu(z[e]) : 0.0f;
        if (n < up16(N))
          *(f32x4*)(W.zs + B32 * d.zpo[k] + (int64_t)m * up16(N) + n) = z;
      }
      *(bf16x4*)(sA + li * d.kp + n) = to_bf16x4(v);
    }
    __syncthreads();
    net_rows_out(sA, d.kp, N, m0, B32,
                 last ? W.g + (int64_t)B32 * d.gpo[k] : W.a + (int64_t)B32 * d.apo[k + 1]);
  }
  // back through the layers: G_{k-1} = (G_k W_k) gelu'(z_{k-1})
  for (int k = d.L - 1; k > 0; --k) {
    const int K = d.n[k + 1], N = d.n[k];
    f32x4 acc[1][NT], z[NT];
    // this thread stored these pre-activations in the forward pass
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = min(16 * (t * WC + wc) + 4 * lq, up16(N) - 4);
      z[t] = *(const f32x4*)(W.zs + B32 * d.zpo[k - 1] + (int64_t)m * up16(N) + n);
    }
    net_gemm<1, NT, WC, PD>(sA, d.kp, 0, wc, N, K, pq + d.qoff[k], w, acc);
    if (k > 1) w.fill(pq + d.qoff[k - 1], wc, d.n[k - 1], N);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = 16 * (t * WC + wc) + 4 * lq;
      if (16 * (t * WC + wc) >= up32(N)) continue;
      f32x4 v = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N && m < B) v[e] = acc[0][t][e] * dgelu(z[t][e]);
      const f32x4 sum = rows16(v);
      if (li == 0) store4(part + d.goff[k - 1], n, N, false, sum);
      *(bf16x4*)(sA + li * d.kp + n) = to_bf16x4(v);
    }
    __syncthreads();
    net_rows_out(sA, d.kp, N, m0, B32, W.g + (int64_t)B32 * d.gpo[k - 1]);
  }
  for (int h = 32; h >= 1; h >>= 1) s += __shfl_xor(s, h);
  if (lane == 0) red[wc] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float a = 0.0f;
    for (int i = 0; i < 8; ++i) a += red[i];
    atomicAdd(loss + q, a * scale);
  }
}

struct AdamArgs {
  float lr, b1, b2, eps, wd, c1, c2;
};

// k_adam's update of one parameter.
__device__ __forceinline__ float adam_one(const AdamArgs& h, float g, float wd, float p, float& m,
                                          float& v) {
  m = h.b1 * m + (1.0f - h.b1) * g;
  v = h.b2 * v + (1.0f - h.b2) * g * g;
  const float mh = m / h.c1, vh = v / h.c2;
  return p - h.lr * (mh / (sqrtf(vh) + h.eps) + wd * p);
}

// Weight gradients G_k^T a_k (64 x 64 tiles, operands straight from the
// workspace, no LDS), bias gradients (the blocks' column sums added up) and
// Adam on the parameters they belong to, with the packed copies of the new
// weights: one launch for all layers and members, the gradients and moments
// of a tile in registers throughout.
__global__ __launch_bounds__(256) void k_net_update(const NetDesc d, int B32,
                                                    float* __restrict__ work,
                                                    float* __restrict__ P, float* __restrict__ G,
                                                    float* __restrict__ mm,
                                                    float* __restrict__ vv, int64_t ps,
                                                    unsigned short* __restrict__ pk, int64_t ks,
                                                    AdamArgs h) {
  const int64_t q = blockIdx.y;
  const NetWork W = net_work(d, work, q, B32);
  P += q * ps;
  G += q * ps;
  mm += q * ps;
  vv += q * ps;
  pk += q * ks;
  int b = blockIdx.x;
  int k = 0, gx = 0;
  for (; k < d.L; ++k) {
    gx = (d.n[k] + 63) / 64;
    const int jobs = gx * ((d.n[k + 1] + 63) / 64) + 1;
    if (b < jobs) break;
    b -= jobs;
  }
  if (k >= d.L) return;
  const int fi = d.n[k], fo = d.n[k + 1];
  if (b == 0) {
    for (int n = threadIdx.x; n < fo; n += 256) {
      float s = 0.0f;
      for (int i = 0; i < B32 / 16; ++i) s += W.part[(int64_t)i * d.ngrad + d.goff[k] + n];
      const int64_t o = d.boff[k] + n;
      float m = mm[o], v = vv[o];
      G[o] = s;
      P[o] = adam_one(h, s, 0.0f, P[o], m, v);
      mm[o] = m;
      vv[o] = v;
    }
    return;
  }
  b -= 1;
  constexpr int PD = 8;  // a minibatch of 256 rows is all in flight at once
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, lq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int o0 = (b / gx) * 64 + (wv >> 1) * 32, i0 = (b % gx) * 64 + (wv & 1) * 32;
  if (o0 >= fo || i0 >= fi) return;
  const int kt = B32 / 32;
  const unsigned short* ga = W.g + (int64_t)B32 * d.gpo[k] + 8 * lane;
  const unsigned short* aa = W.a + (int64_t)B32 * d.apo[k] + 8 * lane;
  // tiles past the layer repeat its last one (unused)
  int64_t go[2], ao[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    go[t] = (int64_t)min(o0 / 16 + t, up16(fo) / 16 - 1) * kt * 512;
    ao[t] = (int64_t)min(i0 / 16 + t, up16(fi) / 16 - 1) * kt * 512;
  }
  bf16x8 gv[PD][2], av[PD][2];
#pragma unroll
  for (int p = 0; p < PD; ++p)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      gv[p][t] = *(const bf16x8*)(ga + go[t] + min(p, kt - 1) * 512);
      av[p][t] = *(const bf16x8*)(aa + ao[t] + min(p, kt - 1) * 512);
    }
  // the tile's parameters and moments, behind the operands (loads return in
  // order); lane: rows o = 4 lq + e, column i = li of each 16 x 16 tile
  f32x4 acc[2][2], pv[2][2], mv[2][2], vm[2][2];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc[r][c] = f32x4{0, 0, 0, 0};
      const int i = min(i0 + 16 * c + li, fi - 1), ob = o0 + 16 * r + 4 * lq;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t o = d.woff[k] + (int64_t)min(ob + e, fo - 1) * fi + i;
        pv[r][c][e] = P[o];
        mv[r][c][e] = mm[o];
        vm[r][c][e] = vv[o];
      }
    }
  for (int s0 = 0; s0 < kt; s0 += PD) {
#pragma unroll
    for (int p = 0; p < PD; ++p) {
      const int s = s0 + p;
      if (s < kt) {
        const bf16x8 g0 = gv[p][0], g1 = gv[p][1], a0 = av[p][0], a1 = av[p][1];
        if (s + PD < kt) {
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            gv[p][t] = *(const bf16x8*)(ga + go[t] + (s + PD) * 512);
            av[p][t] = *(const bf16x8*)(aa + ao[t] + (s + PD) * 512);
          }
        }
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g0, a0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g0, a1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g1, a0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g1, a1, acc[1][1], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int i = i0 + 16 * c + li, ob = o0 + 16 * r + 4 * lq;
      if (i >= fi) continue;
      float pn[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float m = mv[r][c][e], v = vm[r][c][e];
        pn[e] = adam_one(h, acc[r][c][e], h.wd, pv[r][c][e], m, v);
        if (ob + e >= fo) continue;
        const int64_t o = d.woff[k] + (int64_t)(ob + e) * fi + i;
        G[o] = acc[r][c][e];
        P[o] = pn[e];
        mm[o] = m;
        vv[o] = v;
        pk[d.poff[k] + pack_at(ob + e, i, fi)] = to_bf16(pn[e]);
      }
      if (k > 0) {
        unsigned short* qp = pk + d.qoff[k] + pack_at(i, ob, fo);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ob + e < fo) qp[e] = to_bf16(pn[e]);
      }
    }
}

// Mean and standard deviation (divisor nm - 1) over the members' values, four
// per thread; vec: every row of S and both outputs are 16-byte aligned.
__global__ __launch_bounds__(256) void k_net_stats(int nm, int64_t n, const float* __restrict__ S,
                                                   int64_t ss, float* __restrict__ mean,
                                                   float* __restrict__ sd, int vec) {
  for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; e < n;
       e += (int64_t)gridDim.x * 1024) {
    const int c = (int)min((int64_t)4, n - e);
    auto get = [&](int q) __attribute__((always_inline)) {
      const float* p = S + q * ss + e;
      if (vec && c == 4) return *(const f32x4*)p;
      return load4(p, 0, c);
    };
    f32x4 a = {0, 0, 0, 0}, v = {0, 0, 0, 0};
    for (int q = 0; q < nm; ++q) a += get(q);
    a /= (float)nm;
    for (int q = 0; q < nm; ++q) {
      const f32x4 t = get(q) - a;
      v += t * t;
    }
    v /= (float)(nm - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = sqrtf(v[i]);
    const bool w = vec && c == 4;
    store4(mean + e, 0, c, w, a);
    store4(sd + e, 0, c, w, v);
  }
}

// The network's layout, or false when the whole-network kernels do not take it.
bool net_desc(int L, const int32_t* n, NetDesc* out) {
  if (L < 1 || L > kNetL || !n) return false;
  NetDesc d{};
  d.L = L;
  for (int k = 0; k <= L; ++k) {
    if (n[k] < 1 || n[k] > kNetWidth) return false;
    d.n[k] = n[k];
    d.kp = std::max(d.kp, up32(n[k]) + 8);
  }
  int64_t w = 0, pk = 0, a = 0, g = 0;
  for (int k = 0; k < L; ++k) {
    d.woff[k] = w;
    w += (int64_t)n[k] * n[k + 1];
    d.poff[k] = pk;
    pk += (int64_t)up16(n[k + 1]) * up32(n[k]);
    d.aoff[k] = a;
    if (k + 1 < L) a += n[k + 1];
    d.goff[k] = g;
    g += n[k + 1];
    d.apo[k] = d.apad;
    d.apad += up16(n[k]);
    d.gpo[k] = d.gpad;
    d.gpad += up16(n[k + 1]);
    d.zpo[k] = d.zpad;
    if (k + 1 < L) d.zpad += up16(n[k + 1]);
  }
  d.nfwd = pk;
  for (int k = 1; k < L; ++k) {
    d.qoff[k] = pk;
    pk += (int64_t)up16(n[k]) * up32(n[k + 1]);
  }
  d.npack = pk;
  d.nW = w;
  for (int k = 0; k < L; ++k) {
    d.boff[k] = w;
    w += n[k + 1];
  }
  d.nP = w;
  d.nhid = a;
  d.ngrad = g;
  *out = d;
  return true;
}

// Column tiles per wave for the widest layer output over wc waves.
int net_nt(const NetDesc& d, int wc, bool back) {
  int most = 0;
  for (int k = back ? 0 : 1; k <= d.L; ++k) most = std::max(most, up32(d.n[k]) / 16);
  return (most + wc - 1) / wc;
}

// The packed weights are read 16 bytes at a time.
bool packed_ok(const uint16_t* p, int64_t stride) {
  return p && (uintptr_t)p % 16 == 0 && stride % 8 == 0;
}

template <typename F>
int net_launch(F* fn, dim3 grid, dim3 block, size_t lds, hipStream_t s, void** args) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)fn,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  const hipError_t e = hipLaunchKernel((const void*)fn, grid, block, args, lds, s);
  return e == hipSuccess ? 0 : (int)e;
}

int status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

}  // namespace
}  // namespace pm

using namespace pm;

extern "C" {

int pm_mlp_gemm(void* stream, int mode, int32_t M, int32_t N, int32_t K, const float* A,
                int64_t lda_m, int64_t lda_k, const float* B, int64_t ldb_k, int64_t ldb_n,
                float* C, int64_t ldc, const float* bias, float* Z) {
  return pm_mlp_gemm_batched(stream, mode, 1, M, N, K, A, lda_m, lda_k, 0, B, ldb_k, ldb_n, 0,
                             C, ldc, 0, bias, 0, Z, 0);
}

int pm_mlp_gemm_batched(void* stream, int mode, int32_t batch, int32_t M, int32_t N, int32_t K,
                        const float* A, int64_t lda_m, int64_t lda_k, int64_t stride_a,
                        const float* B, int64_t ldb_k, int64_t ldb_n, int64_t stride_b,
                        float* C, int64_t ldc, int64_t stride_c, const float* bias,
                        int64_t stride_bias, float* Z, int64_t stride_z) {
  if (M < 0 || N < 0 || K < 0 || mode < 0 || mode > 3 || !A || !B || !C) return PM_EINVAL;
  if (batch < 1 || batch > 65535) return PM_EINVAL;
  if ((mode == PM_MLP_GELU || mode == PM_MLP_DGELU) && !Z) return PM_EINVAL;
  if (M == 0 || N == 0) return 0;
  dim3 grid((N + kBN - 1) / kBN, (M + kBM - 1) / kBM, batch);
  if (grid.y > 65535) return PM_EINVAL;
  const GemmBatch bs{stride_a, stride_b, stride_c, stride_bias, stride_z};
  hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, (hipStream_t)stream, mode, M, N, K, A,
                     lda_m, lda_k, B, ldb_k, ldb_n, C, ldc, bias, Z, bs);
  return status();
}

int pm_mlp_colsum(void* stream, int32_t M, int32_t N, const float* A, int64_t lda, float* out) {
  return pm_mlp_colsum_batched(stream, 1, M, N, A, lda, 0, out, 0);
}

int pm_mlp_colsum_batched(void* stream, int32_t batch, int32_t M, int32_t N, const float* A,
                          int64_t lda, int64_t stride_a, float* out, int64_t stride_out) {
  if (M < 0 || N < 0 || !A || !out || batch < 1 || batch > 65535) return PM_EINVAL;
  if (N == 0) return 0;
  hipLaunchKernelGGL(k_colsum, dim3((N + 63) / 64, batch), dim3(256), 0, (hipStream_t)stream,
                     M, N, A, lda, out, stride_a, stride_out);
  return status();
}

int pm_mlp_mse(void* stream, int32_t M, int32_t N, const float* Y, const float* T,
               const float* w, float* dY, float* loss) {
  return pm_mlp_mse_batched(stream, 1, M, N, Y, T, 0, w, dY, loss);
}

int pm_mlp_mse_batched(void* stream, int32_t batch, int32_t M, int32_t N, const float* Y,
                       const float* T, int64_t stride, const float* w, float* dY, float* loss) {
  if (M <= 0 || N <= 0 || !Y || !T || !dY || !loss || batch < 1 || batch > 65535)
    return PM_EINVAL;
  const int64_t total = (int64_t)M * N;
  const int blocks = (int)std::min<int64_t>((total + 255) / 256, 1024);
  hipLaunchKernelGGL(k_mse, dim3(blocks, batch), dim3(256), 0, (hipStream_t)stream, M, N, Y, T,
                     w, dY, loss, stride);
  return status();
}

int pm_mlp_adam(void* stream, int64_t n, float* p, const float* g, float* m, float* v,
                float lr, float beta1, float beta2, float eps, float weight_decay, int32_t t) {
  if (n < 0 || !p || !g || !m || !v || t < 1) return PM_EINVAL;
  if (n == 0) return 0;
  const float c1 = 1.0f - powf(beta1, (float)t);
  const float c2 = 1.0f - powf(beta2, (float)t);
  const int blocks = (int)std::min<int64_t>((n + 255) / 256, 2048);
  hipLaunchKernelGGL(k_adam, dim3(blocks), dim3(256), 0, (hipStream_t)stream, n, p, g, m, v,
                     lr, beta1, beta2, eps, weight_decay, c1, c2);
  return status();
}

int64_t pm_mlp_net_packed(int32_t layers, const int32_t* sizes, int32_t train) {
  NetDesc d;
  if (!net_desc(layers, sizes, &d)) return 0;
  return train ? d.npack : d.nfwd;
}

int64_t pm_mlp_net_work(int32_t layers, const int32_t* sizes, int32_t rows) {
  NetDesc d;
  if (!net_desc(layers, sizes, &d) || rows < 1) return 0;
  return (net_work_floats(d, up32(rows)) + 3) & ~3ll;
}

int pm_mlp_net_pack(void* stream, int32_t batch, int32_t layers, const int32_t* sizes,
                    const float* P, int64_t stride_p, uint16_t* packed, int64_t stride_packed,
                    int32_t train) {
  NetDesc d;
  if (!net_desc(layers, sizes, &d) || !P || !packed_ok(packed, stride_packed) || batch < 1 ||
      batch > 65535)
    return PM_EINVAL;
  const int blocks = (int)std::min<int64_t>((d.nW + 255) / 256, 1024);
  hipLaunchKernelGGL(k_net_pack, dim3(blocks, batch), dim3(256), 0, (hipStream_t)stream, d, P,
                     stride_p, packed, stride_packed, train);
  return status();
}

int pm_mlp_net_forward(void* stream, int32_t batch, int32_t M, int32_t layers,
                       const int32_t* sizes, const float* P, int64_t stride_p,
                       const uint16_t* packed, int64_t stride_packed, const float* X,
                       int64_t stride_x, float* Y, int64_t stride_y, float* acts, float* zs,
                       int64_t stride_a) {
  NetDesc d;
  if (!net_desc(layers, sizes, &d) || !P || !packed_ok(packed, stride_packed) || !X || !Y ||
      batch < 1 || batch > 65535 || M < 0 || (acts == nullptr) != (zs == nullptr))
    return PM_EINVAL;
  if (M == 0) return 0;
  void* args[] = {&d, &M, &P, &stride_p, &packed, &stride_packed, &X, &stride_x, &Y, &stride_y,
                  &acts, &zs, &stride_a};
  hipStream_t s = (hipStream_t)stream;
  // 128 rows per workgroup (64 when a layer is wider than 256, for the
  // registers) read the weights once for all of them; when those are too few
  // workgroups for 256 CUs, 16 rows
  const int wide = net_nt(d, 4, false) > 4 ? 64 : 128;
  const bool big = (int64_t)batch * ((M + wide - 1) / wide) >= 256;
  const int bm = big ? wide : 16;
  const dim3 grid((M + bm - 1) / bm, batch), block(512);
  const size_t lds = (size_t)bm * d.kp * sizeof(unsigned short) + d.ngrad * sizeof(float);
  if (big) {
    const int nt = net_nt(d, 4, false);
    if (nt <= 1) return net_launch(k_net_forward<4, 1, 2, 4, 4>, grid, block, lds, s, args);
    if (nt <= 2) return net_launch(k_net_forward<4, 2, 2, 4, 2>, grid, block, lds, s, args);
    if (nt <= 4) return net_launch(k_net_forward<4, 4, 2, 4, 1>, grid, block, lds, s, args);
    return net_launch(k_net_forward<2, 8, 2, 4, 1>, grid, block, lds, s, args);
  }
  const int nt = net_nt(d, 8, false);
  if (nt <= 1) return net_launch(k_net_forward<1, 1, 1, 8, 8>, grid, block, lds, s, args);
  if (nt <= 2) return net_launch(k_net_forward<1, 2, 1, 8, 8>, grid, block, lds, s, args);
  return net_launch(k_net_forward<1, 4, 1, 8, 4>, grid, block, lds, s, args);
}

int pm_mlp_net_train(void* stream, int32_t batch, int32_t layers, const int32_t* sizes, float* P,
                     float* G, float* m, float* v, int64_t stride_p, uint16_t* packed,
                     int64_t stride_packed, const float* X, const float* T, const int64_t* idx,
                     int64_t stride_idx, const float* w, int32_t rows, int32_t batch_rows,
                     float* work, const float* lr, float beta1, float beta2, float eps,
                     float weight_decay, int32_t t0, float* loss) {
  NetDesc d;
  // (work is read and written 16 bytes at a time)
  if (!net_desc(layers, sizes, &d) || !P || !G || !m || !v ||
      !packed_ok(packed, stride_packed) || !X || !T || !idx || !work ||
      (uintptr_t)work % 16 != 0 || !lr || !loss || batch < 1 || batch > 65535 || rows < 1 ||
      batch_rows < 1 || t0 < 0)
    return PM_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const size_t lds = (size_t)16 * d.kp * sizeof(unsigned short) + d.ngrad * sizeof(float);
  const int nt = net_nt(d, 8, true);
  int jobs = 0;
  for (int k = 0; k < d.L; ++k)
    jobs += ((d.n[k + 1] + 63) / 64) * ((d.n[k] + 63) / 64) + 1;
  int step = 0;
  for (int32_t i0 = 0; i0 < rows; i0 += batch_rows, ++step) {
    int B = std::min(batch_rows, rows - i0), B32 = up32(B);
    const int64_t* ix = idx + i0;
    float* ls = loss + (int64_t)step * batch;
    void* args[] = {&d, &B, &B32, &P, &stride_p, &packed, &stride_packed, &X, &T, &ix,
                    &stride_idx, &w, &work, &ls};
    const dim3 grid(B32 / 16, batch);
    int r = nt <= 1   ? net_launch(k_net_train<1, 8>, grid, dim3(512), lds, s, args)
            : nt <= 2 ? net_launch(k_net_train<2, 8>, grid, dim3(512), lds, s, args)
                      : net_launch(k_net_train<4, 4>, grid, dim3(512), lds, s, args);
    if (r) return r;
    const int32_t t = t0 + step + 1;
    const AdamArgs h{lr[step], beta1, beta2, eps, weight_decay,
                     1.0f - powf(beta1, (float)t), 1.0f - powf(beta2, (float)t)};
    hipLaunchKernelGGL(k_net_update, dim3(jobs, batch), dim3(256), 0, s, d, B32, work, P, G, m, v,
                       stride_p, packed, stride_packed, h);
    r = status();
    if (r) return r;
  }
  return 0;
}

int pm_mlp_net_stats(void* stream, int32_t members, int64_t n, const float* S, int64_t stride,
                     float* mean, float* std) {
  if (members < 1 || n < 0 || !S || !mean || !std) return PM_EINVAL;
  if (n == 0) return 0;
  const int blocks = (int)std::min<int64_t>((n + 1023) / 1024, 8192);
  const int vec = (((uintptr_t)S | (uintptr_t)mean | (uintptr_t)std) & 15) == 0 && stride % 4 == 0;
  hipLaunchKernelGGL(k_net_stats, dim3(blocks), dim3(256), 0, (hipStream_t)stream, members, n, S,
                     stride, mean, std, vec);
  return status();
}

}  // extern "C"
