// gemm.hip -- MFMA GEMMs of the projector path (NonLocalPotential::energy
// dgemm calls, src/NonLocalPotential.cpp:1411-1428, 1611, 1716) and of
// SlaterDet::gram (syrk/syr, src/SlaterDet.cpp:487-520).
//
// One kernel shape serves every product: D[p][q] = sum_r P(r,p) Q(r,q) on a
// (32 BI) x (32 BJ) tile per block of 256 threads: 2x2 waves, each a BI x BJ
// grid of 16x16 MFMA blocks.  P is read along r (P(r,p) = P[r + p*ldp]); Q
// along r (TN form, Q[r + q*ldq]) or along q (NN form, Q[q + r*ldq]).  q is
// the contiguous index of the output, so the 16 lanes of an MFMA column group
// store 16 consecutive elements.  The compute type is FP64
// (v_mfma_f64_16x16x4f64) or FP32 (v_mfma_f32_16x16x4f32); operands are
// converted while they are staged.
//
// What bounds it: the FP64 MFMA (64 cycles each; the loop without its loads,
// stores and barriers runs at 74 TFLOP/s), and what stands between the products of two
// chunks.  So that has to be short:
//   - the reduction is staged in chunks of KC through two LDS stages with one
//     barrier per chunk; the loads of the chunk after next are in registers
//     meanwhile, and two blocks share a CU;
//   - operands contiguous along r keep r contiguous in LDS and the MFMA step t
//     of a chunk multiplies the elements r = 4 (lane/16) + t, so a lane's
//     operands of two (FP64) or four (FP32) steps are one 16-byte LDS read, and
//     the 16-byte global loads go to LDS unchanged (transposing stores had
//     8-way bank conflicts here);
//   - rows past the edge are loaded from the last row (their products are not
//     stored), so only the last chunk and the last q tile test anything.
// 512 bands x 1024 projectors x 461336 in FP64: TN 11.8 -> 8.4 ms (58 TFLOP/s),
// NN 10.2 -> 7.9 ms (61 TFLOP/s).  Tried and slower or equal: a barrier in the middle of a
// chunk with the next operands in registers (spills), wave priorities.  The tile
// follows the extents (pick below): the projections of 8 atoms on 16 bands (K = 11364)
// take 9 us where a 128 x 128 tile took 95.  Tiles of 96 win nothing at that size
// (512 x 512 x 109 k: 2.87 ms with and without) and 2 to 6 % of the three products
// where 64 and 128 leave the last tile nearly empty: 90 bands x 288 projectors x 63 k
// 0.294 -> 0.281 ms in FP64, 0.174 -> 0.165 in FP32, 131 x 300 x 109 k 0.427 -> 0.410 in FP32.
//
// MFMA lane layouts on a 64-wide wave (16x16x4): lane l holds A[l%16][l/16]
// and B[l/16][l%16]; accumulator e of lane l is D[4e + l/16][l%16] for f64
// and D[4(l/16) + e][l%16] for f32.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "energy.h"
#include "qbg.h"

namespace qbg {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename TC>
struct Mfma;
template <>
struct Mfma<double> {
  typedef v4d acc;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int e, int lane) { return 4 * e + (lane >> 4); }
};
template <>
struct Mfma<float> {
  typedef v4f acc;
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int e, int lane) { return 4 * (lane >> 4) + e; }
};

// two adjacent elements, at the alignment of one: the callers' arrays promise no more
template <typename T>
struct Pair2;
template <>
struct Pair2<double> {
  typedef double v __attribute__((ext_vector_type(2), aligned(8)));
};
template <>
struct Pair2<float> {
  typedef float v __attribute__((ext_vector_type(2), aligned(4)));
};

constexpr int KC = 16;        // reduction chunk
// LDS row of an operand with r contiguous: KC elements and 16 bytes, so that
// eight rows' 16-byte reads fall on distinct banks
template <typename TC>
constexpr int RS = KC + 16 / (int)sizeof(TC);
constexpr int QPAD = 4;       // row padding of the NN operand (q contiguous)

struct GemmArgs {
  const void* P;
  long ldp;
  const void* Q;
  long ldq;
  int np, nq;       // output extent
  long nr;          // reduction extent
  long rper;        // reduction length of one split (multiple of KC)
  int tp, tq;       // tiles along p and q
  int pfast;        // block order: p tiles fastest (1) or q tiles fastest (0)
  void* out;        // out[split*sstride + q + p*ldo]
  long ldo, sstride;
  int accumulate;
  int tri;          // 1: only tiles with q >= p (symmetric product);
                    // 2: P(r,p) = 0 for r > p (reduction stops at the tile's last p)
  const int* skip;  // if set and *skip != 0 the launch does nothing (a step of
                    // a captured iteration that has already converged)
  int nblk;         // tiles x splits; the grid is that rounded up to 8
};

template <typename TPm, typename TQm, typename TC, bool QR, typename TO, int BI, int BJ>
__global__ __launch_bounds__(256, 2) void k_gemm(GemmArgs g) {
  typedef Mfma<TC> MF;
  constexpr int TP = 32 * BI, TQ = 32 * BJ, R = RS<TC>;
  // a lane's elements of one 16-byte LDS read
  constexpr int NV = 16 / (int)sizeof(TC);
  typedef TC vlds __attribute__((ext_vector_type(NV)));
  typedef TC vst __attribute__((ext_vector_type(2)));
  __shared__ __align__(16) TC Ps[2][TP * R];
  __shared__ __align__(16) TC Qs[2][QR ? TQ * R : KC * (TQ + QPAD)];
  if (g.skip && *g.skip) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  // blocks are dealt to the 8 XCDs round robin: renumber so that runs of
  // consecutive tiles (which share operand panels) stay on one XCD's L2; the
  // grid is nblk rounded up to a multiple of 8, the blocks past nblk return
  const int b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (b >= g.nblk) return;
  // tri == 1 (symmetric, tp == tq): only the tiles q >= p, row by row
  const int ntile = g.tri == 1 ? g.tp * (g.tp + 1) / 2 : g.tp * g.tq;
  const int split = b / ntile, tt = b - split * ntile;
  int ip, iq;
  if (g.tri == 1) {
    int r = tt;
    ip = 0;
    while (r >= g.tp - ip) { r -= g.tp - ip; ip++; }
    iq = ip + r;
  } else if (g.pfast) { ip = tt % g.tp; iq = tt / g.tp; }
  else { iq = tt % g.tq; ip = tt / g.tq; }
  const int p0 = ip * TP, q0 = iq * TQ;
  const long rb = (long)split * g.rper;
  long re = min(g.nr, rb + g.rper);
  if (g.tri == 2) re = min(re, (long)p0 + TP);
  typedef typename Pair2<TPm>::v vp;
  typedef typename Pair2<TQm>::v vq;
  // this thread's rows of the operands read along r: elements sr, sr + 1 of
  // the chunk, rows srow + 32 j
  const int sr = 2 * (tid & 7), srow = tid >> 3;
  const TPm* pp[BI];
#pragma unroll
  for (int j = 0; j < BI; j++)
    pp[j] = (const TPm*)g.P + (long)min(p0 + srow + 32 * j, g.np - 1) * g.ldp + sr;
  // the NN operand: elements nq0, nq0 + 1 of rows nr0 + (16 / BJ) j
  const int nq0 = 2 * (tid % (16 * BJ)), nr0 = tid / (16 * BJ);
  const bool qedge = !QR && q0 + TQ > g.nq;
  const TQm* qp[BJ];
#pragma unroll
  for (int j = 0; j < BJ; j++)
    qp[j] = QR ? (const TQm*)g.Q + (long)min(q0 + srow + 32 * j, g.nq - 1) * g.ldq + sr
               : (const TQm*)g.Q + q0 + nq0 + (long)(nr0 + (16 / BJ) * j) * g.ldq;
  vp pv[BI];
  vq qv[BJ];
  auto load = [&](long r0) {
    const bool full = r0 + KC <= re;
    if (full) {
#pragma unroll
      for (int j = 0; j < BI; j++) pv[j] = *(const vp*)(pp[j] + r0);
    } else {
#pragma unroll
      for (int j = 0; j < BI; j++) {
        pv[j].x = r0 + sr < re ? pp[j][r0] : TPm(0);
        pv[j].y = r0 + sr + 1 < re ? pp[j][r0 + 1] : TPm(0);
      }
    }
    if (QR) {
      if (full) {
#pragma unroll
        for (int j = 0; j < BJ; j++) qv[j] = *(const vq*)(qp[j] + r0);
      } else {
#pragma unroll
        for (int j = 0; j < BJ; j++) {
          qv[j].x = r0 + sr < re ? qp[j][r0] : TQm(0);
          qv[j].y = r0 + sr + 1 < re ? qp[j][r0 + 1] : TQm(0);
        }
      }
    } else {
      if (full && !qedge) {
#pragma unroll
        for (int j = 0; j < BJ; j++) qv[j] = *(const vq*)(qp[j] + r0 * g.ldq);
      } else {
#pragma unroll
        for (int j = 0; j < BJ; j++) {
          const bool ok = r0 + nr0 + (16 / BJ) * j < re;
          qv[j].x = ok && q0 + nq0 < g.nq ? qp[j][r0 * g.ldq] : TQm(0);
          qv[j].y = ok && q0 + nq0 + 1 < g.nq ? qp[j][r0 * g.ldq + 1] : TQm(0);
        }
      }
    }
  };
  auto store = [&](int st) {
#pragma unroll
    for (int j = 0; j < BI; j++)
      *(vst*)&Ps[st][(srow + 32 * j) * R + sr] = vst{(TC)pv[j].x, (TC)pv[j].y};
#pragma unroll
    for (int j = 0; j < BJ; j++)
      *(vst*)&Qs[st][QR ? (srow + 32 * j) * R + sr
                        : (nr0 + (16 / BJ) * j) * (TQ + QPAD) + nq0] =
          vst{(TC)qv[j].x, (TC)qv[j].y};
  };
  const int wp = (w & 1) * 16 * BI, wq = (w >> 1) * 16 * BJ;
  const int c = lane & 15, g4 = 4 * (lane >> 4);
  typename MF::acc acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; i++)
#pragma unroll
    for (int j = 0; j < BJ; j++) acc[i][j] = typename MF::acc{0, 0, 0, 0};
  if (rb < re) {
    load(rb);
    store(0);
    if (rb + KC < re) load(rb + KC);
  }
  __syncthreads();
  int st = 0;
  for (long r0 = rb; r0 < re; r0 += KC, st ^= 1) {
#pragma unroll
    for (int h = 0; h < 4; h += NV) {
      vlds a[BI], bq[BJ];
#pragma unroll
      for (int i = 0; i < BI; i++)
        a[i] = *(const vlds*)&Ps[st][(wp + 16 * i + c) * R + g4 + h];
#pragma unroll
      for (int j = 0; j < BJ; j++) {
        if (QR) {
          bq[j] = *(const vlds*)&Qs[st][(wq + 16 * j + c) * R + g4 + h];
        } else {
#pragma unroll
          for (int t = 0; t < NV; t++)
            bq[j][t] = Qs[st][(g4 + h + t) * (TQ + QPAD) + wq + 16 * j + c];
        }
      }
#pragma unroll
      for (int t = 0; t < NV; t++)
#pragma unroll
        for (int i = 0; i < BI; i++)
#pragma unroll
          for (int j = 0; j < BJ; j++) acc[i][j] = MF::mma(a[i][t], bq[j][t], acc[i][j]);
    }
    if (r0 + KC < re) {
      store(st ^ 1);                       // last read one barrier ago
      if (r0 + 2 * KC < re) load(r0 + 2 * KC);
    }
    __syncthreads();
  }
  TO* o = (TO*)g.out + (long)split * g.sstride;
#pragma unroll
  for (int i = 0; i < BI; i++)
#pragma unroll
    for (int j = 0; j < BJ; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int p = p0 + wp + 16 * i + MF::row(e, lane);
        const int q = q0 + wq + 16 * j + c;
        if (p < g.np && q < g.nq) {
          TO* d = o + q + (long)p * g.ldo;
          const TO v = (TO)acc[i][j][e];
          *d = g.accumulate ? (TO)(*d + v) : v;
        }
      }
}

// out[q + p*ldo] = alpha * sum_s partial[s][p][q] + gamma * Q[q*ldq] * P[p*ldp]
// + delta (p = q) + beta * out; if T: T (as out) = I + 3/4 out, and the sum of
// the squares of a block's outputs to part.  A block sums 64 outputs: wave y takes the splits y, y + 4, ... (eight loads
// in flight), and the four sums are added in that order.
template <typename TQm, typename TPm>
__global__ __launch_bounds__(256) void k_split_reduce(const double* __restrict__ partial, int S,
                                                      int nq, int np, double alpha, double gamma,
                                                      const TQm* __restrict__ Q, long ldq,
                                                      const TPm* __restrict__ P, long ldp,
                                                      double* __restrict__ out, long ldo,
                                                      int sym, const int* __restrict__ skip,
                                                      SplitEnd end) {
  if (skip && *skip) return;
  __shared__ double sums[4][64];
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const long t = (long)blockIdx.x * 64 + x, tot = (long)nq * np;
  const int q = (int)(t % nq), p = (int)(t / nq);
  // symmetric products hold only q >= p: the upper part mirrors it
  const long src = (sym && q < p) ? (long)q * nq + p : t;
  double s = 0.0;
  if (t < tot) {
#pragma unroll 8
    for (int k = y; k < S; k += 4) s += partial[(long)k * tot + src];
  }
  sums[y][x] = s;
  __syncthreads();
  if (y) return;
  double v = 0.0;
  if (t < tot) {
    v = alpha * ((sums[0][x] + sums[1][x]) + (sums[2][x] + sums[3][x]));
    if (gamma != 0.0) v += gamma * (double)Q[(long)q * ldq] * (double)P[(long)p * ldp];
    if (p == q) v += end.delta;
    double* o = out + q + (long)p * ldo;
    if (end.beta != 0.0) v += end.beta * *o;
    *o = v;
    if (end.T) end.T[q + (long)p * ldo] = (p == q ? 1.0 : 0.0) + 0.75 * v;
  }
  if (end.T) {
    double r = v * v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) r += __shfl_down(r, off, 64);
    if (x == 0) end.part[blockIdx.x] = r;
  }
}

namespace {

// compute units of the current device, cached per device
int cu_count() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cache[dev]) {
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      ncu = 256;
    cache[dev] = std::max(1, ncu);
  }
  return cache[dev];
}

// Tile (32 bi x 32 bj) and reduction splits of one product.
struct Pick {
  int bi, bj;
  long S;
};

// cycles of a chunk's barrier and LDS latency that no MFMA covers: with one
// block on a CU, and with two
constexpr double CHUNK_ALONE = 700, CHUNK_SHARED = 200;
constexpr double REDUCE_BYTES = 2000;    // bytes a cycle of the partials' store and sum

// The pick with the fewest cycles of the busiest CU: (blocks per CU) x
// (chunks) x (MFMA cycles of a wave's bi x bj blocks, 64 each in FP64, 32 in
// FP32, and the chunk's fixed cost) + the traffic of the split partials.  It
// makes the tiles follow ragged extents (131 bands: two 96-row tiles), and
// small outputs use small tiles and many splits.  minS, maxS: the fewest and the
// most splits (1, 1: none); bjs: bit j allows bj = j; fixed bi, or 0; sym: square tiles,
// upper ones only.
Pick pick(int np, int nq, long nr, long minS, long maxS, unsigned bjs, int bi_fixed, bool sym,
          int prec) {
  const double cus = cu_count(), mf = prec == QBG_PREC_FP64 ? 256 : 128;
  const long chunks = (nr + KC - 1) / KC;
  Pick best{4, 4, 1};
  double bt = 1e300;
  for (int bi = 1; bi <= 4; bi++) {
    if (bi_fixed && bi != bi_fixed) continue;
    const long tp = (np + 32 * bi - 1) / (32 * bi);
    for (int bj = 1; bj <= 4; bj++) {
      if (!(bjs >> bj & 1) || (sym && bj != bi)) continue;
      const long tq = (nq + 32 * bj - 1) / (32 * bj);
      const long tiles = sym ? tp * (tp + 1) / 2 : tp * tq;
      for (int k = 1; k <= 8; k++) {
        long S = std::max<long>(minS, (long)(k * cus) / tiles);
        S = std::min(S, std::min(maxS, std::max<long>(1, chunks / 2)));
        const double blocks = (double)tiles * S;
        const double rounds = blocks < 16 * cus ? (double)(((long)blocks + (long)cus - 1) /
                                                           (long)cus)
                                                : blocks / cus;
        const double chunk = bi * bj * mf + (rounds < 2 ? CHUNK_ALONE : CHUNK_SHARED);
        double t = rounds * (double)((chunks + S - 1) / S) * chunk;
        if (maxS > 1) t += (double)S * np * nq * 16.0 / REDUCE_BYTES;
        if (t < bt) {
          bt = t;
          best = {bi, bj, S};
        }
        if (maxS <= 1) break;
      }
    }
  }
  return best;
}

// The fewest splits of an FP32 product.  A split is one chain of FP32 sums
// (the splits are added in FP64), whose rounding error grows as the square root
// of its length, and the cycles alone would halve the splits where two blocks share
// a CU anyway: 512 bands x 1024 projectors x 461 k in 16 splits leave the nonlocal H psi
// off by 2.84e-6, in 32 by 1.95e-6, in the same time (31.8 and 31.7 ms an evaluation).
// So a chain holds at most 1/32 of the reduction; where the output has more than 32
// tiles of 128 x 128, of which 1024 blocks are enough, 1/(1024 / tiles); and 64 terms are
// short enough for any.
long fp32_splits(int np, int nq, long nr) {
  const long tiles = (long)((np + 127) / 128) * ((nq + 127) / 128), chunks = (nr + KC - 1) / KC;
  return std::max<long>(1, std::min(std::min<long>(32, (1024 + tiles - 1) / tiles), chunks / 4));
}

template <typename TPm, typename TQm, typename TC, bool QR, typename TO, int BI, int BJ>
void launch_tile(GemmArgs g, hipStream_t s) {
  g.tp = (g.np + 32 * BI - 1) / (32 * BI);
  g.tq = (g.nq + 32 * BJ - 1) / (32 * BJ);
  const int ntile = g.tri == 1 ? g.tp * (g.tp + 1) / 2 : g.tp * g.tq;
  g.nblk = ntile * (int)((g.nr + g.rper - 1) / g.rper);
  const unsigned grid = (unsigned)((g.nblk + 7) & ~7);
  hipLaunchKernelGGL((k_gemm<TPm, TQm, TC, QR, TO, BI, BJ>), dim3(grid), dim3(256), 0, s, g);
}

template <typename TPm, typename TQm, typename TC, bool QR, typename TO>
void launch_gemm(const GemmArgs& g, Pick k, hipStream_t s) {
#define QBG_TILE(I, J) \
  if (k.bi == I && k.bj == J) return launch_tile<TPm, TQm, TC, QR, TO, I, J>(g, s);
#define QBG_TILES(I) QBG_TILE(I, 1) QBG_TILE(I, 2) QBG_TILE(I, 4)
  QBG_TILES(1) QBG_TILES(2) QBG_TILES(3) QBG_TILES(4)
  if constexpr (QR) { QBG_TILE(1, 3) QBG_TILE(2, 3) QBG_TILE(3, 3) QBG_TILE(4, 3) }
#undef QBG_TILES
#undef QBG_TILE
}
constexpr unsigned BJ_TN = 0x1e, BJ_NN = 0x16;   // compiled bj of the two forms

// split-K TN product; partials in FP64, reduced in a fixed order.  sym: the
// product is symmetric (A = B, M = N): only the lower tiles are formed.
template <typename TQm>
int tn_splitk(const TQm* A, long lda, const double* B, long ldb, int M, int N, long K,
              double alpha, double gamma, double* out, long ldo, double* work,
              size_t work_doubles, int prec, int sym, hipStream_t s, const int* skip,
              const SplitEnd& end = {}) {
  if (M <= 0 || N <= 0 || K <= 0) return -1;
  if ((size_t)M * N > work_doubles || (sizeof(TQm) == 4 && prec == QBG_PREC_FP64)) return -1;
  GemmArgs g{};
  g.skip = skip;
  g.P = B; g.ldp = ldb; g.Q = A; g.ldq = lda;
  g.np = N; g.nq = M; g.nr = K;
  g.pfast = 0;
  g.tri = sym ? 1 : 0;
  const long minS = prec == QBG_PREC_FP64 ? 1 : fp32_splits(N, M, K);
  const Pick k = pick(N, M, K, minS, (long)(work_doubles / ((size_t)M * N)), BJ_TN, 0, sym != 0,
                      prec);
  const long chunks = (K + KC - 1) / KC;
  g.rper = ((chunks + k.S - 1) / k.S) * KC;
  const long S = (K + g.rper - 1) / g.rper;
  g.out = work; g.ldo = M; g.sstride = (long)M * N; g.accumulate = 0;
  // FP32 operands come with FP32 products only
  if constexpr (sizeof(TQm) == 8) {
    if (prec == QBG_PREC_FP64) launch_gemm<double, TQm, double, true, double>(g, k, s);
  }
  if (prec != QBG_PREC_FP64) launch_gemm<double, TQm, float, true, double>(g, k, s);
  const long tot = (long)M * N;
  hipLaunchKernelGGL((k_split_reduce<TQm, double>), dim3((unsigned)((tot + 63) / 64)),
                     dim3(256), 0, s, work, (int)S, M, N, alpha, gamma, A, lda, B, ldb, out, ldo,
                     sym, skip, end);
  return 0;
}

// one_p: a single p tile holds all N columns (N <= gemm_nn_tile_p()), so that
// the block that read a row of A is the only one that writes it
template <typename TQm, typename TO>
void nn(const TQm* A, long lda, const double* F, long ldf, long K, int N, int M, TO* C, long ldc,
        int accumulate, int prec, int tri, int one_p, hipStream_t s, const int* skip) {
  if (K <= 0 || N <= 0 || M <= 0) return;
  GemmArgs g{};
  g.skip = skip;
  g.P = F; g.ldp = ldf; g.Q = A; g.ldq = lda;
  g.np = N; g.nq = (int)K; g.nr = M;
  g.pfast = 1;
  g.tri = tri ? 2 : 0;
  g.rper = ((M + KC - 1) / KC) * KC;
  g.out = C; g.ldo = ldc; g.sstride = 0; g.accumulate = accumulate;
  const Pick k = pick(N, (int)K, M, 1, 1, BJ_NN, one_p ? (N + 31) / 32 : 0, false, prec);
  if constexpr (sizeof(TQm) == 8 && sizeof(TO) == 8) {
    if (prec == QBG_PREC_FP64) launch_gemm<double, TQm, double, false, TO>(g, k, s);
  }
  if (prec != QBG_PREC_FP64) launch_gemm<double, TQm, float, false, TO>(g, k, s);
}

}  // namespace

// NN with the reduction (M) split over blocks, partials in work, for products
// whose output has too few tiles to fill the device:
// C[k + n*ldc] = sum_m A[k + m*lda] F[m + n*ldf]
int gemm_nn_splitk(const double* A, long lda, const double* F, long ldf, long K, int N, int M,
                   double* C, long ldc, double* work, size_t work_doubles, hipStream_t s,
                   const int* skip, double alpha, const SplitEnd& end) {
  if (K <= 0 || N <= 0 || M <= 0) return -1;
  if ((size_t)K * N > work_doubles) return -1;
  GemmArgs g{};
  g.skip = skip;
  g.P = F; g.ldp = ldf; g.Q = A; g.ldq = lda;
  g.np = N; g.nq = (int)K; g.nr = M;
  g.pfast = 1;
  g.tri = 0;
  const long chunks = (M + KC - 1) / KC;
  const Pick k = pick(N, (int)K, M, 1, (long)(work_doubles / ((size_t)K * N)), BJ_NN, 0, false,
                      QBG_PREC_FP64);
  g.rper = ((chunks + k.S - 1) / k.S) * KC;
  const long S = (M + g.rper - 1) / g.rper;
  g.out = work; g.ldo = K; g.sstride = K * N; g.accumulate = 0;
  launch_gemm<double, double, double, false, double>(g, k, s);
  const long tot = K * N;
  hipLaunchKernelGGL((k_split_reduce<double, double>), dim3((unsigned)((tot + 63) / 64)),
                     dim3(256), 0, s, work, (int)S, (int)K, N, alpha, 0.0, A, lda, F, ldf, C, ldc,
                     0, skip, end);
  return 0;
}
int gemm_tn_splitk(const double* A, long lda, const double* B, long ldb, int M, int N, long K,
                   double alpha, double gamma, double* out, long ldo, double* work,
                   size_t work_doubles, int prec, hipStream_t s, const int* skip) {
  return tn_splitk(A, lda, B, ldb, M, N, K, alpha, gamma, out, ldo, work, work_doubles, prec, 0,
                   s, skip);
}
int gemm_tn_splitk(const float* A, long lda, const double* B, long ldb, int M, int N, long K,
                   double alpha, double gamma, double* out, long ldo, double* work,
                   size_t work_doubles, int prec, hipStream_t s) {
  return tn_splitk(A, lda, B, ldb, M, N, K, alpha, gamma, out, ldo, work, work_doubles, prec, 0,
                   s, nullptr);
}
int gemm_syrk(const double* A, long lda, int N, long K, double alpha, double gamma, double* out,
              long ldo, double* work, size_t work_doubles, hipStream_t s, const int* skip,
              const SplitEnd& end) {
  return tn_splitk(A, lda, A, lda, N, N, K, alpha, gamma, out, ldo, work, work_doubles,
                   QBG_PREC_FP64, 1, s, skip, end);
}
int split_blocks(long outputs) { return (int)((outputs + 63) / 64); }
int gemm_nn_tile_p() { return 128; }
void gemm_nn_triu(const double* A, long lda, const double* F, long ldf, long K, int N, double* C,
                  long ldc, hipStream_t s) {
  nn(A, lda, F, ldf, K, N, N, C, ldc, 0, QBG_PREC_FP64, 1, 0, s, nullptr);
}
void gemm_nn_inplace(const double* A, long lda, const double* F, long ldf, long K, int N, int M,
                     double* C, long ldc, hipStream_t s) {
  nn(A, lda, F, ldf, K, N, M, C, ldc, 0, QBG_PREC_FP64, 0, 1, s, nullptr);
}
void gemm_nn(const double* A, long lda, const double* F, long ldf, long K, int N, int M,
             double* C, long ldc, int accumulate, int prec, hipStream_t s, const int* skip) {
  nn(A, lda, F, ldf, K, N, M, C, ldc, accumulate, prec, 0, 0, s, skip);
}
void gemm_nn(const float* A, long lda, const double* F, long ldf, long K, int N, int M,
             double* C, long ldc, int accumulate, int prec, hipStream_t s) {
  nn(A, lda, F, ldf, K, N, M, C, ldc, accumulate, prec, 0, 0, s, nullptr);
}
void gemm_nn(const double* A, long lda, const double* F, long ldf, long K, int N, int M,
             float* C, long ldc, int accumulate, int prec, hipStream_t s) {
  nn(A, lda, F, ldf, K, N, M, C, ldc, accumulate, prec, 0, 0, s, nullptr);
}

// zero Im c(G=0) of every band (SlaterDet::cleanup, src/SlaterDet.cpp:1335-1356)
__global__ void k_cleanup(double* c, long ldc, int nst) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n < nst) c[2 * ldc * n + 1] = 0.0;
}
void cleanup(double* c, long ldc, int nst, hipStream_t s) {
  hipLaunchKernelGGL(k_cleanup, dim3((nst + 255) / 256), dim3(256), 0, s, c, ldc, nst);
}

}  // namespace qbg
