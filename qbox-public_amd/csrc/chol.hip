// chol.hip -- the small dense steps of the orthogonalizations: Cholesky with
// the inverse factor (potrf + trtri of SlaterDet::gram and ortho_align,
// src/SlaterDet.cpp:487-520, 768-876) and DoubleMatrix::polar of a matrix that
// one work-group can hold (src/Matrix.cpp:2446-2517).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "energy.h"
#include "qbg.h"
#include "scf.h"

namespace qbg {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

constexpr int CB = CHOL_PANEL;    // columns of a panel, and rows of a block of it
constexpr int CS = 16;            // columns factored between two MFMA updates
// LDS row of a panel: 66 doubles put the 16 rows x 2 columns that half a wave
// reads for an MFMA operand on distinct banks, and keep rows 16-byte aligned
constexpr int CLD = CB + 2;
constexpr int CHOL_LDS = 2 * CB * CLD;

__device__ __forceinline__ double lane_value(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// Rows 0..63 of A: a 64 x 64 diagonal block D (lower part used, identity past
// the matrix), rows 64..127: rows R below it.  D <- its Cholesky factor L, R <- R L^-T.
// Returns 0, or the first pivot that is not positive, plus 1 (the same value
// in every thread).  16 columns at a time: one wave holds them in registers, a
// row of each half per lane, and broadcasts pivots and multipliers by lane
// reads; the columns right of them are updated by MFMA from LDS by all NT / 64 waves.
template <int NT>
__device__ __forceinline__ int chol_rows(double* A, int* bad) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  if (tid == 0) *bad = 0;
  __syncthreads();
  for (int p = 0; p < CB / CS; p++) {
    if (w == 0) {
      double a[CS], b[CS];
      v2d* ra = (v2d*)&A[lane * CLD + CS * p];
      v2d* rb = (v2d*)&A[(CB + lane) * CLD + CS * p];
#pragma unroll
      for (int t = 0; t < CS / 2; t++) {
        const v2d x = ra[t], y = rb[t];
        a[2 * t] = x.x; a[2 * t + 1] = x.y;
        b[2 * t] = y.x; b[2 * t + 1] = y.y;
      }
      int fail = 0;
#pragma unroll
      for (int c = 0; c < CS; c++) {
        const double d = lane_value(a[c], CS * p + c);
        if (!(d > 0.0) && !fail) fail = CS * p + c + 1;
        const double rs = rsqrt(d);
        a[c] *= rs;
        b[c] *= rs;
#pragma unroll
        for (int k = c + 1; k < CS; k++) {
          const double l = lane_value(a[c], CS * p + k);
          a[k] -= a[c] * l;
          b[k] -= b[c] * l;
        }
      }
#pragma unroll
      for (int t = 0; t < CS / 2; t++) {
        ra[t] = v2d{a[2 * t], a[2 * t + 1]};
        rb[t] = v2d{b[2 * t], b[2 * t + 1]};
      }
      if (lane == 0 && fail) *bad = fail;
    }
    __syncthreads();
    if (*bad) return *bad;
    // columns 16 (p + 1) .. 63: A(r, k) -= sum_t A(r, t) D(k, t) over the 16
    const int nct = CB / CS - 1 - p;
    for (int e = w; e < 8 * nct; e += NT / 64) {
      const int rt = e & 7, ct = p + 1 + (e >> 3);
      if (rt < ct) continue;                 // above D's diagonal
      v4d acc;
#pragma unroll
      for (int i = 0; i < 4; i++) acc[i] = A[(16 * rt + 4 * i + lk) * CLD + 16 * ct + li];
#pragma unroll
      for (int t = 0; t < 4; t++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-A[(16 * rt + li) * CLD + CS * p + 4 * t + lk],
                                                   A[(16 * ct + li) * CLD + CS * p + 4 * t + lk],
                                                   acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) A[(16 * rt + 4 * i + lk) * CLD + 16 * ct + li] = acc[i];
    }
    __syncthreads();
  }
  return 0;
}

// One block of 64 rows of a panel of the stacked matrix [S; X] (2n rows, see
// chol_inverse): load the diagonal block at j0 and the rows j1 + 64 blk ...
// below it, factor, store the rows and, of S's rows, the negated transpose
// lt[c + 64 i].  Returns chol_rows' status.
template <int NT>
__device__ __forceinline__ int chol_panel(double* SX, int n, int j0, int jb, int blk, double* lt,
                                          double* A, int* bad) {
  const long ld = 2L * n;
  const int j1 = j0 + jb, i0 = CB * blk;
  // a thread holds one row: all of its loads are in flight together, from
  // clamped addresses so that none depends on a branch
  constexpr int NL = 2 * CB * CB / NT, CSTEP = NT / (2 * CB);
  {
    const int r = threadIdx.x & (2 * CB - 1), c0 = threadIdx.x / (2 * CB);
    const bool diag = r < CB;
    const bool in = diag ? r < jb : i0 + r - CB < n;
    const double* src = SX + (in ? (diag ? j0 + r : j1 + i0 + r - CB) : j0) + j0 * ld;
    double v[NL];
#pragma unroll
    for (int t = 0; t < NL; t++) v[t] = src[min(c0 + CSTEP * t, jb - 1) * ld];
#pragma unroll
    for (int t = 0; t < NL; t++) {
      const int c = c0 + CSTEP * t;
      A[r * CLD + c] = in && c < jb ? v[t] : (diag && r == c ? 1.0 : 0.0);
    }
  }
  const int st = chol_rows<NT>(A, bad);      // begins with a barrier
  if (st) return st;
  for (int e = threadIdx.x; e < CB * CB; e += NT) {
    const int r = e & (CB - 1), c = e >> 6, i = i0 + r;
    if (i < n && c < jb) SX[(j1 + i) + (j0 + c) * ld] = A[(CB + r) * CLD + c];
  }
  for (int e = threadIdx.x; e < CB * CB; e += NT) {
    const int c = e & (CB - 1), r = e >> 6, i = i0 + r;
    if (j1 + i < n && c < jb) lt[c + (long)i * CB] = -A[(CB + r) * CLD + c];
  }
  return 0;
}

}  // namespace

// X = I, S = I - q if q (ld n), and info = 0, or -1 when *skip (every later
// launch of the factorization then does nothing)
__global__ __launch_bounds__(256) void k_chol_init(double* __restrict__ SX, int n,
                                                   const double* __restrict__ q,
                                                   int* __restrict__ info,
                                                   const int* __restrict__ skip) {
  const bool off = skip && *skip;
  if (blockIdx.x == 0 && threadIdx.x == 0) *info = off ? -1 : 0;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (off || e >= (long)n * n) return;
  const long c = e / n, r = e - c * n;
  const double one = r == c ? 1.0 : 0.0;
  SX[n + r + c * 2 * n] = one;
  if (q) SX[r + c * 2 * n] = one - q[e];
}

// The serial chain of 64 pivots (square root, division and the updates of a
// lane's 16 columns) bounds it, not bytes or operations: every block
// factors the diagonal block again, which costs no time and saves a launch.
// 64 columns: 80 us for the diagonal block and 45 us for the rows below it before
// (a barrier or an LDS chain at every column), 18 to 23 us here, of which 14 us are
// the pivots (520 cycles each).
constexpr int CNT = 512;
__global__ __launch_bounds__(CNT) void k_chol_panel(double* SX, int n, int j0, int jb, int* info,
                                                    double* lt) {
  __shared__ __align__(16) double A[CHOL_LDS];
  __shared__ int bad, done;
  if (threadIdx.x == 0) done = *info;
  __syncthreads();
  if (done) return;
  const int st = chol_panel<CNT>(SX, n, j0, jb, blockIdx.x, lt, A, &bad);
  if (st && blockIdx.x == 0 && threadIdx.x == 0) *info = j0 + st;
}

// Right-looking Cholesky of S in panels of 64 columns, carried out on the
// stacked matrix [S; I]: the rows below S become L^-T, so the inverse needs no
// launches of its own.  The rows of a panel that are not
// zero, S's below it and X's to its end, are always n contiguous rows of the
// stack, and so are those that the trailing product updates.
// Per 64 columns one panel kernel and one product: 512 bands 1.8 -> 0.2 ms,
// 90 bands 224 -> 41 us with S factored first and inverted after it.
void chol_inverse(double* SX, int n, const double* q, int* info, double* ws, hipStream_t s,
                  const int* skip) {
  const long ld = 2L * n;
  hipLaunchKernelGGL(k_chol_init, dim3((unsigned)(((long)n * n + 255) / 256)), dim3(256), 0, s, SX,
                     n, q, info, skip);
  for (int j0 = 0; j0 < n; j0 += CB) {
    const int jb = std::min(CB, n - j0), j1 = j0 + jb;
    hipLaunchKernelGGL(k_chol_panel, dim3((n + CB - 1) / CB), dim3(CNT), 0, s, SX, n, j0, jb, info,
                       ws);
    if (j1 < n)
      gemm_nn(SX + j1 + j0 * ld, ld, ws, CB, n, n - j1, jb, SX + j1 + j1 * ld, ld, 1,
              QBG_PREC_FP64, s, info);
  }
}

// ------------------------------------------------------------------ polar
namespace {

constexpr int PNT = 512, PNW = PNT / 64;
constexpr int PLD = POLAR_ONE + 2;     // see CLD: (np + 2) / 2 is odd for every np
constexpr int PTILES = (POLAR_ONE / 16) * (POLAR_ONE / 16) / PNW;            // of a wave
constexpr int PSYM = ((POLAR_ONE / 16) * (POLAR_ONE / 16 + 1) / 2 + PNW - 1) / PNW;
static_assert(POLAR_ONE * PLD >= CHOL_LDS, "a panel overlays the matrix");

// tile u of the upper triangle (ti <= tj) of nt x nt tiles, row by row
__device__ __forceinline__ void sym_tile(int u, int nt, int& ti, int& tj) {
  ti = 0;
  while (u >= nt - ti) { u -= nt - ti; ti++; }
  tj = ti + u;
}

// this wave's tiles ti <= tj of the symmetric product sum_k M(k, i) M(k, j), M(k, i) =
// M[i (np + 2) + k].  MFMA step t of a chunk of 16 takes k = 4 (lane / 16) + t,
// so that a lane's operands of two steps are one 16-byte read.
__device__ __forceinline__ void sym_product(const double* M, int np, v4d (&acc)[PSYM]) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = 4 * (lane >> 4);
  const int nt = np / 16, ld = np + 2;
#pragma unroll
  for (int s = 0; s < PSYM; s++) {
    acc[s] = v4d{0, 0, 0, 0};
    const int u = (threadIdx.x >> 6) + PNW * s;
    if (u >= nt * (nt + 1) / 2) continue;
    int ti, tj;
    sym_tile(u, nt, ti, tj);
    const double* a = M + (16 * ti + li) * ld + lk;
    const double* b = M + (16 * tj + li) * ld + lk;
    for (int k = 0; k < np; k += 16)
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        const v2d x = *(const v2d*)(a + k + t), y = *(const v2d*)(b + k + t);
        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, acc[s], 0, 0, 0);
        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, acc[s], 0, 0, 0);
      }
  }
}

// f(i, j, value) with i <= j tile-wise for every element that sym_product left in acc;
// M(i, j) = M(j, i) = f's result
template <typename F>
__device__ __forceinline__ void sym_store(double* M, int np, const v4d (&acc)[PSYM], F f) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int nt = np / 16, ld = np + 2;
#pragma unroll
  for (int s = 0; s < PSYM; s++) {
    const int u = (threadIdx.x >> 6) + PNW * s;
    if (u >= nt * (nt + 1) / 2) continue;
    int ti, tj;
    sym_tile(u, nt, ti, tj);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = 16 * ti + 4 * e + lk, j = 16 * tj + li;
      const double v = f(i, j, acc[s][e], ti != tj);
      M[i * ld + j] = v;
      if (ti != tj) M[j * ld + i] = v;
    }
  }
}

}  // namespace

// The whole iteration in one work-group, for n <= POLAR_ONE, padded to np (a
// multiple of 16) columns.  One matrix at a time is in LDS: Y for q = I - Y^T Y, q for
// q^2, and the polynomial I + q/2 + 3 q^2 / 8 (or (Y^T Y)^-1) for the new Y,
// whose old columns come from the XCD's L2; Y and its successor alternate between two
// buffers.  The products of one matrix are symmetric: only their upper tiles
// are formed.  One CU's MFMA rate bounds it (13 us a Bjorck-Bowie step at n = 90; 38 us
// measured, 64 us with every operand from L2).
__global__ __launch_bounds__(PNT) void k_polar_one(double* Yio, int n, double tol, int maxiter,
                                                   int* flags, double* qnrm, double* Y,
                                                   double* Y2, double* lt, double* SX) {
  __shared__ __align__(16) double M[POLAR_ONE * PLD];
  __shared__ double sums[PNW];
  __shared__ int bad;
  const int tid = threadIdx.x, np = (n + 15) & ~15, ld = np + 2, ldx = 2 * np;
  const int lane = tid & 63, li = lane & 15, lk = lane >> 4;
  for (int e = tid; e < np * np; e += PNT) {
    const int c = e / np, r = e - c * np;
    const double v = r < n && c < n ? Yio[r + c * n] : 0.0;
    Y[e] = v;
    M[c * ld + r] = v;
  }
  int iters = 0, singular = 0;
  double qn = 0.0;
  __syncthreads();
  for (int it = 0; it < maxiter; it++) {
    v4d acc[PSYM];
    sym_product(M, np, acc);
    __syncthreads();
    double v = 0.0;
    sym_store(M, np, acc, [&](int i, int j, double d, bool twice) {
      const double x = (i == j && i < n ? 1.0 : 0.0) - d;
      v += twice ? 2.0 * (x * x) : x * x;
      return x;
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) sums[tid >> 6] = v;
    __syncthreads();
    v = 0.0;
    for (int i = 0; i < PNW; i++) v += sums[i];
    qn = sqrt(v);
    iters++;
    const bool bjorck = qn < 1.0;
    if (bjorck) {
      // Bjorck-Bowie: Y <- Y (I + q/2 (I + 3q/4))
      sym_product(M, np, acc);
      const int nt = np / 16;
#pragma unroll
      for (int s = 0; s < PSYM; s++) {
        const int u = (tid >> 6) + PNW * s;
        if (u >= nt * (nt + 1) / 2) continue;
        int ti, tj;
        sym_tile(u, nt, ti, tj);
#pragma unroll
        for (int e = 0; e < 4; e++)
          acc[s][e] = 0.5 * (M[(16 * ti + 4 * e + lk) * ld + 16 * tj + li] + 0.75 * acc[s][e]);
      }
      __syncthreads();
      sym_store(M, np, acc, [&](int i, int j, double d, bool) { return (i == j ? 1.0 : 0.0) + d; });
    } else {
      // Higham: Y <- (Y + Y (Y^T Y)^-1) / 2, Y^T Y = I - q = L L^T, with the
      // Cholesky steps of chol_inverse
      for (int e = tid; e < np * np; e += PNT) {
        const int c = e / np, r = e - c * np;
        const double one = r == c ? 1.0 : 0.0;
        SX[r + c * ldx] = one - M[c * ld + r];
        SX[np + r + c * ldx] = one;
      }
      __syncthreads();
      for (int j0 = 0; j0 < np && !singular; j0 += CB) {
        const int jb = min(CB, np - j0), j1 = j0 + jb;
        for (int blk = 0; blk * CB < np && !singular; blk++) {
          singular = chol_panel<PNT>(SX, np, j0, jb, blk, lt, M, &bad);
          __syncthreads();
        }
        // rows j1 .. np + j1 of the columns right of the panel (jb = 64 here)
        const int nr = np / 16, nc = singular ? 0 : (np - j1) / 16;
        for (int t = tid >> 6; t < nr * nc; t += PNW) {
          const int i0 = 16 * (t % nr), k0 = 16 * (t / nr);
          double* d = SX + (j1 + i0 + li) + (j1 + k0 + lk) * ldx;
          v4d x;
#pragma unroll
          for (int e = 0; e < 4; e++) x[e] = d[4 * e * ldx];
          const double* b = SX + (j1 + i0 + li) + (j0 + lk) * ldx;
          const double* a = lt + lk + (k0 + li) * CB;
#pragma unroll 4
          for (int m = 0; m < CB; m += 4)
            x = __builtin_amdgcn_mfma_f64_16x16x4f64(a[m], b[m * ldx], x, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; e++) d[4 * e * ldx] = x[e];
        }
        __syncthreads();
      }
      if (singular) break;
      // X = L^-T by rows: (Y^T Y)^-1 = X X^T
      for (int e = tid; e < np * np; e += PNT) {
        const int c = e / np, r = e - c * np;
        M[r * ld + c] = SX[np + r + c * ldx];
      }
      __syncthreads();
      sym_product(M, np, acc);
      __syncthreads();
      sym_store(M, np, acc, [&](int, int, double d, bool) { return d; });
    }
    __syncthreads();
    // Y2(i, j) = sum_k Y(i, k) M(k, j), M symmetric
    v4d y[PTILES];
    const int nt = np / 16;
#pragma unroll
    for (int s = 0; s < PTILES; s++) {
      y[s] = v4d{0, 0, 0, 0};
      const int u = (tid >> 6) + PNW * s;
      if (u >= nt * nt) continue;
      const int i0 = 16 * (u % nt), j0 = 16 * (u / nt);
      const double* a = M + (j0 + li) * ld + 4 * lk;
      const double* b = Y + i0 + li + 4 * lk * np;
      for (int k = 0; k < np; k += 16) {
        const v2d m0 = *(const v2d*)(a + k), m1 = *(const v2d*)(a + k + 2);
        const double* bk = b + k * np;
        y[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0.x, bk[0], y[s], 0, 0, 0);
        y[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0.y, bk[np], y[s], 0, 0, 0);
        y[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(m1.x, bk[2 * np], y[s], 0, 0, 0);
        y[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(m1.y, bk[3 * np], y[s], 0, 0, 0);
      }
      if (!bjorck)
#pragma unroll
        for (int e = 0; e < 4; e++)
          y[s][e] = 0.5 * (y[s][e] + Y[i0 + li + (j0 + 4 * e + lk) * np]);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < PTILES; s++) {
      const int u = (tid >> 6) + PNW * s;
      if (u >= nt * nt) continue;
      const int i0 = 16 * (u % nt), j0 = 16 * (u / nt);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i = i0 + li, j = j0 + 4 * e + lk;
        Y2[i + j * np] = y[s][e];
        M[j * ld + i] = y[s][e];
      }
    }
    double* x = Y;
    Y = Y2;
    Y2 = x;
    __syncthreads();
    if (qn <= tol) break;
  }
  for (int e = tid; e < n * n; e += PNT) {
    const int c = e / n, r = e - c * n;
    Yio[e] = Y[r + c * np];
  }
  if (tid == 0) {
    flags[0] = iters && qn <= tol ? 1 : 0;
    flags[3] = iters;
    flags[4] = singular ? 1 : 0;
    flags[5] = singular;
    *qnrm = qn;
  }
}

size_t polar_elems(int n) {
  const size_t m = n <= POLAR_ONE ? (size_t)((n + 15) & ~15) : (size_t)n;
  return m * m;
}

void launch_polar_one(double* Y, int n, double tol, int maxiter, int* flags, double* qnrm,
                      double* y1, double* y2, double* lt, double* sx, hipStream_t s) {
  hipLaunchKernelGGL(k_polar_one, dim3(1), dim3(PNT), 0, s, Y, n, tol, maxiter, flags, qnrm, y1,
                     y2, lt, sx);
}

}  // namespace qbg
