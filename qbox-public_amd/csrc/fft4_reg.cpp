// fft4_reg.cpp -- registry of the compiled four-step line lengths: the
// default split of each length (fft4_a..d, fft4_g..o), the alternatives the
// grid's tuner may pick instead (fft4_e, fft4_f), and slower ones that callers' plans
// may hold (fft4_p).
//
// Every even length 16 <= n <= 396 that Basis and ChargeDensity can choose
// for a grid (2^a 3^b 5^c 7^d 11^e with b <= 2 and c, d, e <= 1, a >= 1) is
// compiled, so the grid of any cell and cutoff up to that length runs on the
// register kernels; the generic Stockham passes (fft.hip) are left for callers
// whose own grids have other lengths.  The register kernels exchange a line
// through LDS once instead of once per radix stage, hold the small DFTs as
// compile-time constants and load only the active rows: 47 bands with two spins
// in a 15 x 17.5 x 21 bohr cell (45 Ry, FP32) evaluate in 0.61 ms where the
// Stockham passes take 1.27 ms, 64 bands at three k-points (55 Ry, 15.5 bohr)
// in 2.00 ms where they take 5.66 ms.
//
// Which split: the one whose passes are fastest with every divisor pair timed
// (cubes of 36 to 256, 32 to 128 bands, both precisions).  Two balanced factors of at most
// 16 win everywhere, coprime or not: 80 as 10 x 8 takes 0.60 of the time of
// 20 x 4, 168 as 14 x 12 0.82 of 21 x 8, 180 as 15 x 12 0.81 of 20 x 9.
// A factor above 16 needs more than four waves a block, fewer blocks fit, and the
// long DFT is left to few of the waves; 198, 220, 252 and the lengths above 256
// have no other.
#include "internal.h"

namespace qbg {

const F4Ops* f4_table_a(int* count);
const F4Ops* f4_table_b(int* count);
const F4Ops* f4_table_c(int* count);
const F4Ops* f4_table_d(int* count);
const F4Ops* f4_table_e(int* count);
const F4Ops* f4_table_f(int* count);
const F4Ops* f4_table_g(int* count);
const F4Ops* f4_table_h(int* count);
const F4Ops* f4_table_i(int* count);
const F4Ops* f4_table_j(int* count);
const F4Ops* f4_table_k(int* count);
const F4Ops* f4_table_l(int* count);
const F4Ops* f4_table_m(int* count);
const F4Ops* f4_table_n(int* count);
const F4Ops* f4_table_o(int* count);
const F4Ops* f4_table_p(int* count);

namespace {
// defaults first, so the first match of a length is its default split
const F4Ops* (*const kTables[])(int*) = {f4_table_a, f4_table_b, f4_table_c,
                                          f4_table_d, f4_table_g, f4_table_h, f4_table_i,
                                          f4_table_j, f4_table_k, f4_table_l, f4_table_m,
                                          f4_table_n, f4_table_o, f4_table_e, f4_table_f,
                                          f4_table_p};
constexpr int KEPT = 1;     // of them, at the end: not timed
}  // namespace

const F4Ops* f4_ops(int n) {
  const F4Ops* out = nullptr;
  return f4_candidates(n, &out, 1) ? out : nullptr;
}

int f4_candidates(int n, const F4Ops** out, int cap, bool kept) {
  const int tables = (int)(sizeof(kTables) / sizeof(kTables[0])) - (kept ? 0 : KEPT);
  int k = 0;
  for (int j = 0; j < tables; j++) {
    int cnt = 0;
    const F4Ops* t = kTables[j](&cnt);
    for (int i = 0; i < cnt; i++)
      if (t[i].n == n && k < cap) out[k++] = &t[i];
  }
  return k;
}

}  // namespace qbg
