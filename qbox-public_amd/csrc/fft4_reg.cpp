// fft4_reg.cpp -- registry of the compiled four-step line lengths: the
// default split of each length (fft4_a..d, fft4_g..o), the alternatives the
// grid's tuner may pick instead (fft4_e, fft4_f), and slower or less accurate ones
// that callers' plans may hold (fft4_p).
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
// Which split: to 256 points the one whose passes are fastest with every
// divisor pair timed (cubes of 36 to 256, 32 to 128 bands, both precisions).  Two balanced
// factors of at most 16 win everywhere, coprime or not: 80 as 10 x 8 takes 0.60 of
// the time of 20 x 4, 168 as 14 x 12 0.82 of 21 x 8, 180 as 15 x 12 0.81 of 20 x 9.
// A factor above 16 needs more than four waves a block, fewer blocks fit, and the
// long DFT is left to few of the waves; 198, 220, 252 and the lengths above 256
// have no other.  The lengths above 256 take the most balanced pair untimed.
// Between pairs that are equal to a few per cent the FP32 error decides: the rounding of
// the constants acts on all lines alike, so it stays in a density.  160 as 10 x 16 is
// 4 % faster than 16 x 10 (269 and 279 us, 24 bands in FP32, potential pass and all) and
// its densities are 9 to 14 % further off (9.7e-8 and 8.5e-8); 96 as 8 x 12 3 % and
// 1 to 2 %, 128 as 8 x 16 0 and 2 to 3 %, 168 as 12 x 14 slower and 1 %.
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
