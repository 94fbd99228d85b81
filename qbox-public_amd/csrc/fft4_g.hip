// fft4_g.hip -- four-step / prime-factor pass kernels for line lengths
// 16, 18, 20, 30, 32, 36, 40, 42, 44, 48.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_g[] = {
    QBG_F4(4, 4),   // 16
    QBG_F4(6, 3),   // 18
    QBG_F4(5, 4),   // 20
    QBG_F4(10, 3),   // 30
    QBG_F4(8, 4),   // 32
    QBG_F4(9, 4),   // 36
    QBG_F4(8, 5),   // 40
    QBG_F4(7, 6),   // 42
    QBG_F4(11, 4),   // 44
    QBG_F4(12, 4),   // 48
};

const F4Ops* f4_table_g(int* count) {
  *count = (int)(sizeof(ops_g) / sizeof(ops_g[0]));
  return ops_g;
}

}  // namespace qbg
