// fft4_i.hip -- four-step / prime-factor pass kernels for line lengths
// 88, 110, 120, 132, 140.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_i[] = {
    QBG_F4(11, 8),   // 88
    QBG_F4(11, 10),   // 110
    QBG_F4(15, 8),   // 120
    QBG_F4(12, 11),   // 132
    QBG_F4(14, 10),   // 140
};

const F4Ops* f4_table_i(int* count) {
  *count = (int)(sizeof(ops_i) / sizeof(ops_i[0]));
  return ops_i;
}

}  // namespace qbg
