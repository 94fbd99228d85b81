// fft4_j.hip -- four-step / prime-factor pass kernels for line lengths
// 154, 176, 180, 192.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_j[] = {
    QBG_F4(14, 11),   // 154
    QBG_F4(16, 11),   // 176
    QBG_F4(15, 12),   // 180
    QBG_F4(16, 12),   // 192
};

const F4Ops* f4_table_j(int* count) {
  *count = (int)(sizeof(ops_j) / sizeof(ops_j[0]));
  return ops_j;
}

}  // namespace qbg
