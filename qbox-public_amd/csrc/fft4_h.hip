// fft4_h.hip -- four-step / prime-factor pass kernels for line lengths
// 56, 60, 66, 70, 72, 80, 84.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_h[] = {
    QBG_F4(8, 7),   // 56
    QBG_F4(15, 4),   // 60
    QBG_F4(11, 6),   // 66
    QBG_F4(10, 7),   // 70
    QBG_F4(9, 8),   // 72
    QBG_F4(10, 8),   // 80
    QBG_F4(12, 7),   // 84
};

const F4Ops* f4_table_h(int* count) {
  *count = (int)(sizeof(ops_h) / sizeof(ops_h[0]));
  return ops_h;
}

}  // namespace qbg
