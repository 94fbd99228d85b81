// fft4_l.hip -- four-step / prime-factor pass kernels for line lengths
// 256, 264, 280.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_l[] = {
    QBG_F4(16, 16),   // 256
    QBG_F4(22, 12),   // 264
    QBG_F4(20, 14),   // 280
};

const F4Ops* f4_table_l(int* count) {
  *count = (int)(sizeof(ops_l) / sizeof(ops_l[0]));
  return ops_l;
}

}  // namespace qbg
