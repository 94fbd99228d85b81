// fft4_m.hip -- four-step / prime-factor pass kernels for line lengths
// 288, 308, 320.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_m[] = {
    QBG_F4(18, 16),   // 288
    QBG_F4(22, 14),   // 308
    QBG_F4(20, 16),   // 320
};

const F4Ops* f4_table_m(int* count) {
  *count = (int)(sizeof(ops_m) / sizeof(ops_m[0]));
  return ops_m;
}

}  // namespace qbg
