// fft4_n.hip -- four-step / prime-factor pass kernels for line lengths
// 330, 336, 352.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_n[] = {
    QBG_F4(22, 15),   // 330
    QBG_F4(21, 16),   // 336
    QBG_F4(22, 16),   // 352
};

const F4Ops* f4_table_n(int* count) {
  *count = (int)(sizeof(ops_n) / sizeof(ops_n[0]));
  return ops_n;
}

}  // namespace qbg
