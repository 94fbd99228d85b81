// fft4_o.hip -- four-step / prime-factor pass kernels for line lengths
// 360, 384, 396.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_o[] = {
    QBG_F4(20, 18),   // 360
    QBG_F4(24, 16),   // 384
    QBG_F4(22, 18),   // 396
};

const F4Ops* f4_table_o(int* count) {
  *count = (int)(sizeof(ops_o) / sizeof(ops_o[0]));
  return ops_o;
}

}  // namespace qbg
