// fft4_k.hip -- four-step / prime-factor pass kernels for line lengths
// 220, 240, 252.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_k[] = {
    QBG_F4(20, 11),   // 220
    QBG_F4(16, 15),   // 240
    QBG_F4(21, 12),   // 252
};

const F4Ops* f4_table_k(int* count) {
  *count = (int)(sizeof(ops_k) / sizeof(ops_k[0]));
  return ops_k;
}

}  // namespace qbg
