// fft4_p.hip -- splits of 90, 96, 126, 128, 160, 168, 198 and 224 points that
// qbg_grid_plan accepts from plans kept by callers, and the tuner does not time.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_p[] = {
    QBG_F4(18, 5),    // 90
    QBG_F4(16, 6),    // 96
    QBG_F4(8, 12),    // 96
    QBG_F4(18, 7),    // 126
    QBG_F4(32, 4),    // 128
    QBG_F4(8, 16),    // 128
    QBG_F4(20, 8),    // 160
    QBG_F4(10, 16),   // 160
    QBG_F4(21, 8),    // 168
    QBG_F4(12, 14),   // 168
    QBG_F4(22, 9),    // 198
    QBG_F4(32, 7),    // 224
};

const F4Ops* f4_table_p(int* count) {
  *count = (int)(sizeof(ops_p) / sizeof(ops_p[0]));
  return ops_p;
}

}  // namespace qbg
