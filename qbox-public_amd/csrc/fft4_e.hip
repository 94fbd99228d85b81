// fft4_e.hip -- alternative line splits of the lengths 90, 112, 126 and 144
// (see fft4_kernels.h); the grid's tuner times them against the
// default splits and keeps the faster per axis and precision.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_e[] = {
    QBG_F4(9, 10),    // 90
    QBG_F4(14, 8),    // 112
    QBG_F4(9, 14),    // 126
    QBG_F4(16, 9),    // 144
};

const F4Ops* f4_table_e(int* count) {
  *count = (int)(sizeof(ops_e) / sizeof(ops_e[0]));
  return ops_e;
}

}  // namespace qbg
