// fft4_f.hip -- alternative line splits of the lengths 198, 210 and 224
// (see fft4_kernels.h); the grid's tuner times them against the
// default splits and keeps the faster per axis and precision.
#include "fft4_kernels.h"

namespace qbg {

static const F4Ops ops_f[] = {
    QBG_F4(11, 18),   // 198
    QBG_F4(14, 15),   // 210
    QBG_F4(14, 16),   // 224
};

const F4Ops* f4_table_f(int* count) {
  *count = (int)(sizeof(ops_f) / sizeof(ops_f[0]));
  return ops_f;
}

}  // namespace qbg
