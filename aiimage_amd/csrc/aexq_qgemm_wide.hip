// Eight-wave instantiations of the LDS-direct tiled GEMM (aexq_qgemm_dl.hpp):
// two waves along the activation rows by four along the weight rows.
#include "aexq_qgemm_dl.hpp"

namespace aexq {

#define QGW(FMT, PAIR, SF16, G, FD, KS)                                                    \
  QgemmEntry {                                                                             \
    QgemmConfig{FMT, 128, PAIR, SF16, G == 16, true, FD, (KS) == 128, 2},                  \
        &qgemm_dl_kernel<FMT, 128, PAIR, SF16, G, FD, 2, KS, 3, 2>                         \
  }
// (Q4 takes 128-wide steps: eight waves then load a whole kilobyte of codes each)
#define QGW_ALL(FMT, G, FD, KS)                                                            \
  QGW(FMT, false, true, G, FD, KS), QGW(FMT, false, false, G, FD, KS),                     \
      QGW(FMT, true, true, G, FD, KS), QGW(FMT, true, false, G, FD, KS)

static const QgemmEntry kTableW[] = {QGW_ALL(kQ8, 0, false, 64), QGW_ALL(kQ4, 32, true, 128),
                                     QGW_ALL(kQ4, 16, true, 128)};

const QgemmEntry* qgemm_table_wide(int* count) {
  *count = (int)(sizeof(kTableW) / sizeof(kTableW[0]));
  return kTableW;
}

}  // namespace aexq
