// Q4 instantiations of the wave-split matmul (aexq_qmmk.hpp) with fp16 weight
// tiles, fp16(q * s): the M > 32 form (RMSNorm-in by the row pre-pass).
#include "aexq_qmmk.hpp"

namespace aexq {

#define QMMK(G, SF16, ...) QMMK_ENTRY(kQ4, G, SF16, true, __VA_ARGS__)
#define QMMK_ALL(G, SF16)                                                                          \
  QMMK(G, SF16, 1, 1, 8, false, false, false), QMMK(G, SF16, 2, 1, 8, false, false, false),       \
      QMMK(G, SF16, 2, 2, 8, false, false, false), QMMK(G, SF16, 2, 2, 4, false, false, false),   \
      QMMK(G, SF16, 4, 2, 4, false, false, false), QMMK(G, SF16, 1, 1, 8, true, false, false),    \
      QMMK(G, SF16, 2, 2, 8, true, false, false), QMMK(G, SF16, 2, 2, 4, true, false, false)

static const QmmkEntry kTable[] = {QMMK_ALL(32, true), QMMK_ALL(32, false), QMMK_ALL(16, true),
                                   QMMK_ALL(16, false)};

const QmmkEntry* qmmk_table_q4_fd(int* count) {
  *count = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

}  // namespace aexq
