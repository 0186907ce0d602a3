// Q4 instantiations of the wave-split matmul (aexq_qmmk.hpp) with exact
// products: each scale group's MFMA result scaled in fp32.
#include "aexq_qmmk.hpp"

namespace aexq {

#define QMMK(G, SF16, ...) QMMK_ENTRY(kQ4, G, SF16, false, __VA_ARGS__)
#define QMMK_ALL(G, SF16)                                                                          \
  QMMK(G, SF16, 1, 1, 8, false, false, false), QMMK(G, SF16, 1, 2, 8, false, false, false),       \
      QMMK(G, SF16, 2, 1, 8, false, false, false), QMMK(G, SF16, 2, 2, 8, false, false, false),   \
      QMMK(G, SF16, 2, 2, 4, false, false, false), QMMK(G, SF16, 1, 1, 8, true, false, false),    \
      QMMK(G, SF16, 1, 2, 8, true, false, false), QMMK(G, SF16, 1, 1, 8, false, true, false),     \
      QMMK(G, SF16, 1, 2, 8, false, true, false), QMMK(G, SF16, 2, 1, 8, false, true, false),     \
      QMMK(G, SF16, 2, 2, 8, false, true, false), QMMK(G, SF16, 1, 1, 8, true, true, false),      \
      QMMK(G, SF16, 1, 2, 8, true, true, false), QMMK(G, SF16, 1, 1, 8, false, false, true),      \
      QMMK(G, SF16, 2, 2, 4, false, false, true), QMMK(G, SF16, 1, 1, 8, false, true, true),      \
      QMMK(G, SF16, 2, 2, 4, false, true, true)
// (pairs in groups of 16 hold two scales per MFMA: over 32 rows by 32 that is
// about 100 registers more than there are)
#define QMMK_PAIR22(G, SF16) \
  QMMK(G, SF16, 2, 2, 8, true, false, false), QMMK(G, SF16, 2, 2, 8, true, true, false)

static const QmmkEntry kTable[] = {QMMK_ALL(32, true), QMMK_ALL(32, false), QMMK_ALL(16, true),
                                   QMMK_ALL(16, false), QMMK_PAIR22(32, true),
                                   QMMK_PAIR22(32, false)};

const QmmkEntry* qmmk_table_q4(int* count) {
  *count = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

}  // namespace aexq
