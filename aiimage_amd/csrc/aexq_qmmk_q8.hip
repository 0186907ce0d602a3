// Q8 instantiations of the wave-split matmul (aexq_qmmk.hpp) and the lookup.
#include "aexq_qmmk.hpp"

namespace aexq {

#define QMMK(G, SF16, MT, NT, W, PAIR, RMS, RAG)                              \
  QmmkEntry {                                                                \
    QmmkConfig{kQ8, G, SF16, false, MT, NT, W, PAIR, RMS, RAG},               \
        &qmmk_kernel<kQ8, G, SF16, false, MT, NT, W, PAIR, RMS, RAG>,         \
        QmmK<kQ8, G, SF16, false, MT, NT, PAIR, RMS, RAG>::SLOT               \
  }
#define QMMK_ALL(G, SF16)                                                                          \
  QMMK(G, SF16, 1, 1, 8, false, false, false), QMMK(G, SF16, 1, 2, 8, false, false, false),       \
      QMMK(G, SF16, 2, 1, 8, false, false, false), QMMK(G, SF16, 2, 2, 8, false, false, false),   \
      QMMK(G, SF16, 2, 2, 4, false, false, false), QMMK(G, SF16, 4, 2, 4, false, false, false),   \
      QMMK(G, SF16, 1, 1, 8, true, false, false), QMMK(G, SF16, 1, 2, 8, true, false, false),     \
      QMMK(G, SF16, 2, 2, 8, true, false, false), QMMK(G, SF16, 2, 2, 4, true, false, false),     \
      QMMK(G, SF16, 1, 1, 8, false, true, false), QMMK(G, SF16, 1, 2, 8, false, true, false),     \
      QMMK(G, SF16, 2, 1, 8, false, true, false), QMMK(G, SF16, 2, 2, 8, false, true, false),     \
      QMMK(G, SF16, 1, 1, 8, true, true, false), QMMK(G, SF16, 1, 2, 8, true, true, false),       \
      QMMK(G, SF16, 2, 2, 8, true, true, false), QMMK(G, SF16, 1, 1, 8, false, false, true),      \
      QMMK(G, SF16, 2, 2, 4, false, false, true), QMMK(G, SF16, 1, 1, 8, false, true, true),      \
      QMMK(G, SF16, 2, 2, 4, false, true, true)

static const QmmkEntry kTable[] = {QMMK_ALL(0, true), QMMK_ALL(0, false)};

const QmmkEntry* qmmk_table_q8(int* count) {
  *count = (int)(sizeof(kTable) / sizeof(kTable[0]));
  return kTable;
}

const QmmkEntry* qmmk_find(const QmmkConfig& c) {
  int n = 0;
  const QmmkEntry* t = c.fmt == kQ8 ? qmmk_table_q8(&n) : (c.fd ? qmmk_table_q4_fd(&n) : qmmk_table_q4(&n));
  for (int i = 0; i < n; ++i) {
    const QmmkConfig& q = t[i].cfg;
    if (q.fmt == c.fmt && q.g == c.g && q.sf16 == c.sf16 && q.fd == c.fd && q.mt == c.mt &&
        q.nt == c.nt && q.waves == c.waves && q.pair == c.pair && q.rms == c.rms && q.rag == c.rag)
      return &t[i];
  }
  return nullptr;
}

// Most LDS a launch's rings take together (160 KB a CU, less the kernel's own arrays).
static constexpr int kRingLds = 152 * 1024;

// The tile and wave count of a launch.
// Measured per call on single layers, rotated weights (Q4 groups of 32 / Q8,
// us): N = 1024, K = 2048, M = 16: 5.4 / 5.2 against 8.8 / 7.9 on the MFMA
// block kernels with their split-K fix-up, M = 64: 5.9 / 5.7 against 10.4 / 9.9
// on the tiled GEMM, M = 512: 9.9 / 9.5 against 23.8 / 23.2.
bool qmmk_pick(int m, long long t16, bool q8, bool pair, bool rag, int* mt, int* nt, int* waves) {
  const long long m16 = (m + 15) / 16, m32 = (m + 31) / 32, m64 = (m + 63) / 64;
  const long long t32 = (t16 + 1) / 2;
  auto take = [&](int a, int b, int w) {
    *mt = a;
    *nt = b;
    *waves = w;
    return true;
  };
  // about a workgroup per CU: the smallest tiles, whose workgroups fetch least
  if (t16 * m16 <= 320) return take(1, 1, 8);
  // ragged K: no other matrix-core kernel takes it
  if (rag) return take(2, 2, 4);
  if (m <= 16) {
    // two weight blocks halve the activation bytes (N = 16384, K = 1024: 7.0
    // us against 9.1 with one block).  Beyond 1024 workgroups the launch
    // streams from HBM, which the wide kernel's persistent workgroups do better
    // (Q4, 3584 x 1024 by 120 copies: 80 us against 98; N = 32768, K = 4096: 32
    // against 28)
    return t32 <= 1024 && take(1, 2, 8);
  }
  if (m <= 32) {
    if (pair) {
      if (t16 <= 320) return take(1, 2, 8);  // 3584 pairs, M = 32: 8.6 us; 1:1 9.4, 2:1 8.9
    } else if (t16 <= 320) {
      return take(2, 1, 8);  // 3072 x 1024, M = 32: 5.2 us; 1:1 6.1, 2:2 5.7
    }
    return t32 <= 512 && take(2, 2, 8);
  }
  // Q8 from 96 tiles of 128 x 128: the tiled GEMM's eight-wave form (512 x 3072 x
  // 1024: 18.8 us against 21.1; Q4, which expands its codes twice there, 22.0
  // against 21.6)
  if (q8 && m > 64 && (t16 + (pair ? 3 : 7)) / (pair ? 4 : 8) * ((m + 127) / 128) >= 96) return false;
  if (!pair && t16 * m16 <= 640) return take(2, 1, 8);  // 1024 x 2048, M = 128: 6.7 us; 2:2 7.2
  if (t32 * m32 <= 256) return take(2, 2, 8);           // 4096 x 4096, M = 64: 9.9 us; 4 waves 10.9
  // more workgroups than CUs: four waves each, several workgroups per CU
  // (3072 x 1024, M = 256: 9.2 us against 13.9 with eight waves)
  if (t32 * m32 <= 900) return take(2, 2, 4);
  // larger tiles fetch less per product (4096 x 4096, M = 256: 21.6 us against
  // 25.7); beyond this the tiled GEMM, whose waves share their tiles, wins
  // (M = 512 SwiGLU pair of 3584: 23 us against 28)
  return !pair && t32 * m64 <= 768 && take(4, 2, 4);
}

int qmmk_depth(const QmmkEntry* e, int k, long long wgs, int cus) {
  // a ring takes up to a CU's whole LDS where each CU gets one workgroup, half
  // of it for larger launches (RMSNorm-in reads rows longer than it twice)
  const int ring = e->cfg.waves * e->slot;  // LDS bytes per slot of every wave
  const int slices = (k + kQmmkSlice - 1) / kQmmkSlice;
  const int ns = (slices + e->cfg.waves - 1) / e->cfg.waves;  // of one wave
  int depth = (wgs <= cus || e->cfg.rms ? kRingLds : kRingLds / 2) / ring;
  depth = depth < 1 ? 1 : (depth > kQmmkMaxDepth ? kQmmkMaxDepth : depth);
  return depth < ns ? depth : ns;
}

hipError_t qmmk_launch(const QmmkEntry* e, const QmvParams& p, int depth, hipStream_t stream) {
  if (!e || depth < 1 || depth > kQmmkMaxDepth || p.nmat < 1 || p.nmat > kMaxGroup)
    return hipErrorInvalidConfiguration;
  const int mtiles = (p.m + 16 * e->cfg.mt - 1) / (16 * e->cfg.mt);
  const long long grid = (p.total_tiles + 7LL) / 8 * 8 * mtiles;
  if (grid <= 0 || grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  const size_t bytes = (size_t)e->cfg.waves * depth * e->slot;
  if (bytes > 64 * 1024) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    const uint64_t bit = 1ull << (dev & 63);
    if (dev > 63 || !(e->large_lds.load(std::memory_order_relaxed) & bit)) {
      err = hipFuncSetAttribute((const void*)e->fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                kRingLds);
      if (err != hipSuccess) return err;
      if (dev <= 63) e->large_lds.fetch_or(bit, std::memory_order_relaxed);
    }
  }
  hipLaunchKernelGGL(e->fn, dim3((unsigned)grid), dim3(64 * e->cfg.waves), bytes, stream,
                     p, mtiles, depth);
  return hipGetLastError();
}

}  // namespace aexq
