// Q8 instantiations of the wave-split matmul (aexq_qmmk.hpp) and the lookup.
#include "aexq_qmmk.hpp"

namespace aexq {

#define QMMK(G, SF16, ...) QMMK_ENTRY(kQ8, G, SF16, false, __VA_ARGS__)
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

// The tile and wave count of a launch, or false where another kernel is the
// better one.  Limits on the grid are in workgroups per CU, and count the grid's
// padding to 8 weight tiles (a tile of the last group adds a whole column of row
// tiles to one XCD); limits on K are there because a workgroup walks all of it
// while the other kernels split it over more of them.  The lines are drawn where
// 55 thousand random launches (M 2..2048, N 32..40000, K 128..32768, rotated
// weights, each against the kernel that it takes with this one off) turn; of 36
// thousand others that they let through, stacked copies and groups among them, 20
// are more than 3% slower and five in six more than 20% faster.  Both sides of the
// lines, us, here / there:
bool qmmk_pick(const QmmkShape& q, int* mt, int* nt, int* waves) {
  const int m = q.m, K = q.k;
  const bool q8 = q.fmt == kQ8, g16 = q.g == 16, pair = q.pair;
  const bool exact = q.fmt == kQ4 && !q.fd;
  const long long m16 = (m + 15) / 16, m32 = (m + 31) / 32, m64 = (m + 63) / 64;
  const long long t16 = q.t16, t32 = q.t32;
  const long long cu = q.cus;
  auto take = [&](int a, int b, int w) {
    *mt = a;
    *nt = b;
    *waves = w;
    return true;
  };
  // workgroups of tiles of 16 nt weight rows, as the grid pads them
  auto grid = [&](int nt_, long long mtiles) { return ((nt_ == 1 ? t16 : t32) + 7) / 8 * 8 * mtiles; };
  // ragged K: no other matrix-core kernel takes it, and one row of less than half
  // a slice is all launch (N = 97, K = 48: 4.4 / 3.9)
  if (q.rag && m == 1 && K < 64) return false;
  if (q.rag) return t16 * m16 <= cu * 5 / 4 ? take(1, 1, 8) : take(2, 2, 4);
  if (m <= 32) {
    if (t16 * m16 <= cu * 5 / 4) {
      // about a workgroup per CU: the smallest tiles, whose workgroups fetch least
      // (N = 1024, K = 2048, M = 16: 5.4 / 8.8).  RMSNorm-in spares the other
      // kernel's pre-pass at any K; past one workgroup per CU the longer rows are
      // read twice by two workgroups a CU (Q4, N = 4563, K = 2816, M = 5: 16.0 / 13.4)
      const long long g = grid(1, m16);
      if (g > cu) return K <= (q.rms ? 1024 : 8192) && take(1, 1, 8);
      // without it, long rows of few tiles: N = 1024, K = 28672, M = 16: Q8 27 /
      // 18, groups of 16 30 / 20; N = 64, K = 8192, M = 5, groups of 16: 9.3 / 8.9
      const int most = q8 ? 12288 : (g16 && pair ? 4096 : 6144);
      return (q.rms || K <= (g <= cu / 2 ? most : 2 * most)) && take(1, 1, 8);
    }
    if (m <= 16 || (pair && t16 <= cu * 5 / 4)) {
      // two weight blocks halve the activation bytes (N = 16384, K = 1024: 7.0 /
      // 9.1 with one block)
      const long long g = grid(2, m16);
      if (g <= cu) return (q.rms || K <= (pair ? 8192 : 16384)) && take(1, 2, 8);
      // a pair's second workgroup on a CU waits for its LDS (Q8, 12676 pairs, K =
      // 256, M = 7: 10.6 / 6.4; groups of 32, whose other kernel is slower, 7.6 / 8.3)
      if (pair) return !q8 && !g16 && g <= 2 * cu && K <= 1024 && take(1, 2, 8);
      // the norm reads rows longer than the ring twice
      if (q.rms) return g <= 2 * cu && K <= 1024 && take(1, 2, 8);
      // past two per CU the launch streams from HBM, which persistent workgroups
      // do better (Q8, N = 26496, K = 256, M = 7: 8.3 / 6.1), but for groups of 32
      // (N = 24150, K = 128: 5.2 / 6.4)
      return K <= 6144 && g <= (q8 || g16 ? 2 : 4) * cu && take(1, 2, 8);
    }
    if (!pair && t16 <= cu * 5 / 4) {
      // 3072 x 1024, M = 32: 5.2 us; 1:1 6.1, 2:2 5.7
      const long long g = grid(1, m32);
      if (g <= cu) return (q.rms || K <= 12288) && take(2, 1, 8);
      return !q.rms && K <= 6144 && take(2, 1, 8);
    }
    // exact products of a pair in groups of 16 hold more than the registers there
    // are (8192 pairs, K = 7936, M = 23: 177 / 63)
    if (pair && g16) return false;
    const long long g = grid(2, 1);
    if (g <= cu) return take(2, 2, 8);
    return !g16 && !q.rms && !pair && g <= cu * 3 / 2 && K >= 512 && K <= 3072 && take(2, 2, 8);
  }
  if (t16 * m16 <= cu * 5 / 4)  // M = 64, N = 1024, K = 2048: 5.9 / 10.4
    return (grid(1, m16) <= cu || K <= 6144) && take(1, 1, 8);
  // Q8 from 96 tiles of 128 x 128: the tiled GEMM's eight-wave form (512 x 3072 x
  // 1024: 18.8 us against 21.1)
  if (q8 && m > 64 && (t16 + (pair ? 3 : 7)) / (pair ? 4 : 8) * ((m + 127) / 128) >= cu * 3 / 8)
    return false;
  if (!pair && t16 * m16 <= cu * 5 / 2)  // 1024 x 2048, M = 128: 6.7 us; 2:2 7.2
    return K <= (grid(1, m32) <= cu ? 24576 : 6144) && take(2, 1, 8);
  if (t32 * m32 <= cu)  // 4096 x 4096, M = 64: 9.9 us; 4 waves 10.9; K = 28672: 48 / 39
    return !(exact && pair && g16) && K <= (pair ? 4096 : 6144) && take(2, 2, 8);
  if (t32 * m32 <= cu * 7 / 2) {
    // more workgroups than CUs: four waves each, several workgroups per CU
    // (3072 x 1024, M = 256: 9.2 us against 13.9 with eight waves).  Up to 64
    // rows the tiled GEMM reads each weight tile once, not twice (N = 12672, K =
    // 640, M = 43: 9.7 / 8.4; 11968 pairs, K = 768, M = 37: 14.3 / 11.4)
    const long long g = grid(2, m32);
    // exact products scale every MFMA's result in fp32: a pair's go faster through
    // tiles that are expanded once for more rows (groups of 32, 5056 pairs, K =
    // 2304, M = 39: 23.8 / 19.1)
    if (exact) return !pair && g <= 3 * cu && K <= 3072 && take(2, 2, 4);
    if (pair)
      return ((g <= 2 * cu && K <= 3072) || (m > 64 && g <= 3 * cu && K <= 2048)) && take(2, 2, 4);
    if (g <= 3 * cu) return K <= (g <= 2 * cu ? 6144 : 4096) && take(2, 2, 4);
    return m > 64 && K <= 3072 && take(2, 2, 4);
  }
  // larger tiles fetch less per product (2459 x 1024, M = 556: 14.9 / 24.8); short
  // rows leave their four waves a slice or two each (N = 2816, K = 768, M = 398:
  // 14.1 / 13.1), long ones wait for them (N = 993, K = 3840, M = 1499: 54 / 40),
  // and a single row of tiles is the tiled GEMM's sooner (Q8, N = 24030, K = 1280,
  // M = 45: 19.1 / 14.0)
  const long long g = grid(2, m64);
  return !pair && !exact && g <= (m > 64 ? 3 : 2) * cu && K >= 896 &&
         K <= (g <= cu * 5 / 2 ? 2048 : 1280) && take(4, 2, 4);
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
