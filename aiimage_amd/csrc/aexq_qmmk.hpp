// Quantized matmul for launches with few output tiles (one layer's linears at
// M = 2 to some hundreds; K that is no multiple of 64 at any M): Y[M][N] =
// X[M][K] W[N][K]^T, the K of a tile split over the waves of one workgroup.
//
// A workgroup owns 16 MT activation rows by 16 NT weight rows (a SwiGLU pair:
// the same rows of both weights) and the whole of K, so nothing is left for a
// second launch: wave w takes the 128-wide K slices w, w + W, ..., and the
// waves' fp32 sums meet in LDS in wave order.  Such a launch is a short chain
// of dependent round trips, so a wave asks for as many of its slices as its
// share of LDS holds at once (LDS-direct loads into a ring of `depth` slots of
// its own, which needs no barrier: a wave waits for its own loads only), and
// the residual and the Q8 row scales are requested at the start.  With one
// workgroup per CU that is up to four slices; launches of more, whose rings
// share a CU, hold one slice a wave on 32 x 32 and 64 x 32 tiles (a slot of all
// waves takes 42 to 80 KB), and there only the other workgroups of the CU cover
// the wait for the next.
//
// The loads go through LDS rather than straight into fragments because of how
// a CU fetches: consecutive lanes reading 16 consecutive bytes of one row keep
// to one cache line, while MFMA lanes (row l % 16, lane group l / 16) would
// touch 16 lines per instruction (measured below).  Slots hold rows with their
// 16-byte chunks XOR-swizzled against bank conflicts in the fragment reads.
// That does not take them all: SQ_LDS_BANK_CONFLICT counts 1.0 to 4.2 stall cycles
// per LDS instruction over a layer's linears.  The MFMA units are busy 0.5 to 2.4%
// of the time on 16-row tiles, 2.2 to 10.5% on larger ones.
//
// Which K the lane groups g of an MFMA carry:
//  * Q8: of each 64-code half codes 16 g .. 16 g + 15, eight to each of its
//    two MFMAs; the row scale comes last, so any order of K will do.
//  * Q4, fp16 weight tiles (FD): codes 32 g .. 32 g + 31 of the slice, eight to
//    each of four MFMAs, and B = fp16(q s).
//  * Q4 exact: an MFMA must cover one scale group, so the 4 x 4 dwords of the
//    lane groups are transposed in registers (two v_permlane32_swap and two
//    v_permlane16_swap per 16 bytes): MFMA e then covers codes 32 e .. 32 e +
//    31, and its product is scaled in fp32 into the accumulator, so the weight
//    is exactly float(q) * scale.  Groups of 16: two MFMAs per extent, each
//    with the other group's activations zeroed (not its codes: an infinite
//    activation times a zeroed code would be NaN in every output).
// The activation fragments are read in the same order.
//
// RMSNorm-in (RMS): the workgroup holds whole activation rows, so it forms
// their sums of squares itself and normalises the fragments as
// fp16(x * inv * gamma), the row pre-pass's arithmetic, without its launch.
// Rows longer than the ring are read twice, for the squares and for the
// products.
//
// Measured per call, graph-replayed single layers with rotated weights (us,
// before -> now): Q4 N = 1024, K = 2048, M = 16: 8.8 -> 5.4 (with fragments
// loaded straight to registers 7.0); N = 1024, K = 3584: 9.7 -> 6.4 (9.5);
// q/k/v with RMSNorm-in 10.6 -> 6.2; the 3584-row SwiGLU pair with RMSNorm-in
// 12.5 -> 7.5.  An empty launch takes 4 there, so what is left over it is the
// memory round trip, the products of one to four slices and the waves' meeting.
//
// RAG: K any multiple of 16 (Q8, Q4 groups of 16) or 32: activations past K
// are read as 0 and scales past the row's last as 0.
#pragma once

#include "aexq_dma.hpp"
#include "aexq_qmm.hpp"

namespace aexq {

constexpr int kQmmkSlice = 128;    // K per slice
constexpr int kQmmkMaxDepth = 4;   // slots of a wave's ring
constexpr int kOutOfRange = 0x7FFFFFF0;  // a buffer offset past every resource

// Transposes the 4 x 4 dwords of the four lane groups: dword d of lane group g
// to dword g of lane group d.  permlane32_swap exchanges the upper half of the
// first operand with the lower half of the second, permlane16_swap the odd
// 16-lane rows of the first with the even ones of the second.
__device__ __forceinline__ u32x4 lane_group_transpose(u32x4 v) {
  auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
  auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return u32x4{c[0], c[1], d[0], d[1]};
}

template <int FMT, int G, bool SF16, bool FD, int MT, int NT, bool PAIR, bool RMS, bool RAG>
struct QmmK {
  static_assert(FMT == kQ8 ? G == 0 : (G == 16 || G == 32), "Q8 row scales or Q4 groups of 16, 32");
  static_assert(!FD || FMT == kQ4, "fp16 weight tiles are a Q4 form");
  static_assert(!RAG || (!FD && !PAIR), "ragged K: exact products");
  static_assert(NT <= 2, "a weight's scales of a slice come in one load");
  static constexpr bool EXACT = FMT == kQ4 && !FD;
  static constexpr int NW = PAIR ? 2 : 1;
  static constexpr int NB = NW * NT;                // 16-row weight blocks
  static constexpr int CB = FMT == kQ8 ? 128 : 64;  // code bytes of a row per slice
  static constexpr int CL = CB / 64;                // 16-byte code loads per block and slice
  static constexpr int SPS = FMT == kQ8 ? 0 : kQmmkSlice / G;  // scales of a row per slice
  static constexpr int SB = SF16 ? 2 : 4;
  // bytes of a row's scales per slice as loaded: ragged fp16 rows start at any
  // even byte, so they take the dwords around them, by dword loads
  static constexpr int SRB = SPS * SB + (RAG && SF16 ? 4 : 0);
  static constexpr int SDW = !RAG && SRB % 16 == 0 ? 16 : 4;  // bytes per lane of a scale load
  static constexpr int SLR = SDW == 0 || SRB == 0 ? 1 : SRB / SDW;  // lanes per row
  static constexpr int SLN = 16 * NT * SLR;         // lanes of a weight's scale loads
  static constexpr int SI = FMT == kQ8 ? 0 : (SLN + 63) / 64;  // scale loads per weight

  // LDS slot of a slice
  static constexpr int XB = MT * 4096;              // 16 rows x 256 bytes per block
  static constexpr int C0 = XB, S0 = C0 + NB * 16 * CB;
  static constexpr int SW = 16 * NT * SRB;          // scale bytes per weight
  static constexpr int G0 = (S0 + NW * SW + 15) & ~15;
  static constexpr int SLOT = G0 + (RMS ? kQmmkSlice * 4 : 0);
  static constexpr int NL = MT * 4 + NB * CL + NW * SI + (RMS ? 1 : 0);  // loads per slice
  static_assert(SLOT >= MT * NB * 1024, "a wave's partial sums reuse its ring");

  struct Src {
    __amdgpu_buffer_rsrc_t xr, wr[NW], sr[NW], gr;
    int xo;   // the lane's byte offset in activation row lane / 16 (slice 0, rows 0..3)
    int wo;   // ... in the weight rows of a block's first code load
    int so;   // ... in the scales
    int rs2, rb, spr;  // activation row stride; code and scale bytes per weight row
    int k, groups;
  };

  // Chunk swizzles (16-byte chunk c of row r at slot c ^ swz(r)).
  static __device__ __forceinline__ constexpr int xswz(int r) {
    if (EXACT) return r & 14;                                    // chunk 4 e + g
    if (FMT == kQ4) return ((r >> 1) & 3) + 8 * ((r >> 3) & 1);  // chunk 4 g + e
    return ((r >> 1) & 1) + 4 * ((r >> 2) & 3);                  // chunk 8 (e / 2) + 2 g + e % 2
  }
  static __device__ __forceinline__ constexpr int cswz(int r) {
    return FMT == kQ8 ? 2 * (r >> 2) : 2 * (r >> 3);
  }
  // The lane group's 16-byte activation chunk of MFMA e in a slice.
  static __device__ __forceinline__ constexpr int xchunk(int e, int g) {
    return EXACT ? 4 * e + g : (FMT == kQ4 ? 4 * g + e : 8 * (e >> 1) + 2 * g + (e & 1));
  }

  static __device__ __forceinline__ Src source(const QmvParams& p, const QmvMat& mt, int b, int n0,
                                               int m0, int lane) {
    Src s;
    s.k = p.k;
    s.groups = p.groups_per_row;
    s.rb = FMT == kQ8 ? p.k : p.k / 2;
    s.spr = p.groups_per_row * SB;
    s.rs2 = (int)(p.x_rstride * 2);
    const int rows = max(min(mt.n - n0, 16 * NT), 0);
    const int mrows = min(p.m - m0, 16 * MT);
    const char* xb = (const char*)mt.x + ((long long)b * mt.x_bstride + (long long)m0 * p.x_rstride) * 2;
    // (the last row ends at K; rows past M read zero)
    s.xr = __builtin_amdgcn_make_buffer_rsrc((void*)sreg(xb), (short)0,
                                             sreg((mrows - 1) * s.rs2 + 2 * p.k),
                                             kBufferRsrcWord3);
#pragma unroll
    for (int h = 0; h < NW; ++h) {
      const char* wb = (const char*)(h ? mt.w2 : mt.w) + (long long)b * mt.w_bstride * 4 +
                       (long long)n0 * s.rb;
      // (whole 16-byte chunks: a copy's storage is padded to 256 bytes)
      s.wr[h] = __builtin_amdgcn_make_buffer_rsrc((void*)sreg(wb), (short)0, sreg((rows * s.rb + 15) & ~15),
                                                  kBufferRsrcWord3);
      const char* sb = (const char*)(h ? mt.s2 : mt.s) + (long long)b * mt.s_bstride * SB +
                       (long long)n0 * s.spr;
      // (whole dwords: a dword only partly inside reads zero; a weight's scale
      // storage runs at least 16 bytes past its last scale)
      s.sr[h] = __builtin_amdgcn_make_buffer_rsrc((void*)sreg(sb), (short)0, sreg((rows * s.spr + 3) & ~3),
                                                  kBufferRsrcWord3);
    }
    if constexpr (RMS)
      s.gr = __builtin_amdgcn_make_buffer_rsrc((void*)sreg(p.gamma), (short)0, sreg(p.gamma ? p.k * 4 : 0),
                                               kBufferRsrcWord3);
    // x: an instruction covers 4 rows of a block; the row swizzles of rows r
    // and r + 4 differ, so load_slice adds the chunk
    s.xo = (lane >> 4) * s.rs2;
    constexpr int CPR = CB / 16;  // chunks per weight row
    s.wo = (lane / CPR) * s.rb;
    if constexpr (FMT == kQ4) {
      const int row = lane / SLR, part = lane % SLR;
      if constexpr (RAG && SF16)
        s.so = ((row * s.spr) & ~3) + 4 * part;
      else
        s.so = row * s.spr + SDW * part;
    }
    return s;
  }

  // The activation rows of one slice into the slot at LDS byte `base`.
  static __device__ __forceinline__ void load_x(const Src& s, uint32_t base, int slice, int lane) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 4 * t + (lane >> 4);
        const int c = (lane & 15) ^ xswz(r);
        int off = s.xo + (16 * m + 4 * t) * s.rs2 + slice * (2 * kQmmkSlice) + 16 * c;
        if constexpr (RAG) off = slice * kQmmkSlice + 8 * c < s.k ? off : kOutOfRange;
        dma<16>(s.xr, base + m * 4096 + t * 1024, off);
      }
  }

  // The loads of one slice into the slot at LDS byte `base`.
  static __device__ __forceinline__ void load(const Src& s, uint32_t base, int slice, int lane) {
#pragma unroll
    for (int h = 0; h < NW; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < CL; ++i) {
          // Q4: 16 rows x 64 bytes; Q8: 8 rows x 128 bytes per load
          constexpr int CPR = CB / 16;
          const int r = (64 / CPR) * i + lane / CPR;
          dma<16>(s.wr[h], base + C0 + ((h * NT + t) * CL + i) * 1024,
                  s.wo + (16 * t + (64 / CPR) * i) * s.rb + slice * CB +
                      16 * ((lane % CPR) ^ cswz(r)));
        }
    if constexpr (FMT == kQ4) {
#pragma unroll
      for (int h = 0; h < NW; ++h)
#pragma unroll
        for (int i = 0; i < SI; ++i) {
          int off = s.so + slice * (SPS * SB);
          if (i > 0) {
            // (ragged fp16 groups of 16: five dwords a row, lanes 64 and on)
            const int l = lane + 64 * i, row = l / SLR;
            off = ((row * s.spr) & (RAG && SF16 ? ~3 : ~0)) + SDW * (l % SLR) + slice * (SPS * SB);
          }
          if (lane + 64 * i < SLN) dma<SDW>(s.sr[h], base + S0 + h * SW + i * 64 * SDW, off);
        }
    }
    load_x(s, base, slice, lane);
    if constexpr (RMS)
      if (lane < 32) dma<16>(s.gr, base + G0, slice * (4 * kQmmkSlice) + 16 * lane);
  }

  static __device__ __forceinline__ void read_x(const char* slot, int lane, f16x8 (&x)[MT][4]) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        x[m][e] = *(const f16x8*)(slot + m * 4096 + r * 256 + 16 * (xchunk(e, g) ^ xswz(r)));
  }

  // The slice's scales of a block the lane needs: every group's (exact), or
  // those of its own 32 codes (FD).
  static constexpr int NS = FMT == kQ8 ? 1 : (EXACT ? SPS : 32 / G);
  static __device__ __forceinline__ void read_s(const Src& s, const char* slot, int h, int t, int slice,
                                                int lane, float (&sc)[NS]) {
    const int r = 16 * t + (lane & 15), g = lane >> 4;
    const char* a = slot + S0 + h * SW + r * SRB;
    if constexpr (RAG) {
      const int odd = SF16 ? (r * s.spr) & 2 : 0;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const float v = SF16 ? (float)*(const f16*)(a + odd + 2 * i) : *(const float*)(a + 4 * i);
        sc[i] = slice * SPS + i < s.groups ? v : 0.0f;
      }
    } else {
      if constexpr (FD) a += g * NS * SB;
#pragma unroll
      for (int i = 0; i < NS; ++i)
        sc[i] = SF16 ? (float)*(const f16*)(a + 2 * i) : *(const float*)(a + 4 * i);
    }
  }

  // fp16(x * inv * gamma) of the lane's fragments.
  static __device__ __forceinline__ void normalise(const char* slot, bool gamma, int lane,
                                                   const float (&inv)[MT], f16x8 (&x)[MT][4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float gm[8];
      const float* gp = (const float*)(slot + G0) + 8 * xchunk(e, lane >> 4);
      const f32x4 a = *(const f32x4*)gp, b = *(const f32x4*)(gp + 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        gm[q] = gamma ? a[q] : 1.0f;
        gm[4 + q] = gamma ? b[q] : 1.0f;
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int q = 0; q < 8; ++q) x[m][e][q] = (f16)((float)x[m][e][q] * inv[m] * gm[q]);
    }
  }

  static __device__ __forceinline__ void compute(const Src& s, const char* slot, int slice, int lane,
                                                 const f16x8 (&x)[MT][4], f32x4 (&acc)[MT][NB]) {
    const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      u32x4 c[CL];
#pragma unroll
      for (int i = 0; i < CL; ++i)
        c[i] = *(const u32x4*)(slot + C0 + t * 16 * CB + r16 * CB + 16 * ((4 * i + g) ^ cswz(r16)));
      float sc[NS];
      if constexpr (FMT == kQ4) read_s(s, slot, t / NT, t % NT, slice, lane, sc);
      if constexpr (EXACT) c[0] = lane_group_transpose(c[0]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t q[4];
        if constexpr (FMT == kQ8) {
          q8_pairs(c[e >> 1][2 * (e & 1)], q[0], q[1]);
          q8_pairs(c[e >> 1][2 * (e & 1) + 1], q[2], q[3]);
        } else {
          q4_pairs_seq(c[0][e], q);
        }
        if constexpr (FD) {
          const f16 s16 = (f16)sc[e * NS / 4];
          const f16x2 s2 = {s16, s16};
#pragma unroll
          for (int j = 0; j < 4; ++j) q[j] = as_u(as_h2(q[j]) * s2);
        }
        const f16x8 bq = pack8(q[0], q[1], q[2], q[3]);
        const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (!EXACT) {
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[m][e], bq, acc[m][t], 0, 0, 0);
        } else if constexpr (G == 32) {
          const float s0 = sc[e];
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[m][e], bq, z, 0, 0, 0);
            acc[m][t] = __builtin_elementwise_fma(f32x4{s0, s0, s0, s0}, v, acc[m][t]);
          }
        } else {
          const float s0 = sc[2 * e], s1 = sc[2 * e + 1];
          const bool first = lane < 32;
          const f16x8 zero = {};
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const f16x8 x0 = first ? x[m][e] : zero, x1 = first ? zero : x[m][e];
            const f32x4 v0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x0, bq, z, 0, 0, 0);
            const f32x4 v1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x1, bq, z, 0, 0, 0);
            acc[m][t] = __builtin_elementwise_fma(f32x4{s0, s0, s0, s0}, v0, acc[m][t]);
            acc[m][t] = __builtin_elementwise_fma(f32x4{s1, s1, s1, s1}, v1, acc[m][t]);
          }
        }
      }
    }
  }
};

// `depth` slots per wave (1 .. kQmmkMaxDepth) in dynamic LDS.
template <int FMT, int G, bool SF16, bool FD, int MT, int NT, int W, bool PAIR, bool RMS, bool RAG>
__global__ __launch_bounds__(64 * W) void qmmk_kernel(const QmvParams p, int mtiles, int depth) {
  using Q = QmmK<FMT, G, SF16, FD, MT, NT, PAIR, RMS, RAG>;
  constexpr int OB = MT * NT;  // 16 x 16 output blocks
  extern __shared__ __align__(16) char lds[];
  __shared__ float ssq[RMS ? W : 1][RMS ? 16 * MT : 1];
  int tile, rem;
  gemm_block_tile(blockIdx.x, p.total_tiles, mtiles, tile, rem);
  const int tn = __builtin_amdgcn_readfirstlane(tile);
  const int tm = __builtin_amdgcn_readfirstlane(rem);
  if (tn < 0) return;
  int j = 0;
  for (int q = 1; q < p.nmat; ++q)
    if (tn >= p.mat[q].tile_base) j = q;
  j = __builtin_amdgcn_readfirstlane(j);
  const QmvMat& mt = p.mat[j];
  const int local = tn - mt.tile_base;
  const int b = __builtin_amdgcn_readfirstlane(local / mt.tiles);
  const int n0 = __builtin_amdgcn_readfirstlane((local - b * mt.tiles) * 16 * NT);
  const int m0 = tm * 16 * MT;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int slices = (p.k + kQmmkSlice - 1) / kQmmkSlice;
  const int ns = wave < slices ? (slices - wave + W - 1) / W : 0;  // this wave's slices
  char* const ring = lds + wave * depth * Q::SLOT;
  const uint32_t ring0 = lds_addr(ring);

  // The outputs this thread finishes -- output block i of wave w, w + W, ... --
  // and what their epilogue reads, requested first (through resources that are
  // empty where there is nothing to read, so no branch holds a wait).
  constexpr int FIN = (OB + W - 1) / W;
  const bool yf32 = (p.flags & kFlagYf32) != 0;
  const int esz = yf32 ? 4 : 2;
  uint32_t res[FIN][4], rsc[FIN][Q::NW];
  {
    const bool resid = mt.res && (p.flags & kFlagResidual);
    const char* rb = (const char*)mt.res + ((long long)b * mt.r_bstride + (long long)m0 * p.r_rstride) * esz;
    const int mrows = min(p.m - m0, 16 * MT);
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)rb, (short)0, resid ? (int)((mrows - 1) * p.r_rstride + mt.n) * esz : 0, kBufferRsrcWord3);
#pragma unroll
    for (int i = 0; i < FIN; ++i) {
      const int ob = wave + i * W;
      const int n = n0 + 16 * (ob % NT) + l16;
      const bool live = ob < OB && n < mt.n;
      const int o0 = (int)((16 * (ob / NT) + 4 * lk) * p.r_rstride + n) * esz;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = live ? o0 + r * (int)p.r_rstride * esz : kOutOfRange;
        if (yf32)
          res[i][r] = __builtin_amdgcn_raw_buffer_load_b32(rr, o, 0, 0);
        else
          res[i][r] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rr, o, 0, 0);
      }
#pragma unroll
      for (int h = 0; h < Q::NW; ++h) {
        rsc[i][h] = 0;
        if constexpr (FMT == kQ8) {
          const char* sb = (const char*)(h ? mt.s2 : mt.s) + (long long)b * mt.s_bstride * Q::SB;
          const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
              (void*)sb, (short)0, (mt.n * Q::SB + 3) & ~3, kBufferRsrcWord3);
          const int o = live ? n * Q::SB : kOutOfRange;
          rsc[i][h] = SF16 ? (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr, o, 0, 0)
                           : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(sr, o, 0, 0);
        }
      }
    }
  }

  const typename Q::Src src = Q::source(p, mt, b, n0, m0, lane);
  f32x4 acc[MT][Q::NB];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int c = 0; c < Q::NB; ++c) acc[a][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  f16x8 x[MT][4];
  float inv[MT], ss[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) ss[m] = 0.0f;
  auto squares = [&](int slots) {  // of the slices in the first slots
    wait_vm<0>();
    asm volatile("" ::: "memory");
    for (int i = 0; i < slots; ++i) {
      Q::read_x(ring + i * Q::SLOT, lane, x);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int q = 0; q < 8; ++q) ss[m] = fmaf((float)x[m][e][q], (float)x[m][e][q], ss[m]);
    }
  };
  // RMSNorm-in over more slices than slots: the later ones' activations pass
  // through the ring for their squares first
  if constexpr (RMS)
    for (int i0 = depth; i0 < ns; i0 += depth) {
      const int cnt = min(depth, ns - i0);
      for (int i = 0; i < cnt; ++i)
        Q::load_x(src, ring0 + i * Q::SLOT, wave + (i0 + i) * W, lane);
      squares(cnt);
      wait_lgkm0();  // read before the next loads
      asm volatile("" ::: "memory");
    }
  for (int i = 0; i < min(depth, ns); ++i) Q::load(src, ring0 + i * Q::SLOT, wave + i * W, lane);

  if constexpr (RMS) {
    squares(min(depth, ns));
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      ss[m] += __shfl_xor(ss[m], 16, 64);
      ss[m] += __shfl_xor(ss[m], 32, 64);
      if (lane < 16) ssq[wave][16 * m + lane] = ss[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float t = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w) t += ssq[w][16 * m + l16];
      inv[m] = rsqrtf(fmaxf(t / (float)p.k + p.eps, 1e-20f));
    }
  }

  int sl = 0;
  for (int i = 0; i < ns; ++i) {
    char* const slot = ring + sl * Q::SLOT;
    const int slice = wave + i * W;
    if (!RMS || i > 0) {
      wait_steps<Q::NL, (63 / Q::NL < kQmmkMaxDepth ? 63 / Q::NL : kQmmkMaxDepth - 1)>(min(ns, i + depth) - i - 1);
      asm volatile("" ::: "memory");
    }
    Q::read_x(slot, lane, x);
    if constexpr (RMS) Q::normalise(slot, p.gamma != nullptr, lane, inv, x);
    Q::compute(src, slot, slice, lane, x, acc);
    if (i + depth < ns) {
      wait_lgkm0();  // the slot's fragments are in registers
      asm volatile("" ::: "memory");
      Q::load(src, ring0 + sl * Q::SLOT, slice + depth * W, lane);
    }
    sl = sl + 1 < depth ? sl + 1 : 0;
  }

  // partial sums into the wave's own ring (its slots are read), blocks of 1 KB
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int c = 0; c < Q::NB; ++c)
      *(f32x4*)(ring + (a * Q::NB + c) * 1024 + 16 * lane) = acc[a][c];
  __syncthreads();

  const EpiArgs E = epi_args(p);
  char* const yb = (char*)mt.y + (long long)b * mt.y_bstride * esz;
  if (!mt.y) return;
#pragma unroll
  for (int i = 0; i < FIN; ++i) {
    const int ob = wave + i * W;
    if (ob >= OB) break;
    const int a = ob / NT, c = ob % NT;
    f32x4 v[Q::NW];
#pragma unroll
    for (int h = 0; h < Q::NW; ++h) {
      const char* red = lds + (a * Q::NB + h * NT + c) * 1024 + 16 * lane;
      v[h] = *(const f32x4*)red;
#pragma unroll
      for (int w = 1; w < W; ++w) v[h] += *(const f32x4*)(red + w * depth * Q::SLOT);
    }
    float rs[Q::NW];
#pragma unroll
    for (int h = 0; h < Q::NW; ++h) rs[h] = FMT == kQ8 ? scale_of(rsc[i][h], SF16) : 1.0f;
    const int n = n0 + 16 * c + l16;
    if (n >= mt.n_store) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * a + 4 * lk + r;
      if (m >= p.m) continue;
      float o = 0.0f;
      if (n < mt.n) {
        o = gemm_epilogue(E, p.m_base + m, n, v[0][r] * rs[0]);
        if constexpr (PAIR) o = silu(o) * gemm_epilogue(E, p.m_base + m, n, v[1][r] * rs[1]);
        o += yf32 ? as_f32(res[i][r]) : (float)__builtin_bit_cast(f16, (uint16_t)res[i][r]);
      }
      const long long yi = out_index(p, mt, m, n);
      if (yf32)
        ((float*)yb)[yi] = o;
      else
        ((f16*)yb)[yi] = (f16)o;
    }
  }
}

// An entry of a table of instantiations.
#define QMMK_ENTRY(FMT, G, SF16, FD, MT, NT, W, PAIR, RMS, RAG)          \
  QmmkEntry {                                                           \
    QmmkConfig{FMT, G, SF16, FD, MT, NT, W, PAIR, RMS, RAG},             \
        &qmmk_kernel<FMT, G, SF16, FD, MT, NT, W, PAIR, RMS, RAG>,       \
        QmmK<FMT, G, SF16, FD, MT, NT, PAIR, RMS, RAG>::SLOT             \
  }

}  // namespace aexq
