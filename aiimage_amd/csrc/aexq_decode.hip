// Decode-step kernels around the quantized linears (gfx950): the tied Q8 token
// embedding, RoPE with KV-cache append, GQA decode attention over an fp16 KV
// cache (split over positions, the splits merged by the last one to finish),
// and a standalone RMSNorm.
//
// Reference semantics (paths relative to the reference root):
//   embedding gather   Qwen35SharedTokenEmbeddingWeights.cs:185-198, BT:13-26
//   RoPE (rotate-half) AexisKernels.Pack4PointwiseNorm.hlsl:414-473
//   SDPA               AexisKernels.Pack4Matmul.hlsl:420-544 (scale, max-subtracted
//                      softmax divided by max(sum, 1e-20), GQA key head = head / group)
#include <math.h>

#include <type_traits>

#include "aexq_device.hpp"

namespace aexq {

// ---------------------------------------------------------------------------
// Embedding: out[m][d] = fp16(q[tok_m][d] * scale[tok_m]) from the device Q8
// copy (bytes hold q + 128).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void embed_q8_kernel(const uint32_t* codes,
                                                            const void* scales, int scale_f16,
                                                            int k, const int32_t* tokens,
                                                            int vocab, f16* out) {
  const int m = blockIdx.x;
  int tok = tokens[m];
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  const float s = load_scale(scales, tok, scale_f16 != 0);
  const uint8_t* row = (const uint8_t*)codes + (long long)tok * k;
  for (int d = threadIdx.x; d < k; d += kThreads)
    out[(long long)m * k + d] = (f16)((float)((int)row[d] - 128) * s);
}

hipError_t embed_q8_launch(const uint32_t* codes, const void* scales, int scale_f16, int k,
                           const int32_t* tokens, int m, int vocab, void* out,
                           hipStream_t stream) {
  hipLaunchKernelGGL(embed_q8_kernel, dim3(m), dim3(kThreads), 0, stream, codes, scales,
                     scale_f16, k, tokens, vocab, (f16*)out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// RoPE + KV append for one decode position.  q [hq][d], k/v [hkv][d] (fp16,
// rows contiguous); caches [hkv][cap][d].  cos/sin hold the position's
// d/2 table entries (fp32).  One workgroup per head (q heads, then kv heads);
// q is rotated in place, k is rotated into the cache, v is copied.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void rope_kv_kernel(f16* q, const f16* k, const f16* v,
                                                           f16* kcache, f16* vcache, int hq,
                                                           int hkv, int d, int cap, int pos,
                                                           const float* cosv,
                                                           const float* sinv) {
  const int head = blockIdx.x;
  const int half = d / 2;
  for (int j = threadIdx.x; j < half; j += kThreads) {
    const float c = cosv[j], s = sinv[j];
    if (head < hq) {
      f16* row = q + (long long)head * d;
      const float x0 = (float)row[j], x1 = (float)row[j + half];
      row[j] = (f16)(x0 * c - x1 * s);
      row[j + half] = (f16)(x0 * s + x1 * c);
    } else {
      const int g = head - hq;
      const f16* kr = k + (long long)g * d;
      const float x0 = (float)kr[j], x1 = (float)kr[j + half];
      f16* kc = kcache + ((long long)g * cap + pos) * d;
      kc[j] = (f16)(x0 * c - x1 * s);
      kc[j + half] = (f16)(x0 * s + x1 * c);
      const f16* vr = v + (long long)g * d;
      f16* vc = vcache + ((long long)g * cap + pos) * d;
      vc[j] = vr[j];
      vc[j + half] = vr[j + half];
    }
  }
}

hipError_t rope_kv_launch(void* q, const void* k, const void* v, void* kcache, void* vcache,
                          int hq, int hkv, int d, int cap, int pos, const float* cosv,
                          const float* sinv, hipStream_t stream) {
  hipLaunchKernelGGL(rope_kv_kernel, dim3(hq + hkv), dim3(kThreads), 0, stream, (f16*)q,
                     (const f16*)k, (const f16*)v, (f16*)kcache, (f16*)vcache, hq, hkv, d, cap,
                     pos, cosv, sinv);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// GQA decode attention in one launch.  Workgroup (kv head g, split c) covers
// `per` positions (a multiple of 64) of the `len` cached ones for the G = hq /
// hkv query heads of g, so every cached K and V row is read once.  Its waves
// (four or eight) run by themselves, 16 positions of each 64 per wave, with a running
// maximum each and no barrier until the end:
//   scores   lanes 4i..4i+3 own position i of the wave's 16, lane 4i + j the
//            dims 32 r + 8 j + [0, 8) for r < 4 (so one load instruction covers
//            64 contiguous bytes of 16 rows), for all G heads (v_dot2 with fp32
//            accumulation, quad reduction by DPP);
//   softmax  running max / sum per head over the wave's positions (DPP rows,
//            then across rows);
//   P V      lane group g4 = l / 16 owns positions 4 g4 + j, whose weights sit in
//            its own DPP row (row_newbcast), lane l the dims 8 (l % 16) + [0, 8):
//            four 16-byte loads cover the wave's 16 rows.
// The next pass's K and V rows are requested before the current ones'
// products (eight waves for splits of more than one four-wave pass), and q
// (rotated here when RoPE is fused) meets K after one barrier.
// The waves' (max, sum, acc) meet in LDS; the split's go to part[h][split].
// The last workgroup of kv head g to finish (a device-scope counter that the
// same workgroup resets to 0, so the launch needs no clearing and replays
// inside a graph) merges the splits of its G heads:
//   M = max m_s, L = sum l_s e^(m_s - M), out = sum acc_s e^(m_s - M) / max(L, 1e-20).
// That merge reads splits x G rows of 528 bytes through one CU, so a long cache
// takes longer splits rather than more of them (attn_splits): with 64 positions
// a split, 16 heads over 4 x 16384 positions (32 MB) took 21.0 us, half of them
// in the merge, now 12.5 with the rows in the last-level cache (5 us at the rate
// that gives); on caches in turn, whose rows come from HBM, 22.5 -> 13.3; the
// first pass over rows just written, 62 -> 51.  Up to 64 positions there is one
// split and nothing to merge (7.4 -> 5.0 us).
// head_dim == 128.
// ---------------------------------------------------------------------------
constexpr int kAttnDim = 128;

// Device-coherent (agent scope) fp32 store / load: written through to, and
// read from, the level all XCDs share.
__device__ __forceinline__ void store_coherent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_coherent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
constexpr int kAttnPos = 64;         // positions of a four-wave pass
constexpr int kAttnStride = kAttnDim + 4;  // partial row: max, sum, 2 pad, acc[128] (16-byte aligned)
constexpr int kCoherentAux = 16;     // buffer-load cache policy sc1: read at agent coherence
// One counter per 256-byte line: atomics to one line are serialized where they
// are performed (about 15 ns each), so the kv heads' counters do not share one.
constexpr int kAttnCounterStride = 64;
constexpr int kAttnMaxSplits = 96;   // combine staging in LDS
constexpr int kAttnMaxLen = 32768;   // positions a launch takes

// LDS of a workgroup of W waves.
template <int G, int W>
struct AttnLds {
  // P V sums: the waves of a split, then the merge's row groups
  alignas(16) float pv[2 * W][G][kAttnDim];
  alignas(16) f16 qs[G][kAttnDim];
  alignas(16) f16 kn[kAttnDim];
  alignas(16) f16 vn[kAttnDim];
  float wm[W][G], wl[W][G];
  float cm[G * kAttnMaxSplits];  // split maxima, then weights
  float cl[G * kAttnMaxSplits];  // split sums
  float hl[G];
  int last;
};

// Passes of a split, where the launch knows them: one, several, or either (a
// device-side position).  Code for one pass alone starts sooner: 16/4 heads at
// 1024 positions 6.5 us with both forms in the kernel, 6.3 with one.
enum AttnPasses { kOnePass, kManyPasses, kAnyPasses };

template <int G, int W, AttnPasses PASSES>
__device__ __forceinline__ void attn_decode(
    AttnLds<G, W>& lds, const f16* q, const f16* kcache, const f16* vcache, int cap, int len,
    float scale, int splits, float* part, int* counters, f16* out, const f16* knew, const f16* vnew,
    f16* kcache_w, f16* vcache_w, const float* cosv, const float* sinv) {
  const int g = blockIdx.x, c = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  constexpr int half = kAttnDim / 2;
  constexpr int T = 64 * W;     // threads
  constexpr int P = 16 * W;     // positions of one pass
  constexpr int RG = T / 32;    // row groups of the merge
  // positions per split: the live length over the grid's splits
  const int per = PASSES == kOnePass ? P : ((len + splits - 1) / splits + P - 1) / P * P;
  const int live_splits = (len + per - 1) / per;
  const int p0 = c * per, p1 = min(p0 + per, len);
  const int pl = t >> 2, qq = t & 3;  // scores: position p0 + pl of a pass, dims 32 r + 8 qq ..
  const bool rope = knew != nullptr;
  const int pos = len - 1;             // the appended position when RoPE is fused
  const bool has_new = rope && pos >= p0 && pos < p0 + per;
  const long long head_off = (long long)g * cap * kAttnDim;
  auto& pv = lds.pv;
  auto& wm = lds.wm;
  auto& wl = lds.wl;
  int& last = lds.last;
  if (c >= live_splits) {
    // a split past the live length (the grid was sized for the capacity):
    // nothing to score, but it still counts in so the merge starts once
    if (t == 0) last = atomicAdd(&counters[g * kAttnCounterStride], 1) == splits - 1;
    __syncthreads();
    if (!last) return;
  } else {

    // 1. loads, all issued before the first wait; q and the new row first, so
    // that waiting for them leaves the K/V loads in flight.  Absent tables and
    // rows come through empty buffer resources (they read 0).
    constexpr int QI = (G * half + T - 1) / T;  // (head, j) pairs per thread
    float qa[QI], qb[QI], cs[QI], sn[QI];
    const __amdgpu_buffer_rsrc_t trs_c = __builtin_amdgcn_make_buffer_rsrc(
        (void*)cosv, (short)0, rope ? half * 4 : 0, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t trs_s = __builtin_amdgcn_make_buffer_rsrc(
        (void*)sinv, (short)0, rope ? half * 4 : 0, kBufferRsrcWord3);
#pragma unroll
    for (int r = 0; r < QI; ++r) {
      const int i = min(t + r * T, G * half - 1);
      const int h = i / half, j = i % half;
      const f16* qr = q + ((long long)g * G + h) * kAttnDim;
      qa[r] = (float)qr[j];
      qb[r] = (float)qr[j + half];
      cs[r] = as_f32(__builtin_amdgcn_raw_buffer_load_b32(trs_c, j * 4, 0, 0));
      sn[r] = as_f32(__builtin_amdgcn_raw_buffer_load_b32(trs_s, j * 4, 0, 0));
    }
    const int jn = t & (half - 1);
    const __amdgpu_buffer_rsrc_t nrs_k = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(rope ? knew + (long long)g * kAttnDim : q), (short)0, has_new ? kAttnDim * 2 : 0,
        kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t nrs_v = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(rope ? vnew + (long long)g * kAttnDim : q), (short)0, has_new ? kAttnDim * 2 : 0,
        kBufferRsrcWord3);
    const uint32_t kn0 = __builtin_amdgcn_raw_buffer_load_b16(nrs_k, jn * 2, 0, 0);
    const uint32_t kn1 = __builtin_amdgcn_raw_buffer_load_b16(nrs_k, (jn + half) * 2, 0, 0);
    const uint32_t vn0 = __builtin_amdgcn_raw_buffer_load_b16(nrs_v, jn * 2, 0, 0);
    const uint32_t vn1 = __builtin_amdgcn_raw_buffer_load_b16(nrs_v, (jn + half) * 2, 0, 0);
    const float tc = as_f32(__builtin_amdgcn_raw_buffer_load_b32(trs_c, jn * 4, 0, 0));
    const float ts = as_f32(__builtin_amdgcn_raw_buffer_load_b32(trs_s, jn * 4, 0, 0));
    __builtin_amdgcn_sched_barrier(0);  // keeps the q-side loads ahead of K and V
    // K rows of the split (rows >= len read 0): position p0 + pl, 64 bytes per lane
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kcache + head_off), (short)0, len * kAttnDim * 2, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(vcache + head_off), (short)0, len * kAttnDim * 2, kBufferRsrcWord3);
    // K: position q0 + pl of the P from q0, 64 bytes per lane; V: wave w's 16
    // positions, lane group g4 rows 4 g4 + j, dims 8 (lane % 16) ..
    const int g4 = lane >> 4, d8 = lane & 15;
    struct Rows {
      u32x4 k[4], v[4];
    };
    auto fetch = [&](int q0, Rows& r) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r.k[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               krs, (q0 + pl) * 256 + i * 64 + qq * 16, 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j)
        r.v[j] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       vrs, (q0 + 16 * wave + 4 * g4 + j) * 256 + d8 * 16, 0, 0));
    };
    Rows cur, nxt;
    fetch(p0, cur);

    // 2. q of the G heads (rotated and rounded to fp16 when RoPE is fused) and,
    // in the split that holds it, the appended K/V row
    auto& qs = lds.qs;
    auto& kn = lds.kn;
    auto& vn = lds.vn;
#pragma unroll
    for (int r = 0; r < QI; ++r) {
      const int i = t + r * T;
      if (i < G * half) {
        const int h = i / half, j = i % half;
        qs[h][j] = rope ? (f16)(qa[r] * cs[r] - qb[r] * sn[r]) : (f16)qa[r];
        qs[h][j + half] = rope ? (f16)(qa[r] * sn[r] + qb[r] * cs[r]) : (f16)qb[r];
      }
    }
    if (has_new && t < half) {
      const float x0 = (float)__builtin_bit_cast(f16, (uint16_t)kn0);
      const float x1 = (float)__builtin_bit_cast(f16, (uint16_t)kn1);
      const f16 k0 = (f16)(x0 * tc - x1 * ts), k1 = (f16)(x0 * ts + x1 * tc);
      const f16 v0 = __builtin_bit_cast(f16, (uint16_t)vn0);
      const f16 v1 = __builtin_bit_cast(f16, (uint16_t)vn1);
      kn[t] = k0;
      kn[t + half] = k1;
      vn[t] = v0;
      vn[t + half] = v1;
      f16* kc = kcache_w + head_off + (long long)pos * kAttnDim;
      f16* vc = vcache_w + head_off + (long long)pos * kAttnDim;
      kc[t] = k0;
      kc[t + half] = k1;
      vc[t] = v0;
      vc[t + half] = v1;
    }
    __syncthreads();
    // 3. the split's positions, P at a time; every wave keeps its own running
    // maximum, sum and accumulators
    float mx[G], sm[G], ac[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
      mx[h] = -INFINITY;
      sm[h] = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ac[h][e] = 0.0f;
    }
    auto take = [&](int q0, Rows& r, auto first) {
      constexpr bool FIRST = decltype(first)::value;
      if (has_new && q0 + P > pos) {
        // the cache row at `pos` was loaded before it was written: take the new one
        if (q0 + pl == pos) {
#pragma unroll
          for (int i = 0; i < 4; ++i) r.k[i] = *(const u32x4*)&kn[i * 32 + qq * 8];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (q0 + 16 * wave + 4 * g4 + j == pos) r.v[j] = *(const u32x4*)&vn[8 * d8];
      }
      if (q0 + 16 * wave < p1) {  // the wave's first position is live
        const bool live = q0 + pl < len;
        float sc[G];
#pragma unroll
        for (int h = 0; h < G; ++h) {
          float acc = 0.0f;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const u32x4 qw = *(const u32x4*)&qs[h][i * 32 + qq * 8];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = dot2(r.k[i][e], qw[e], acc);
          }
          sc[h] = acc;
        }
#pragma unroll
        for (int h = 0; h < G; ++h) sc[h] += dpp<0xB1>(sc[h]);  // quad_perm [1,0,3,2]
#pragma unroll
        for (int h = 0; h < G; ++h) {
          sc[h] += dpp<0x4E>(sc[h]);  // quad_perm [2,3,0,1]
          sc[h] = live ? sc[h] * scale : -INFINITY;
        }
        float ex[G], mx0[G];
#pragma unroll
        for (int h = 0; h < G; ++h) {
          // maximum over the wave's 16 positions: within DPP rows, then across
          float m = fmaxf(sc[h], dpp<0x124>(sc[h]));
          m = fmaxf(m, dpp<0x128>(m));
          m = fmaxf(m, dpp_rows<0x142, 0xA>(m, m));
          m = fmaxf(m, dpp_rows<0x143, 0xC>(m, m));
          mx0[h] = mx[h];
          mx[h] = fmaxf(mx0[h], lane_value(m, 63));
          // (scores that are all -inf so far weigh 0, not NaN)
          const float base = mx[h] == -INFINITY ? 0.0f : mx[h];
          ex[h] = live ? __expf(sc[h] - base) : 0.0f;
          float s = ex[h] + dpp<0x124>(ex[h]);
          s += dpp<0x128>(s);
          // what came before, on the new maximum (nothing in the first pass)
          const float corr = FIRST ? 0.0f : __expf(mx0[h] - base);
          sm[h] = fmaf(sm[h], corr, s);  // of the lane's own row until the end
          if constexpr (!FIRST) {
#pragma unroll
            for (int e = 0; e < 8; ++e) ac[h][e] *= corr;
          }
        }
        // rows past the end read 0 and weigh 0
        auto weigh = [&](int j, float w, int h) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f16x2 vv = as_h2(r.v[j][e]);
            ac[h][2 * e] = fmaf(w, (float)vv[0], ac[h][2 * e]);
            ac[h][2 * e + 1] = fmaf(w, (float)vv[1], ac[h][2 * e + 1]);
          }
        };
#pragma unroll
        for (int h = 0; h < G; ++h) {
          weigh(0, dpp<0x150>(ex[h]), h);  // row_newbcast: lane 4 j of the lane's row
          weigh(1, dpp<0x154>(ex[h]), h);
          weigh(2, dpp<0x158>(ex[h]), h);
          weigh(3, dpp<0x15C>(ex[h]), h);
        }
      }
    };
    // a split of one pass, with no rows of a next one on the way
    if (PASSES == kOnePass || (PASSES == kAnyPasses && per == P)) {
      take(p0, cur, std::true_type{});
    } else {
      for (int q0 = p0; q0 < p1; q0 += P) {
        fetch(q0 + P < p1 ? q0 + P : len, nxt);  // past the last row: no traffic
        __builtin_amdgcn_sched_barrier(0);
        take(q0, cur, std::false_type{});
        cur = nxt;
      }
    }

    // 4. over the four rows of the wave, then over the waves in LDS
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float l = sm[h];
      l += dpp_rows<0x142, 0xA>(0.0f, l);
      l += dpp_rows<0x143, 0xC>(0.0f, l);
      if (lane == 63) {
        wm[wave][h] = mx[h];
        wl[wave][h] = l;
      }
      // two sums per swap: halves of the wave, then rows of the halves; row
      // r ends with dims 8 d8 + (0, 2, 1, 3)[r] and that + 4
      float s2[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto r = __builtin_amdgcn_permlane32_swap(f32_bits(ac[h][2 * e]),
                                                        f32_bits(ac[h][2 * e + 1]), false, false);
        s2[e] = as_f32(r[0]) + as_f32(r[1]);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const auto r = __builtin_amdgcn_permlane16_swap(f32_bits(s2[2 * e]), f32_bits(s2[2 * e + 1]),
                                                        false, false);
        pv[wave][h][8 * d8 + 4 * e + (g4 >> 1) + 2 * (g4 & 1)] = as_f32(r[0]) + as_f32(r[1]);
      }
    }
    __syncthreads();
    for (int i = t; i < G * kAttnDim; i += T) {
      const int h = i / kAttnDim, d = i % kAttnDim;
      float m = wm[0][h];
#pragma unroll
      for (int w = 1; w < W; ++w) m = fmaxf(m, wm[w][h]);
      const float base = m == -INFINITY ? 0.0f : m;
      float a = 0.0f, l = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        const float f = __expf(wm[w][h] - base);  // a wave with no live position: 0
        a = fmaf(pv[w][h][d], f, a);
        l = fmaf(wl[w][h], f, l);
      }
      if (splits == 1) {  // nothing to merge
        const float f = __expf(m - m);  // NaN where every score is -inf, as in the merge
        out[((long long)g * G + h) * kAttnDim + d] = (f16)(a * f / fmaxf(l * f, 1e-20f));
        continue;
      }
      float* o = part + ((long long)(g * G + h) * splits + c) * kAttnStride;
      store_coherent(o + 4 + d, a);
      if (d == 0) {
        store_coherent(o, m);
        store_coherent(o + 1, l);
      }
    }
    if (splits == 1) return;

    // 5. the last split of kv head g merges all of them.  Partials travel
    // through device-coherent stores and loads (they bypass the per-XCD L2
    // that plain accesses would leave stale), ordered by waiting for the
    // stores before the counter increment.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) last = atomicAdd(&counters[g * kAttnCounterStride], 1) == splits - 1;
    __syncthreads();
    if (!last) return;
  }
  // Loads of the merge: the split statistics (row t of the G * splits rows
  // (head, split) in registers), then the first chunk of accumulator rows, all
  // in flight together.  Thread (rg = t / 32, dq = t % 32) reads dims 4 dq ..
  // 4 dq + 3 of splits rg + RG j of every head; splits past the last live one
  // are sent out of the buffer range, which reads 0.  Rows keep the grid's
  // pitch (`splits`); only the first live_splits of each head hold partials
  // of this launch.
  const int nsp = live_splits;
  auto& cm = lds.cm;
  auto& cl = lds.cl;
  auto& hl = lds.hl;
  const int rows = G * splits;
  const float* pg = part + (long long)g * rows * kAttnStride;
  const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)pg, (short)0, rows * kAttnStride * 4, kBufferRsrcWord3);
  constexpr int JJ = 16 / G;  // accumulator rows per head and thread in one chunk
  constexpr int kChunk = RG * JJ;
  const int dq = t & 31, rg = t >> 5;
  const float m0 = as_f32(__builtin_amdgcn_raw_buffer_load_b32(prs, t * kAttnStride * 4, 0, kCoherentAux));
  const float l0 = as_f32(__builtin_amdgcn_raw_buffer_load_b32(prs, (t * kAttnStride + 1) * 4, 0, kCoherentAux));
  u32x4 av[G][JJ];
  auto issue = [&](int s0) {
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
      for (int j = 0; j < JJ; ++j) {
        const int s2 = s0 + rg + RG * j;
        const int off = s2 < nsp ? ((h * splits + s2) * kAttnStride + 4 + 4 * dq) * 4 : 0x7FFFFFF0;
        av[h][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, off, 0, kCoherentAux));
      }
  };
  issue(0);
  if (t < rows) {
    const bool ok = t % splits < nsp;
    cm[t] = ok ? m0 : -INFINITY;
    cl[t] = ok ? l0 : 0.0f;
  }
  for (int i = t + T; i < rows; i += T) {
    const bool ok = i % splits < nsp;
    cm[i] = ok ? as_f32(__builtin_amdgcn_raw_buffer_load_b32(prs, i * kAttnStride * 4, 0, kCoherentAux))
               : -INFINITY;
    cl[i] = ok ? as_f32(__builtin_amdgcn_raw_buffer_load_b32(prs, (i * kAttnStride + 1) * 4, 0, kCoherentAux))
               : 0.0f;
  }
  __syncthreads();
  // per head: M = max m_s (each wave reduces the heads h == wave mod W)
  for (int h = wave; h < G; h += W) {
    float m = -INFINITY;
    for (int s2 = lane; s2 < nsp; s2 += 64) m = fmaxf(m, cm[h * splits + s2]);
    m = wave_max(m);
    float l = 0.0f;
    for (int s2 = lane; s2 < nsp; s2 += 64) {
      const float w = __expf(cm[h * splits + s2] - m);
      cm[h * splits + s2] = w;
      l = fmaf(cl[h * splits + s2], w, l);
    }
    l = wave_sum(l);
    if (lane == 0) hl[h] = l;
  }
  __syncthreads();
  float ac[G][4];
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) ac[h][e] = 0.0f;
  for (int s0 = 0;;) {
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
      for (int j = 0; j < JJ; ++j) {
        const int s2 = min(s0 + rg + RG * j, nsp - 1);  // rows past the end loaded 0
        const float w = cm[h * splits + s2];
#pragma unroll
        for (int e = 0; e < 4; ++e) ac[h][e] = fmaf(as_f32(av[h][j][e]), w, ac[h][e]);
      }
    s0 += kChunk;
    if (s0 >= nsp) break;
    issue(s0);
  }
  // the row groups' sums meet in LDS
#pragma unroll
  for (int h = 0; h < G; ++h) {
    const f32x4 v = {ac[h][0], ac[h][1], ac[h][2], ac[h][3]};
    *(f32x4*)&pv[rg][h][4 * dq] = v;
  }
  __syncthreads();
  for (int i = t; i < G * kAttnDim; i += T) {
    const int h = i / kAttnDim, dd = i % kAttnDim;
    float a = 0.0f;
#pragma unroll
    for (int w = 0; w < RG; ++w) a += pv[w][h][dd];
    out[((long long)g * G + h) * kAttnDim + dd] = (f16)(a / fmaxf(hl[h], 1e-20f));
  }
  if (t == 0) counters[g * kAttnCounterStride] = 0;  // ready for the next launch
}

template <int G, int W, AttnPasses PASSES>
__global__ __launch_bounds__(64 * W) void attn_decode_kernel(
    const f16* q, const f16* kcache, const f16* vcache, int cap, int len, float scale,
    int splits, float* part, int* counters, f16* out, const f16* knew, const f16* vnew,
    f16* kcache_w, f16* vcache_w, const float* cosv, const float* sinv, const int* posp) {
  __shared__ AttnLds<G, W> lds;
  if (posp) {
    // decode position in device memory (a captured graph advances it): the
    // grid covers the cache capacity, the tables hold [cap][half] rows
    const int pp = min(max(*posp, 0), cap - 1);
    len = __builtin_amdgcn_readfirstlane(pp + 1);
    cosv += (long long)pp * (kAttnDim / 2);
    sinv += (long long)pp * (kAttnDim / 2);
  }
  if constexpr (W == 8 && PASSES == kAnyPasses) {
    // The capacity asks for eight waves, the live length for no more than one
    // four-wave pass per split: the upper waves end here (a barrier waits only
    // for waves that have not ended) and the others do what a launch for that
    // length does.  16/4 heads, capacity 4096: 6.5 us at 256 live positions and
    // 6.7 at 1024, where eight waves of one pass took 7.7 (two waves a SIMD, and
    // twice as many to merge in LDS); at 4096 live 7.9.
    if (len <= kAttnPos * splits) {
      if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= 4) return;
      attn_decode<G, 4, kOnePass>(reinterpret_cast<AttnLds<G, 4>&>(lds), q, kcache, vcache, cap, len,
                                  scale, splits, part, counters, out, knew, vnew, kcache_w, vcache_w,
                                  cosv, sinv);
      return;
    }
  }
  attn_decode<G, W, PASSES>(lds, q, kcache, vcache, cap, len, scale, splits, part, counters, out,
                            knew, vnew, kcache_w, vcache_w, cosv, sinv);
}

// ---------------------------------------------------------------------------
// End of a decode step (Qwen35DecoderSession.Generate, DEC:1160-1237: the
// argmax becomes the next input token and the position advances), done on the
// device so that one captured step replays token after token.
// ---------------------------------------------------------------------------
__global__ void decode_advance_kernel(int* position, int* token, const int* argmax,
                                      int* tokens_out, int out_cap) {
  const int pos = *position;
  const int tok = *argmax;
  if (tokens_out && pos >= 0 && pos < out_cap) tokens_out[pos] = tok;
  *token = tok;
  *position = pos + 1;
}

hipError_t decode_advance_launch(int* position, int* token, const int* argmax, int* tokens_out,
                                 int out_cap, hipStream_t stream) {
  hipLaunchKernelGGL(decode_advance_kernel, dim3(1), dim3(1), 0, stream, position, token, argmax,
                     tokens_out, out_cap);
  return hipGetLastError();
}

// Splits per kv head of a launch over len positions: 64 positions each as long
// as that keeps the merge short, then longer ones, past 4096 positions about a
// workgroup of eight waves per CU.  Measured (us on rotated caches, so K and V
// come from HBM; heads_q / heads_kv, splits at most 16, 32, 64; with 64 positions
// a split always): 16/4 at 4000 10.5, 8.2, 8.9 (8.7), at 16384 21.5, 14.7, 13.3
// (22.6); 4/4 at 4000 8.4, 6.9, 6.6 (6.6); 32/8 at 8192 14.8, 12.8, 15.8 (18.4);
// 32/16 at 8192 17.5, 20.5, 24.1 (20.8).  64/16 at 3000 takes 11.9 with 12 splits
// and 13.9 with 24.  One query head a kv head merges a quarter of that, so on
// eight kv heads the many short splits stay the better ones for longer: 8/8 at
// 6000 9.3 against 9.8, at 7000 11.1 against 10.5.
int attn_splits(int len, int heads_kv, int group) {
  const int s = (len + kAttnPos - 1) / kAttnPos;
  if (group == 1 && heads_kv > 4 && heads_kv <= 8 && len <= kAttnPos * kAttnMaxSplits) return s;
  const int chip = heads_kv < 256 ? 256 / heads_kv : 1;
  int most = 64;
  if (group >= 4 && len <= 4096) most = 32;
  if (len > (group >= 4 ? 2048 : 4096) && most > chip) most = chip;
  return s < most ? s : most;
}
// The number turns back at 4097 positions, so the scratch is sized for the most
// that any length up to len takes: one run at the longest length then covers
// the shorter ones that a caller captures later.
int attn_most_splits(int len) {
  const int s = (len + kAttnPos - 1) / kAttnPos;
  return s < kAttnMaxSplits ? s : kAttnMaxSplits;
}
int attn_max_len() { return kAttnMaxLen; }
int attn_part_stride() { return kAttnStride; }
int attn_counter_stride() { return kAttnCounterStride; }

hipError_t attn_decode_launch(const void* q, const void* kcache, const void* vcache, int hq,
                              int hkv, int cap, int len, float scale, float* part, int* counters,
                              void* out, const void* knew, const void* vnew, const float* cosv,
                              const float* sinv, const int* posp, hipStream_t stream) {
  const int group = hq / hkv;
  // a device-side position: the grid covers the capacity, the kernel reads
  // the live length
  if (posp) len = cap;
  const int splits = attn_splits(len, hkv, group);
  if (len > kAttnMaxLen || splits < 1 || splits > kAttnMaxSplits) return hipErrorInvalidValue;
  const dim3 grid(hkv, splits);
  // longer splits take eight waves: twice the rows on the way to each CU
  const bool wide = len > kAttnPos * splits;
#define AEXQ_ATTN_W(G, W, PASSES)                                                                \
  hipLaunchKernelGGL((attn_decode_kernel<G, W, PASSES>), grid, dim3(64 * W), 0, stream, (const f16*)q, \
                     (const f16*)kcache, (const f16*)vcache, cap, len, scale, splits, part,      \
                     counters, (f16*)out, (const f16*)knew, (const f16*)vnew, (f16*)kcache,      \
                     (f16*)vcache, cosv, sinv, (const int*)posp)
#define AEXQ_ATTN(G)                                                        \
  if (!wide) AEXQ_ATTN_W(G, 4, kOnePass);                                   \
  else if (posp) AEXQ_ATTN_W(G, 8, kAnyPasses);                             \
  else if (len <= 2 * kAttnPos * splits) AEXQ_ATTN_W(G, 8, kOnePass);       \
  else AEXQ_ATTN_W(G, 8, kManyPasses)
  switch (group) {
    case 1: AEXQ_ATTN(1); break;
    case 2: AEXQ_ATTN(2); break;
    case 4: AEXQ_ATTN(4); break;
    case 8: AEXQ_ATTN(8); break;
    default: return hipErrorInvalidValue;
  }
#undef AEXQ_ATTN
#undef AEXQ_ATTN_W
  return hipGetLastError();
}

}  // namespace aexq
