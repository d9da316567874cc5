// The small operators between the quantized matmuls of one decode step, for
// gfx950: RMSNorm, RoPE + KV-cache write, GQA decode attention over an fp16
// KV cache, SiLU(gate) * up, arg-max.  Semantics follow the reference
// kernels (operators/impl/rmsnorm/RMSNorm.cu, attention/FusedRoPEKVWrite.cu,
// attention/Attention.cu): fp32 arithmetic, half-split RoPE with cos / sin
// tables [pos][headDim/2], cache rows [pos][alignedKvDim], position and
// sequence length read from a device buffer so that a captured graph can be
// replayed for the next token.
//
// The attention differs from the reference in structure, not in result: the
// reference runs one workgroup per query head over the whole context (every
// K/V row is read nRep times, scores staged in 8 KB of shared memory).  Here
// a workgroup owns one KV head and chunks of 64 positions, and leaves (max,
// sum, weighted V) partials of its query heads (the usual split-context decode
// attention).  Two kernels do that: attn_rows_kernel (head dimensions 128 and
// 64) keeps K and V in the registers that they are loaded into, 16 positions a
// wave for one, two or four query heads; attn_partial_kernel (the other
// dimensions, and where attn_route says so) stages a chunk in LDS, and its four
// waves are four query heads.  A third, small kernel merges the partials.
// Merging inside the first kernel
// (the workgroup that draws the last ticket of a KV head's counter reads the
// records back; all workgroups of a head placed on one XCD so that records
// and tickets stay in that XCD's L2; no fences) was built and measured: the
// three dependent hops (stores acknowledged, ticket, records read back) cost
// 5.5 us against the 4.5 us of the merge launch (12.8 us against 11.4 us per
// layer), because every dependent memory access costs about a microsecond
// here, in the XCD's own L2 as well.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "gemv_formats.hpp"

namespace cuthip {

__device__ inline float ld_act(const void *p, int f16, size_t i) {
  return f16 ? (float)reinterpret_cast<const half_t *>(p)[i] : reinterpret_cast<const float *>(p)[i];
}
__device__ inline void st_act(void *p, int f16, size_t i, float v) {
  if (f16)
    reinterpret_cast<half_t *>(p)[i] = (half_t)v;
  else
    reinterpret_cast<float *>(p)[i] = v;
}
// Exchange with lane ^ O across the wave: rotations inside a row of 16 once the larger groups hold equal values, so in the
// order 32, 16, 8, ... only, with every lane active.  With six trips through the LDS crossbar per fold, and one per record
// for the weights of the attention merge, a decode step of an 8B shape took 1907 us at position 15,999 (now 1852), 1522 at
// 2047 (1513).
template <class F> __device__ __forceinline__ float wave_fold(float v, F f) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  const auto r32 = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  const uint32_t a0 = r32[0], a1 = r32[1];
  const uint32_t c = __builtin_bit_cast(uint32_t, f(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1)));
  const auto r16 = __builtin_amdgcn_permlane16_swap(c, c, false, false);
  const uint32_t e0 = r16[0], e1 = r16[1];
  v = f(__builtin_bit_cast(float, e0), __builtin_bit_cast(float, e1));
  auto ror = [](float x, auto ctrl) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  v = f(v, ror(v, std::integral_constant<int, 0x128>{}));
  v = f(v, ror(v, std::integral_constant<int, 0x124>{}));
  v = f(v, ror(v, std::integral_constant<int, 0x122>{}));
  return f(v, ror(v, std::integral_constant<int, 0x121>{}));
}
__device__ __forceinline__ float wave_sum(float v) { return wave_fold(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float wave_max(float v) { return wave_fold(v, [](float a, float b) { return fmaxf(a, b); }); }

// ---- RMSNorm: out = x * rsqrt(mean(x^2) + eps) * weight; one workgroup per row ----
// A thread owns groups of 8 consecutive elements; up to kNormGroups of them stay in registers between the two
// passes and all their loads are issued before the first use (a decode row is a few KB: one memory round trip).
constexpr int kNormGroups = 4;   // 256 threads x 8 elements x 4 = rows of up to 8192 elements without a re-read

// vec_ok: the row allows 16-byte loads; otherwise (or in the last, short group) the up to 8 elements are loaded singly
template <bool F16> __device__ inline void ld8(const void *p, size_t i, uint32_t n_left, bool vec_ok, float (&v)[8]) {
  if (vec_ok && n_left >= 8) {
    if (F16) {
      half8_t h = *reinterpret_cast<const half8_t *>(reinterpret_cast<const half_t *>(p) + i);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (float)h[e];
    } else {
      f32x4 a = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(p) + i);
      f32x4 b = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(p) + i + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (uint32_t)e < n_left ? ld_act(p, F16, i + e) : 0.0f;
  }
}

// Rows whose x, weight and out allow 16-byte accesses, of up to 2048 NG elements in groups of eight.  Bound: latency (a few
// rows) or HBM (thousands).  The weights are requested together with x and wait in registers: requested behind the
// reduction they cost a second memory round trip.  Four layers of 8 rows with 4096
// elements 291 -> 268 us (8 norms), eight layers of 300 rows with 2048 1121 -> 1097 (16).
template <bool XF16, bool OF16, int NG>
__global__ void __launch_bounds__(256) rmsnorm8_kernel(const void *x, const float *weight, void *out, uint32_t dim,
                                                       uint32_t stride, float eps) {
  __shared__ float red[4];
  const uint32_t tid = threadIdx.x;
  const size_t off = (size_t)blockIdx.x * stride;
  float v[NG][8], w[NG][8];
  // threads past the end repeat the last group and drop it: no condition around a load
#pragma unroll
  for (int g = 0; g < NG; ++g) ld8<XF16>(x, off + min((g * 256 + tid) * 8, dim - 8), 8, true, v[g]);
#pragma unroll
  for (int g = 0; g < NG; ++g) ld8<false>(weight, min((g * 256 + tid) * 8, dim - 8), 8, true, w[g]);
  float s = 0.0f;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    float t = s;
#pragma unroll
    for (int e = 0; e < 8; ++e) t = fmaf(v[g][e], v[g][e], t);
    s = (g * 256 + tid) * 8 < dim ? t : s;
  }
  s = wave_sum(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  const float total = red[0] + red[1] + red[2] + red[3];
  const float scale = 1.0f / sqrtf(total / (float)dim + eps);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const uint32_t i = (g * 256 + tid) * 8;
    if (i >= dim) break;
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = v[g][e] * scale * w[g][e];
    if constexpr (OF16) {
      half8_t h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = (half_t)r[e];
      *reinterpret_cast<half8_t *>(reinterpret_cast<half_t *>(out) + off + i) = h;
    } else {
      float *o = reinterpret_cast<float *>(out) + off + i;
      *reinterpret_cast<f32x4 *>(o) = f32x4{r[0], r[1], r[2], r[3]};
      *reinterpret_cast<f32x4 *>(o + 4) = f32x4{r[4], r[5], r[6], r[7]};
    }
  }
}

template <bool XF16, bool OF16>
__global__ void __launch_bounds__(256) rmsnorm_kernel(const void *x, const float *weight, void *out, uint32_t dim,
                                                      uint32_t stride, float eps, int aligned) {
  __shared__ float red[4];
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  const size_t off = (size_t)row * stride;
  float v[kNormGroups][8];
  float s = 0.0f;
#pragma unroll
  for (int g = 0; g < kNormGroups; ++g) {
    uint32_t i = (g * 256 + tid) * 8;
    if (i < dim) ld8<XF16>(x, off + i, dim - i, aligned != 0, v[g]);   // unaligned rows: element loads
  }
#pragma unroll
  for (int g = 0; g < kNormGroups; ++g) {
    uint32_t i = (g * 256 + tid) * 8;
    if (i < dim)
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf(v[g][e], v[g][e], s);
  }
  for (uint32_t i = kNormGroups * 2048 + tid; i < dim; i += 256) {   // rows longer than the register window
    float t = ld_act(x, XF16, off + i);
    s = fmaf(t, t, s);
  }
  s = wave_sum(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  float total = red[0] + red[1] + red[2] + red[3];
  float scale = 1.0f / sqrtf(total / (float)dim + eps);
  const bool wide = aligned && reinterpret_cast<uintptr_t>(out) % 16 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0;
#pragma unroll
  for (int g = 0; g < kNormGroups; ++g) {
    uint32_t i = (g * 256 + tid) * 8;
    if (i < dim) {
      uint32_t n = min(dim - i, 8u);
      if (wide && n == 8) {   // 16-byte weight loads and output stores
        f32x4 w0 = *reinterpret_cast<const f32x4 *>(weight + i), w1 = *reinterpret_cast<const f32x4 *>(weight + i + 4);
        float r[8] = {v[g][0] * scale * w0.x, v[g][1] * scale * w0.y, v[g][2] * scale * w0.z, v[g][3] * scale * w0.w,
                      v[g][4] * scale * w1.x, v[g][5] * scale * w1.y, v[g][6] * scale * w1.z, v[g][7] * scale * w1.w};
        if (OF16) {
          half8_t h;
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = (half_t)r[e];
          *reinterpret_cast<half8_t *>(reinterpret_cast<half_t *>(out) + off + i) = h;
        } else {
          float *o = reinterpret_cast<float *>(out) + off + i;
          *reinterpret_cast<f32x4 *>(o) = f32x4{r[0], r[1], r[2], r[3]};
          *reinterpret_cast<f32x4 *>(o + 4) = f32x4{r[4], r[5], r[6], r[7]};
        }
      } else {
        for (uint32_t e = 0; e < n; ++e) st_act(out, OF16, off + i + e, v[g][e] * scale * weight[i + e]);
      }
    }
  }
  for (uint32_t i = kNormGroups * 2048 + tid; i < dim; i += 256)
    st_act(out, OF16, off + i, ld_act(x, XF16, off + i) * scale * weight[i]);
}

// ---- RoPE on q and k, k and v appended to the cache at position params[0] ----
__global__ void __launch_bounds__(256) rope_kv_kernel(const void *q, const void *k, const void *v, int in_f16,
                                                      const uint32_t *params, const float *cosT, const float *sinT,
                                                      half_t *kCache, half_t *vCache, void *qOut, int qout_f16, uint32_t qDim,
                                                      uint32_t kvDim, uint32_t headDim, uint32_t alignedKvDim,
                                                      uint32_t maxPositions) {
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x, halfDim = headDim / 2;
  if (gid >= qDim + 2 * kvDim) return;
  const uint32_t pos = params[0];
  if (pos >= maxPositions) return;   // past the caches and the tables: nothing is read or written
  const float *c = cosT + (size_t)pos * halfDim, *s = sinT + (size_t)pos * halfDim;
  auto rot = [&](const void *src, uint32_t i) {
    uint32_t d = i % headDim;
    if (d < halfDim) return ld_act(src, in_f16, i) * c[d] - ld_act(src, in_f16, i + halfDim) * s[d];
    return ld_act(src, in_f16, i - halfDim) * s[d - halfDim] + ld_act(src, in_f16, i) * c[d - halfDim];
  };
  if (gid < qDim) {
    st_act(qOut, qout_f16, gid, rot(q, gid));
  } else if (gid < qDim + kvDim) {
    uint32_t i = gid - qDim;
    kCache[(size_t)pos * alignedKvDim + i] = (half_t)rot(k, i);
  } else {
    uint32_t i = gid - qDim - kvDim;
    vCache[(size_t)pos * alignedKvDim + i] = (half_t)ld_act(v, in_f16, i);
  }
}

// ---- decode attention, split over the context ----
constexpr int kAttnChunk = 64;    // positions per workgroup (one per lane)
constexpr int kAttnMaxHd = 128;   // head dimension limit (as the reference's sharedQ[128])
constexpr int kAttnRow = kAttnMaxHd + 8;   // LDS row in halfs: +16 bytes keeps the 64 rows off each other's banks

// partial layout per (query head h, split s): [m, l, o[headDim]] floats at ((h * nsplit + s) * (2 + headDim))
// Bound: HBM on long contexts (K and V once), latency on short ones.  Split s takes the 64-position chunks s, s + nsplit,
// s + 2 nsplit, ...: a workgroup that has several keeps (m, l, o) of its heads in registers and requests the next chunk
// while it works on the present one, so that memory does not idle between workgroups and a long context leaves 64
// records per head to merge instead of 256 (attn_splits draws the line).  32 / 8 heads of 128 over 16,384 positions, partials and merge: a chunk
// per workgroup 30.6 us, several 21 (that shape is attn_rows_kernel's now, 18 us).
// HD: the head dimension where it is 128 or 64 (loops over it unroll and their LDS reads overlap), 0 = any
// NG: query heads of a KV head in groups of four (one per wave); gridDim.z covers the heads beyond 4 * NG, each of its
// workgroups with its own reading of K and V (the L2 serves all but one): one KV head of 128 with 71 query heads over 65,536
// positions 143 -> 84 us against one workgroup that went through all heads.
// The arguments that the first loads need (up to and including headDimArg: 14 dwords) lead the list: with
// kernel-argument preloading they arrive in SGPRs with the wave, and the loads of q, K and V wait for no scalar load.
template <int HD, int NG>
__global__ void __launch_bounds__(256) attn_partial_kernel(const void *q, const half_t *kCache, const half_t *vCache,
                                                           const uint32_t *params, uint32_t alignedKvDim, uint32_t maxSeqLen,
                                                           uint32_t nHeads, uint32_t nKvHeads, int q_f16, uint32_t headDimArg,
                                                           float *partial, float scale, uint32_t nsplit) {
  const uint32_t headDim = HD ? (uint32_t)HD : headDimArg;
  constexpr uint32_t kRow = (HD ? HD : kAttnMaxHd) + 8;   // LDS row in halfs: +16 bytes keeps the 64 rows off each other's banks
  __shared__ __attribute__((aligned(16))) half_t Ks[kAttnChunk * kRow];
  __shared__ __attribute__((aligned(16))) half_t Vs[kAttnChunk * kRow];
  __shared__ __attribute__((aligned(16))) float Qs[4 * NG * kAttnMaxHd];
  __shared__ __attribute__((aligned(16))) float Ps[4 * kAttnChunk];
  const uint32_t kvH = blockIdx.x, split = blockIdx.y, nRep = nHeads / nKvHeads, rep0 = blockIdx.z * 4 * NG;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // Every load of the start-up is requested before the first of them is used, so that the kernel begins with one
  // memory round trip: the queries (raw bits, converted later: a conversion right behind the load is a use, and the
  // compiler then waits for it on the spot), then the first chunk of K and V.  Written as a loop with the
  // store right behind each load, the staging waited for four round trips in turn, and the query for two more.
  uint32_t q_raw[NG][2];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const uint32_t rep = rep0 + 4 * g + wave, h = kvH * nRep + (rep < nRep ? rep : 0);
    const size_t qi = (size_t)h * headDim + min(lane, headDim - 1);   // lanes beyond the head dimension read a valid element
    const size_t qj = (size_t)h * headDim + min(lane + 64, headDim - 1);
    if (q_f16) {
      q_raw[g][0] = reinterpret_cast<const uint16_t *>(q)[qi];
      q_raw[g][1] = reinterpret_cast<const uint16_t *>(q)[qj];
    } else {
      q_raw[g][0] = reinterpret_cast<const uint32_t *>(q)[qi];
      q_raw[g][1] = reinterpret_cast<const uint32_t *>(q)[qj];
    }
  }
  // a chunk of K and V in 16-byte pieces, IT per thread.  The first chunk's loads do not wait for the sequence length
  // (every row below the cache capacity is readable); rows past the sequence are zeroed on their way into LDS.
  const uint32_t pieces = headDim / 8, npieces = kAttnChunk * pieces;
  constexpr int IT = kAttnChunk * ((HD ? HD : kAttnMaxHd) / 8) / 256;
  static_assert(HD == 0 || IT * 256 == kAttnChunk * (HD / 8), "one 16-byte piece per thread and round");
  u32x4 kraw[IT], vraw[IT];
  auto fetch = [&](uint32_t t0) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t i = min(tid + 256u * it, npieces - 1), r = i / pieces, c8 = i % pieces;
      const size_t off = (size_t)min(t0 + r, maxSeqLen - 1) * alignedKvDim + kvH * headDim + c8 * 8;
      kraw[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(kCache + off));
      vraw[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(vCache + off));
    }
  };
  uint32_t t0 = split * kAttnChunk;
  fetch(t0);
  __builtin_amdgcn_sched_barrier(0);
  const uint32_t seqLen = min(params[1], maxSeqLen);   // a length beyond the cache capacity attends the capacity only
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (lane + 64 * e < headDim)   // each wave reads only its own queries
        Qs[(4 * g + wave) * kAttnMaxHd + lane + 64 * e] =
            q_f16 ? (float)__builtin_bit_cast(half_t, (uint16_t)q_raw[g][e]) : __builtin_bit_cast(float, q_raw[g][e]);

  float m_run[NG], l_run[NG], o_run[NG][2];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    m_run[g] = -INFINITY;
    l_run[g] = o_run[g][0] = o_run[g][1] = 0.0f;
  }
  for (bool first = true;; first = false) {
    const uint32_t nvalid = t0 < seqLen ? min((uint32_t)kAttnChunk, seqLen - t0) : 0u;   // 0 only in the first chunk
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t i = tid + 256u * it, r = i / pieces, c8 = i % pieces;
      if (HD == 0 && i >= npieces) break;
      const bool past = r >= nvalid;
      *reinterpret_cast<u32x4 *>(Ks + r * kRow + c8 * 8) = past ? u32x4{0, 0, 0, 0} : kraw[it];
      *reinterpret_cast<u32x4 *>(Vs + r * kRow + c8 * 8) = past ? u32x4{0, 0, 0, 0} : vraw[it];
    }
    __syncthreads();   // K, V staged
    const uint32_t t_next = t0 + nsplit * kAttnChunk;
    const bool more = t_next < seqLen;
    if (more) fetch(t_next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g > 0 && rep0 + 4 * g >= nRep) break;
      // score of position t0 + lane: q is read as broadcast 16-byte pieces
      float sc = 0.0f;
      const half_t *krow = Ks + lane * kRow;
      const f32x4 *qv = reinterpret_cast<const f32x4 *>(Qs + (4 * g + wave) * kAttnMaxHd);
#pragma unroll
      for (uint32_t d = 0; d < headDim; d += 8) {
        half8_t k8 = *reinterpret_cast<const half8_t *>(krow + d);
        f32x4 qa = qv[d / 4], qb = qv[d / 4 + 1];
        sc = fmaf(qa.x, (float)k8[0], sc); sc = fmaf(qa.y, (float)k8[1], sc);
        sc = fmaf(qa.z, (float)k8[2], sc); sc = fmaf(qa.w, (float)k8[3], sc);
        sc = fmaf(qb.x, (float)k8[4], sc); sc = fmaf(qb.y, (float)k8[5], sc);
        sc = fmaf(qb.z, (float)k8[6], sc); sc = fmaf(qb.w, (float)k8[7], sc);
      }
      sc = lane < nvalid ? sc * scale : -INFINITY;
      const float mc = wave_max(sc), m = first ? mc : fmaxf(m_run[g], mc);
      const float p = lane < nvalid ? expf(sc - m) : 0.0f;
      const float l = wave_sum(p);
      Ps[wave * kAttnChunk + lane] = p;   // zero for positions past the sequence
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (!first) {
        const float keep = expf(m_run[g] - m);
        l_run[g] *= keep;
        o_run[g][0] *= keep;
        o_run[g][1] *= keep;
      }
      m_run[g] = m;
      l_run[g] += l;
      // weighted V: lane owns the adjacent dims 2 * lane and 2 * lane + 1 (one 4-byte LDS read per position),
      // four weights per 16-byte read; rows past the sequence are zero and carry zero weight.  Heads of 64: lanes
      // 0-31 take the first 32 positions, lanes 32-63 the others, added at the end.
      float o0 = o_run[g][0], o1 = o_run[g][1];
      typedef _Float16 half2v __attribute__((ext_vector_type(2)));
      constexpr uint32_t kSpan = HD == 64 ? kAttnChunk / 2 : kAttnChunk;
      const uint32_t tb = HD == 64 ? (lane >> 5) * kSpan : 0u;
      const f32x4 *pv = reinterpret_cast<const f32x4 *>(Ps + wave * kAttnChunk + tb);
      const half_t *vcol = Vs + tb * kRow + (HD == 64 ? 2 * (lane & 31) : min(2 * lane, (uint32_t)kAttnMaxHd - 2));
#pragma unroll
      for (uint32_t t = 0; t < kSpan; t += 4) {
        f32x4 p4 = pv[t / 4];
        half2v v0 = *reinterpret_cast<const half2v *>(vcol + (t + 0) * kRow);
        half2v v1 = *reinterpret_cast<const half2v *>(vcol + (t + 1) * kRow);
        half2v v2 = *reinterpret_cast<const half2v *>(vcol + (t + 2) * kRow);
        half2v v3 = *reinterpret_cast<const half2v *>(vcol + (t + 3) * kRow);
        o0 = fmaf(p4.x, (float)v0.x, o0); o1 = fmaf(p4.x, (float)v0.y, o1);
        o0 = fmaf(p4.y, (float)v1.x, o0); o1 = fmaf(p4.y, (float)v1.y, o1);
        o0 = fmaf(p4.z, (float)v2.x, o0); o1 = fmaf(p4.z, (float)v2.y, o1);
        o0 = fmaf(p4.w, (float)v3.x, o0); o1 = fmaf(p4.w, (float)v3.y, o1);
      }
      o_run[g][0] = o0;
      o_run[g][1] = o1;
    }
    if (!more) break;
    __syncthreads();   // every wave is done with this chunk
    t0 = t_next;
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    float o0 = o_run[g][0], o1 = o_run[g][1];
    if (HD == 64) {
      o0 += __shfl_xor(o0, 32);
      o1 += __shfl_xor(o1, 32);
    }
    const uint32_t rep = rep0 + 4 * g + wave;
    if (rep >= nRep) continue;
    float *dst = partial + ((size_t)(kvH * nRep + rep) * nsplit + split) * (2 + headDim);
    if (lane == 0) {
      dst[0] = m_run[g];   // -inf for a split past the sequence
      dst[1] = l_run[g];
    }
    if (2 * lane + 1 < headDim) {
      dst[2 + 2 * lane] = o0;
      dst[2 + 2 * lane + 1] = o1;
    }
  }
}

// The same for head dimensions of 128 and 64 and up to four query heads (NH) of a KV head; gridDim.y goes through the groups of NH.
// Bound: HBM on long contexts, latency on short ones.  K and V stay in the registers that they are loaded into: lane = (row of G, piece
// of 8 dimensions).  A wave takes 16 positions of a chunk for its heads; its products of 8 dimensions meet across the lanes of a row in halving
// steps, which leaves each lane the score of one (position, head), so that softmax costs every lane one exponential; the weights
// pass through a strip of LDS that belongs to the wave, and the sums of p V stay in registers until the four waves meet at the
// end.  No barrier in the loop: a wave requests its next 16 positions and works on.  attn_partial_kernel has K and V staged in LDS, two barriers
// a chunk, four waves that read all of both back for one head each, whether there are four heads or one.
// ONE: a chunk per workgroup.  Two copies of the work on a chunk in the loop, one without it: with four (every way out of the loop had its own)
// the kernel was three times as long, and the instruction cache, which six kernels of a layer share, cost 0.2 to 0.4 us a launch.
// Partials and merge, us, graph replay over 600 MB of caches, before -> now (query / KV heads, positions):
//   dimension 128  32 / 32: 64 6.2 -> 5.1, 2500 15.6 -> 11.9, 4096 (64 / 64) 34.3 -> 28.8;  32 / 16: 3000 11.8 -> 9.3, 16,384 34.1 -> 28.3
//                  32 / 8: 64 5.9 -> 5.1, 2048 7.4 -> 7.1, 6000 12.6 -> 10.6, 16,384 21.2 -> 17.7;  32 / 4: 1500 7.8 -> 6.3, 3500 9.1 -> 8.2
//                  64 / 8: 4096 11.6 -> 10.4;  32 / 1: 16,384 17.1 -> 14.2;  6 / 1: 65,536 23.8 -> 16.8
//   dimension 64   32 / 32: 4096 12.1 -> 10.9;  32 / 8: 6000 8.4 -> 7.7;  64 / 8: 4096 8.6 -> 7.8;  16 / 1: 16,384 9.9 -> 8.1
// Against 64 bits 1.2 to 2.4e-7 where that kernel has 2.2 to 7.1e-7 (shorter chains of additions).
template <int HD, int NH, bool ONE>
__global__ void __launch_bounds__(256) attn_rows_kernel(const void *q, const half_t *kCache, const half_t *vCache, const uint32_t *params,
                                                        uint32_t alignedKvDim, uint32_t maxSeqLen, uint32_t nRep, uint32_t nKvHeads,
                                                        int q_f16, uint32_t nsplit, float *partial, float scale) {
  constexpr int LPR = HD / 8, G = 64 / LPR, IT = 16 / G, NV = IT * NH;   // NV scores per lane of a row
  static_assert(kAttnChunk == 4 * 16 && NV <= LPR, "four waves of 16 positions; a lane of a row ends with one score");
  __shared__ __attribute__((aligned(16))) float Ps[4][16][NH];
  __shared__ float Os[4][NH * HD], Ms[4][NH], Ls[4][NH];
  // blockIdx.x: XCD, .y: group of NH query heads, .z: eighths of the (KV head, split) pairs
  const uint32_t pair = blockIdx.z * 8 + blockIdx.x, split = __builtin_amdgcn_readfirstlane(pair / nKvHeads), kvH = pair - split * nKvHeads;
  const uint32_t rep0 = blockIdx.y * NH;
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t piece = lane % LPR, row = lane / LPR;
  if (split >= nsplit) return;   // (the last eight pairs may be fewer)

  // the queries first, then the first positions: one memory round trip for both (attn_partial_kernel)
  u32x4 q_raw[NH][2];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    const size_t qi = (size_t)(kvH * nRep + min(rep0 + h, nRep - 1)) * HD + 8 * piece;
    if (q_f16) {
      q_raw[h][0] = ld_u32x4(reinterpret_cast<const uint8_t *>(q) + 2 * qi);
    } else {
      q_raw[h][0] = ld_u32x4(reinterpret_cast<const uint8_t *>(q) + 4 * qi);
      q_raw[h][1] = ld_u32x4(reinterpret_cast<const uint8_t *>(q) + 4 * qi + 16);
    }
  }
  struct Tile { u32x4 k[IT], v[IT]; } ta, tb;
  auto fetch = [&](Tile &t, uint32_t t0, uint32_t end) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const size_t off = (size_t)min(t0 + 16 * wave + it * G + row, max(end, 1u) - 1) * alignedKvDim + kvH * HD + 8 * piece;
      t.k[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(kCache + off));
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const size_t off = (size_t)min(t0 + 16 * wave + it * G + row, max(end, 1u) - 1) * alignedKvDim + kvH * HD + 8 * piece;
      t.v[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(vCache + off));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  uint32_t t0 = split * kAttnChunk;
  const uint32_t step = nsplit * kAttnChunk;
  fetch(ta, t0, maxSeqLen);
  const uint32_t seqLen = min(params[1], maxSeqLen);   // a length beyond the cache capacity attends the capacity only
  float qv[NH][8];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    if (q_f16) {
      const half8_t x = __builtin_bit_cast(half8_t, q_raw[h][0]);
#pragma unroll
      for (int e = 0; e < 8; ++e) qv[h][e] = (float)x[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) qv[h][e] = __builtin_bit_cast(f32x4, q_raw[h][e / 4])[e % 4];
    }
  }

  auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  // over the positions of a wave: the lane bits 5, 4, 3 and 2 (what is below tells heads apart, or repeats)
  auto fold = [&](float v, auto f) __attribute__((always_inline)) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r32 = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    const uint32_t a0 = r32[0], a1 = r32[1];
    const uint32_t c = __builtin_bit_cast(uint32_t, f(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1)));
    const auto r16 = __builtin_amdgcn_permlane16_swap(c, c, false, false);
    const uint32_t e0 = r16[0], e1 = r16[1];
    v = f(__builtin_bit_cast(float, e0), __builtin_bit_cast(float, e1));
    v = f(v, dpp(v, std::integral_constant<int, 0x128>{}));
    return f(v, dpp(v, std::integral_constant<int, 0x124>{}));
  };

  // the lane's (position, head) after the halving steps: value v = it * NH + head of the row's NV, the same in REP lanes
  constexpr int REP = LPR / NV;
  const uint32_t myRow = piece / REP / NH * G + row, myHead = piece / REP % NH;
  float m_run = -INFINITY, l_run = 0.0f, acc[NH * 8];
#pragma unroll
  for (int i = 0; i < NH * 8; ++i) acc[i] = 0.0f;

  auto use = [&](Tile &t, uint32_t at) __attribute__((always_inline)) {
    const uint32_t first = at + 16 * wave;
    if (first >= seqLen) return;
    const uint32_t nvalid = min(16u, seqLen - first);
    float s[NV];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const half8_t k8 = __builtin_bit_cast(half8_t, t.k[it]);
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        float d = qv[h][0] * (float)k8[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) d = fmaf(qv[h][e], (float)k8[e], d);
        s[it * NH + h] = d;
      }
    }
    // a step leaves a lane half of the values, summed with its mirror image's, then its neighbours'
    auto join = [&](auto nc, auto ctrl, uint32_t bit) __attribute__((always_inline)) {
      constexpr int n = decltype(nc)::value;
      if constexpr (n <= 1) {
        s[0] += dpp(s[0], ctrl);
      } else {
        const bool up = (lane & bit) != 0;
#pragma unroll
        for (int i = 0; i < n / 2; ++i) {
          const float send = up ? s[i] : s[i + n / 2], mine = up ? s[i + n / 2] : s[i];
          s[i] = mine + dpp(send, ctrl);
        }
      }
    };
    constexpr int n1 = LPR == 16 ? NV / 2 : NV, n2 = n1 / 2, n3 = n2 / 2;
    if constexpr (LPR == 16) join(std::integral_constant<int, NV>{}, std::integral_constant<int, 0x140>{}, 8);   // row_mirror
    join(std::integral_constant<int, n1>{}, std::integral_constant<int, 0x141>{}, 4);   // row_half_mirror
    join(std::integral_constant<int, n2>{}, std::integral_constant<int, 0x4E>{}, 2);    // lane ^ 2
    join(std::integral_constant<int, n3>{}, std::integral_constant<int, 0xB1>{}, 1);    // lane ^ 1
    const float sc = myRow < nvalid ? s[0] * scale : -INFINITY;
    const float m = fmaxf(m_run, fold(sc, [](float a, float b) { return fmaxf(a, b); }));
    const float p = sc == -INFINITY ? 0.0f : expf(sc - m);   // zero for positions past the sequence
    Ps[wave][myRow][myHead] = p;
    if (__builtin_amdgcn_ballot_w64(m > m_run) != 0) {
      const float keep = m_run == -INFINITY ? 0.0f : expf(m_run - m);
      l_run *= keep;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, keep), h * REP));
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[8 * h + e] *= f;
      }
    }
    m_run = m;
    l_run += p;
    if (nvalid < 16) {   // what lies past the sequence carries no weight, but an infinity there times zero would be no zero
#pragma unroll
      for (int it = 0; it < IT; ++it)
        if (it * G + row >= nvalid) t.v[it] = u32x4{0, 0, 0, 0};
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const half8_t v8 = __builtin_bit_cast(half8_t, t.v[it]);
      float w[NH];
#pragma unroll
      for (int h = 0; h < NH; ++h) w[h] = Ps[wave][it * G + row][h];
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[8 * h + e] = fmaf(w[h], (float)v8[e], acc[8 * h + e]);
    }
    __builtin_amdgcn_wave_barrier();
  };

  if constexpr (ONE) {
    use(ta, t0);
  } else {
    // the next chunk is requested whether there is one or not (then the last position, again and again): under a condition, the
    // wait for the present one would wait for it too
    for (;;) {
      fetch(tb, t0 + step, seqLen);
      use(ta, t0);
      t0 += step;
      if (t0 >= seqLen) break;
      fetch(ta, t0 + step, seqLen);
      use(tb, t0);
      t0 += step;
      if (t0 >= seqLen) break;
    }
  }

  // the rows of a wave: each step leaves a lane half of the NH * 8 sums
  auto swap_add = [](float a, float b, auto wide) __attribute__((always_inline)) {
    const uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
    uint32_t u, v;
    if constexpr (decltype(wide)::value) {
      const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
      u = r[0]; v = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
      u = r[0]; v = r[1];
    }
    return __builtin_bit_cast(float, u) + __builtin_bit_cast(float, v);
  };
#pragma unroll
  for (int i = 0; i < NH * 4; ++i) acc[i] = swap_add(acc[2 * i], acc[2 * i + 1], std::true_type{});
#pragma unroll
  for (int i = 0; i < NH * 2; ++i) acc[i] = swap_add(acc[2 * i], acc[2 * i + 1], std::false_type{});
  uint32_t idx = 2 * ((lane >> 4) & 1) + (lane >> 5);
  constexpr int LEFT = HD == 128 ? NH * 2 : NH;
  if constexpr (HD == 64) {
    const bool up = (lane & 8) != 0;
#pragma unroll
    for (int i = 0; i < NH; ++i) acc[i] = (up ? acc[2 * i + 1] : acc[2 * i]) + dpp(up ? acc[2 * i] : acc[2 * i + 1], std::integral_constant<int, 0x128>{});
    idx += up ? 4 : 0;
  }
#pragma unroll
  for (int i = 0; i < LEFT; ++i) {
    const uint32_t x = i * (NH * 8 / LEFT) + idx;   // head * 8 + element of the lane's piece
    Os[wave][x / 8 * HD + 8 * piece + x % 8] = acc[i];
  }
  const float l = fold(l_run, [](float a, float b) { return a + b; });
  if (lane < NH * REP) {
    Ms[wave][myHead] = m_run;
    Ls[wave][myHead] = l;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < NH * HD; i += 256) {
    const uint32_t h = i / HD, d = i % HD;
    if (rep0 + h >= nRep) break;
    float M = Ms[0][h], L = 0.0f, o = 0.0f;
#pragma unroll
    for (int w = 1; w < 4; ++w) M = fmaxf(M, Ms[w][h]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = Ms[w][h] == -INFINITY ? 0.0f : expf(Ms[w][h] - M);
      L = fmaf(Ls[w][h], f, L);
      o = fmaf(Os[w][i], f, o);
    }
    float *dst = partial + ((size_t)(kvH * nRep + rep0 + h) * nsplit + split) * (2 + HD);
    if (d == 0) {
      dst[0] = M;   // -inf for a split past the sequence
      dst[1] = L;
    }
    dst[2 + d] = o;
  }
}

// ---- decode attention with few, wide context splits (head dimension 128) ----
// One workgroup per (query head, split), at most kAttnWideSplits splits per head, so that a consumer can fold the
// records of a head while it stages its activations (the output projection, gemv_rows8.hpp) and the merge launch
// disappears.  Split s takes the 64-position chunks s, s + nsplit, s + 2 * nsplit, ...: one chunk per wave and pass,
// so a short sequence in a large cache still spreads over the splits.  Every wave works alone until the end (its own
// K chunk in LDS, V straight from memory into registers: a lane's 16-byte piece of V covers 8 dimensions of one
// position, and the lane multiplies it by that position's weight), then the four waves' (max, sum, o) are folded
// into the one record [max, sum, o[128]] of the split.  The query heads that share a KV head read the same chunk:
// the block index puts them on the same XCD (equal index modulo 8 when nKvHeads * nsplit is a multiple of 8), so
// the chunk crosses the fabric once.
constexpr int kAttnWideSplits = 8;
constexpr size_t kAttnWideLds = 4 * (size_t)kAttnChunk * kAttnRow * 2 + 4 * kAttnChunk * 4 + kAttnMaxHd * 4;

__global__ void __launch_bounds__(256) attn_partial_wide_kernel(const void *q, const half_t *kCache, const half_t *vCache,
                                                                const uint32_t *params, uint32_t alignedKvDim,
                                                                uint32_t maxSeqLen, uint32_t nHeads, uint32_t nKvHeads,
                                                                int q_f16, uint32_t nsplit, float *partial, float scale) {
  constexpr uint32_t HD = 128;
  extern __shared__ __attribute__((aligned(16))) uint8_t wide_lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  half_t *Ks = reinterpret_cast<half_t *>(wide_lds) + (size_t)wave * kAttnChunk * kAttnRow;   // this wave's chunk of K
  float *Pp = reinterpret_cast<float *>(wide_lds + 4 * (size_t)kAttnChunk * kAttnRow * 2) + wave * kAttnChunk;
  float *Qs = reinterpret_cast<float *>(wide_lds + 4 * (size_t)kAttnChunk * kAttnRow * 2 + 4 * kAttnChunk * 4);
  const uint32_t nRep = nHeads / nKvHeads, per_rep = nKvHeads * nsplit;
  const uint32_t rep = blockIdx.x / per_rep, rem = blockIdx.x - rep * per_rep;
  const uint32_t kvH = rem / nsplit, split = rem - kvH * nsplit, h = kvH * nRep + rep;
  const uint32_t grp = lane >> 4, c8 = lane & 15;   // V / K piece of a pass: position 4 * it + grp, dimensions 8 * c8 ..

  // the query (raw bits) and the first pass's chunk of K and V are requested before anything is used; none of these
  // loads waits for the sequence length (every row below the cache capacity is readable, rows past the sequence are
  // masked afterwards)
  uint32_t q_raw = 0u;
  if (tid < HD) q_raw = q_f16 ? (uint32_t)reinterpret_cast<const uint16_t *>(q)[(size_t)h * HD + tid]
                              : reinterpret_cast<const uint32_t *>(q)[(size_t)h * HD + tid];
  float m_run = -INFINITY, l_run = 0.0f, o_run[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o_run[e] = 0.0f;
  uint32_t seqLen = 0u;
  for (uint32_t pass = 0;; ++pass) {
    const uint32_t t0 = (split + nsplit * (wave + 4u * pass)) * (uint32_t)kAttnChunk;
    // pass 0 runs for every wave (its barrier publishes the query); later passes end at the sequence length
    if (pass > 0 && t0 >= seqLen) break;
    u32x4 kr[16], vr[16];
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      const size_t off = (size_t)min(t0 + 4u * it + grp, maxSeqLen - 1) * alignedKvDim + kvH * HD + c8 * 8;
      kr[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(kCache + off));
    }
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      const size_t off = (size_t)min(t0 + 4u * it + grp, maxSeqLen - 1) * alignedKvDim + kvH * HD + c8 * 8;
      vr[it] = ld_u32x4(reinterpret_cast<const uint8_t *>(vCache + off));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (pass == 0) {
      seqLen = min(params[1], maxSeqLen);   // a length beyond the cache capacity attends the capacity only
      if (tid < HD) Qs[tid] = q_f16 ? (float)__builtin_bit_cast(half_t, (uint16_t)q_raw) : __builtin_bit_cast(float, q_raw);
    }
    const uint32_t nvalid = t0 < seqLen ? min((uint32_t)kAttnChunk, seqLen - t0) : 0u;
#pragma unroll
    for (int it = 0; it < 16; ++it) *reinterpret_cast<u32x4 *>(Ks + (4 * it + grp) * kAttnRow + c8 * 8) = kr[it];
    if (pass == 0) __syncthreads();   // the query, and this wave's K
    else {
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // score of position t0 + lane
    float sc = 0.0f;
    const half_t *krow = Ks + lane * kAttnRow;
    const f32x4 *qv = reinterpret_cast<const f32x4 *>(Qs);
#pragma unroll
    for (uint32_t d = 0; d < HD; d += 8) {
      half8_t k8 = *reinterpret_cast<const half8_t *>(krow + d);
      f32x4 qa = qv[d / 4], qb = qv[d / 4 + 1];
      sc = fmaf(qa.x, (float)k8[0], sc); sc = fmaf(qa.y, (float)k8[1], sc);
      sc = fmaf(qa.z, (float)k8[2], sc); sc = fmaf(qa.w, (float)k8[3], sc);
      sc = fmaf(qb.x, (float)k8[4], sc); sc = fmaf(qb.y, (float)k8[5], sc);
      sc = fmaf(qb.z, (float)k8[6], sc); sc = fmaf(qb.w, (float)k8[7], sc);
    }
    sc = lane < nvalid ? sc * scale : -INFINITY;
    const float m_c = wave_max(sc);
    const float pw = lane < nvalid ? expf(sc - m_c) : 0.0f;
    const float l_c = wave_sum(pw);
    // weights to LDS in the order the V pieces want them: group g holds positions g, g + 4, g + 8, ...
    Pp[(lane & 3) * 16 + (lane >> 2)] = pw;
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float o_c[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o_c[e] = 0.0f;
    const f32x4 *pv = reinterpret_cast<const f32x4 *>(Pp + grp * 16);
    // rows past the sequence carry weight zero, but what the cache holds there is anything: masked to zero (only a
    // chunk that the sequence ends in pays for the masks)
    if (nvalid < (uint32_t)kAttnChunk) {
#pragma unroll
      for (int it = 0; it < 16; ++it)
        if (4u * it + grp >= nvalid) vr[it] = u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 p4 = pv[i4];
      const float pj[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const half8_t v8 = __builtin_bit_cast(half8_t, vr[4 * i4 + u]);
#pragma unroll
        for (int e = 0; e < 8; ++e) o_c[e] = fmaf(pj[u], (float)v8[e], o_c[e]);
      }
    }
    // fold the chunk into the wave's running (max, sum, o)
    const float m_new = fmaxf(m_run, m_c);
    const float a = m_run == -INFINITY ? 0.0f : expf(m_run - m_new), b = m_c == -INFINITY ? 0.0f : expf(m_c - m_new);
    l_run = a * l_run + b * l_c;
#pragma unroll
    for (int e = 0; e < 8; ++e) o_run[e] = a * o_run[e] + b * o_c[e];
    m_run = m_new;
    __builtin_amdgcn_wave_barrier();   // the next pass overwrites Ks and Pp
  }
  // the four position groups of the wave hold shares of the same dimensions
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    o_run[e] += __shfl_xor(o_run[e], 16);
    o_run[e] += __shfl_xor(o_run[e], 32);
  }
  // fold the waves: their (max, sum, o) go through LDS (each wave's own K region is free now)
  float *mine = reinterpret_cast<float *>(Ks);
  if (lane < 16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) mine[2 + 8 * lane + e] = o_run[e];
  }
  if (lane == 0) {
    mine[0] = m_run;
    mine[1] = l_run;
  }
  __syncthreads();
  if (tid < HD) {
    const float *w0 = reinterpret_cast<const float *>(wide_lds);
    constexpr size_t kStride = (size_t)kAttnChunk * kAttnRow * 2 / 4;   // floats between the waves' regions
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, w0[w * kStride]);
    float L = 0.0f, o = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = w0[w * kStride];
      const float f = mw == -INFINITY ? 0.0f : expf(mw - M);
      L = fmaf(w0[w * kStride + 1], f, L);
      o = fmaf(w0[w * kStride + 2 + tid], f, o);
    }
    float *dst = partial + ((size_t)h * nsplit + split) * (2 + HD);
    if (tid == 0) {
      dst[0] = M;
      dst[1] = L;
    }
    dst[2 + tid] = o;
  }
}

// One workgroup per query head and 64 dimensions, GROUPS waves: wave g takes the splits g, g + GROUPS, ..., lane d of it dimension d of
// each, and the waves meet in LDS.  Bound: the latency of its loads.  Up to 32 splits: four waves (one, with 32 loads per
// thread, made the step of an 8B shape at position 2047 1513 us instead of 1487).  More: eight (one walked 256 records in
// 13.3 us).  With all dimensions of a head in one workgroup of twice the waves, half of them idle at heads of 64, both launches of
// the attention took, us: 32 / 8 heads of 128 at 2048 positions 6.93 (now 6.83), 16,384 17.89 (17.79); of 64 at 4096 7.14 (6.87); 16 / 1 at 16,384
// 8.24 (7.85).
constexpr int kAttnMaxSplit = 1024;   // splits per head the merge kernel holds weights for

template <int GROUPS>
__global__ void __launch_bounds__(64 * GROUPS) attn_merge_kernel(const float *partial, void *out, int out_f16, uint32_t headDim,
                                                                 uint32_t nsplit) {
  constexpr uint32_t kPre = 8;   // records a thread requests at the start
  constexpr int kPairs = kAttnMaxSplit / (64 * GROUPS);   // (max, sum) pairs per thread where there are many
  __shared__ float Ws[GROUPS < 8 ? 1 : kAttnMaxSplit];
  __shared__ float red[GROUPS], reds[GROUPS];
  __shared__ float os[GROUPS][64];
  const uint32_t h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, g = __builtin_amdgcn_readfirstlane(tid >> 6), d = blockIdx.y * 64 + lane;
  // every split has a record (empty ones carry max = -inf, sum = 0), so the merge does not need the sequence length
  // and its loads do not wait for it
  const uint32_t rec = 2 + headDim;
  const float *base = partial + (size_t)h * nsplit * rec;
  // this thread's dimension of the first splits is requested together with the (max, sum) pairs, so that a merge of up
  // to 32 (64) splits costs one memory round trip instead of three
  float ov[kPre];
#pragma unroll
  for (uint32_t u = 0; u < kPre; ++u) {
    const uint32_t s = g + GROUPS * u;
    ov[u] = (s < nsplit && d < headDim) ? base[(size_t)s * rec + 2 + d] : 0.0f;
  }
  float o = 0.0f, L;
  if (GROUPS < 8 || nsplit <= GROUPS * kPre) {   // fewer groups are launched for up to 32 splits only
    // every wave holds all (max, sum) pairs, one per lane, and folds them by itself: no workgroup barrier; the weight of
    // split s comes out of lane s (threads beyond the head dimension hold zeros)
    const bool have = lane < nsplit;
    const float ms = have ? base[(size_t)lane * rec] : -INFINITY, lsum = have ? base[(size_t)lane * rec + 1] : 0.0f;
    const float M = wave_max(ms);
    const float w = ms == -INFINITY ? 0.0f : expf(ms - M);   // an empty split (and an empty sequence: M = -inf) weighs nothing
    L = wave_sum(lsum * w);
#pragma unroll
    for (uint32_t u = 0; u < kPre; ++u)
      o = fmaf(ov[u], __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), (int)(g + GROUPS * u))), o);
  } else {
    float m[kPairs], l[kPairs], wm = -INFINITY;
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
      const uint32_t s = tid + 64 * GROUPS * k;
      m[k] = s < nsplit ? base[(size_t)s * rec] : -INFINITY;
      l[k] = s < nsplit ? base[(size_t)s * rec + 1] : 0.0f;
      wm = fmaxf(wm, m[k]);
    }
    wm = wave_max(wm);
    if (lane == 0) red[g] = wm;
    __syncthreads();
    const float M = wave_max(lane < GROUPS ? red[lane] : -INFINITY);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kPairs; ++k) {
      const float w = m[k] == -INFINITY ? 0.0f : expf(m[k] - M);
      Ws[tid + 64 * GROUPS * k] = w;
      sum = fmaf(l[k], w, sum);
    }
    sum = wave_sum(sum);
    if (lane == 0) reds[g] = sum;
    __syncthreads();
    L = wave_sum(lane < GROUPS ? reds[lane] : 0.0f);
#pragma unroll
    for (uint32_t u = 0; u < kPre; ++u) {
      const uint32_t s = g + GROUPS * u;   // < 64 < nsplit
      o = fmaf(ov[u], Ws[s], o);
    }
    if (d < headDim) {
#pragma unroll 8
      for (uint32_t s = g + GROUPS * kPre; s < nsplit; s += GROUPS) o = fmaf(base[(size_t)s * rec + 2 + d], Ws[s], o);
    }
  }
  os[g][lane] = o;
  __syncthreads();
  if (g > 0) return;
#pragma unroll
  for (int k = 1; k < GROUPS; ++k) o += os[k][lane];
  if (d < headDim) st_act(out, out_f16, (size_t)h * headDim + d, L > 0.0f ? o / L : 0.0f);
}

static int launch_attn_merge(const void *records, uint32_t nsplit, uint32_t n_heads, uint32_t head_dim, void *out, int out_f16,
                             hipStream_t s) {
  const dim3 grid(n_heads, (head_dim + 63) / 64);
  if (nsplit <= 32)
    hipLaunchKernelGGL(attn_merge_kernel<4>, grid, dim3(256), 0, s, (const float *)records, out, out_f16, head_dim, nsplit);
  else
    hipLaunchKernelGGL(attn_merge_kernel<8>, grid, dim3(512), 0, s, (const float *)records, out, out_f16, head_dim, nsplit);
  return check_hip(hipGetLastError(), "attention merge launch");
}

// ---- SiLU(gate) * up on the output of a fused gate+up matmul: in = [gate(n) | up(n)] ----
__device__ __forceinline__ float silu_times(float g, float u) { return g / (1.0f + __expf(-g)) * u; }

__global__ void __launch_bounds__(256) silu_mul_kernel(const void *in, int in_f16, void *out, int out_f16, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  st_act(out, out_f16, i, silu_times(ld_act(in, in_f16, i), ld_act(in, in_f16, (size_t)n + i)));
}
// Eight elements per thread, where both halves and the output allow 16-byte accesses (n a multiple of 8).  Bound: HBM.
// 2048 rows of 14336 in fp16: 28 us (6.2 TB/s), with one element per thread 89 us.
template <bool IN16, bool OUT16>
__global__ void __launch_bounds__(256) silu_mul8_kernel(const void *in, void *out, uint32_t n) {
  const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= n) return;
  float g[8], u[8];
  ld8<IN16>(in, i, 8, true, g);
  ld8<IN16>(in, (size_t)n + i, 8, true, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = silu_times(g[e], u[e]);
  if (OUT16) {
    half8_t h;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = (half_t)g[e];
    *reinterpret_cast<half8_t *>(reinterpret_cast<half_t *>(out) + i) = h;
  } else {
    float *o = reinterpret_cast<float *>(out) + i;
    *reinterpret_cast<f32x4 *>(o) = f32x4{g[0], g[1], g[2], g[3]};
    *reinterpret_cast<f32x4 *>(o + 4) = f32x4{g[4], g[5], g[6], g[7]};
  }
}

// ---- arg-max (first index of the maximum), one workgroup ----
__global__ void __launch_bounds__(1024) argmax_kernel(const void *x, int x_f16, uint32_t n, uint32_t *out) {
  __shared__ float bv[16];
  __shared__ uint32_t bi[16];
  const uint32_t tid = threadIdx.x;
  float best = -INFINITY;
  uint32_t idx = 0xFFFFFFFFu;
  auto consider = [&](float v, uint32_t i) {
    if (v > best || (v == best && i < idx)) {
      best = v;
      idx = i;
    }
  };
  // 16-byte loads, four per thread in flight: with one scalar load per trip every trip pays a memory latency
  uint32_t done = 0;
  if ((uintptr_t)x % 16 == 0) {
    const uint32_t per = x_f16 ? 8 : 4, nvec = n / per;
    const u32x4 *xv = reinterpret_cast<const u32x4 *>(x);
    for (uint32_t b = tid; b < nvec; b += 4 * 1024) {
      u32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = xv[min(b + u * 1024, nvec - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t vi = b + u * 1024;
        if (vi >= nvec) break;
        if (x_f16) {
          half8_t h = __builtin_bit_cast(half8_t, v[u]);
#pragma unroll
          for (int e = 0; e < 8; ++e) consider((float)h[e], vi * 8 + e);
        } else {
          f32x4 f = __builtin_bit_cast(f32x4, v[u]);
#pragma unroll
          for (int e = 0; e < 4; ++e) consider(f[e], vi * 4 + e);
        }
      }
    }
    done = nvec * per;
  }
  for (uint32_t i = done + tid; i < n; i += 1024) consider(ld_act(x, x_f16, i), i);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float ov = __shfl_xor(best, o);
    uint32_t oi = __shfl_xor(idx, o);
    if (ov > best || (ov == best && oi < idx)) {
      best = ov;
      idx = oi;
    }
  }
  if ((tid & 63) == 0) {
    bv[tid >> 6] = best;
    bi[tid >> 6] = idx;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w)
      if (bv[w] > best || (bv[w] == best && bi[w] < idx)) {
        best = bv[w];
        idx = bi[w];
      }
    out[0] = idx;
  }
}

// ---- greedy sampling after the matmul that produced the logits ----
// One workgroup.  The matmul left, per group of 8 vocabulary rows, the largest logit and its row (ArgmaxPart); this
// kernel applies the repetition penalty to the listed tokens (RepetitionPenalty.cu:19-41: logit > 0 ? logit / f :
// logit * f, written back to the logits), re-derives the groups whose winner was one of them, and reduces.  Without
// parts (parts == nullptr) it scans the logits themselves.  List semantics are those of the dense factor vector the
// runner fills (llama.cpp:2566-2592): a token listed several times is penalised once, with the factor of its last entry.
constexpr uint32_t kMaxPenalized = 1024;

__device__ inline void better(float v, uint32_t i, float &best, uint32_t &idx) {
  if (v > best || (v == best && i < idx)) {
    best = v;
    idx = i;
  }
}

__global__ void __launch_bounds__(1024) argmax_finish_kernel(const ArgmaxPart *parts, void *logits, int x_f16, uint32_t n,
                                                             const int32_t *pen_tokens, const float *pen_factors,
                                                             uint32_t n_pen, uint32_t *out) {
  __shared__ int32_t ptok[kMaxPenalized];
  __shared__ float pval[kMaxPenalized];   // the penalised logit of an effective entry
  __shared__ float bv[16];
  __shared__ uint32_t bi[16];
  const uint32_t tid = threadIdx.x;
  float best = -INFINITY;
  uint32_t idx = 0xFFFFFFFFu;
  if (tid < n_pen) ptok[tid] = pen_tokens[tid];
  __syncthreads();
  // every barrier below is reached by all threads: the per-entry work is predicated, never the barrier
  const bool mine = tid < n_pen;
  const int32_t t = mine ? ptok[tid] : -1;
  bool effective = mine && t >= 0 && (uint32_t)t < n;
  for (uint32_t k = tid + 1; effective && k < n_pen; ++k) effective = ptok[k] != t;   // a later entry of the same token wins
  float v = 0.0f;
  if (effective) {
    const float l = ld_act(logits, x_f16, (size_t)t), f = pen_factors[tid];
    v = l > 0.0f ? l / f : l * f;
    st_act(logits, x_f16, (size_t)t, v);
    if (x_f16) v = (float)(half_t)v;   // as stored
  }
  __syncthreads();            // every entry has read its token before any is marked
  if (mine) {
    if (!effective) ptok[tid] = -1;
    pval[tid] = v;
  }
  __syncthreads();
  // value of row r as the penalised logits hold it: listed rows from the table above (their stores may not be
  // visible to the other waves yet), all others from memory
  auto row_value = [&](uint32_t r) {
    for (uint32_t k = 0; k < n_pen; ++k)
      if (ptok[k] == (int32_t)r) return pval[k];
    return ld_act(logits, x_f16, (size_t)r);
  };
  if (parts) {
    const uint32_t ngroups = (n + 7) / 8;
    constexpr int kInFlight = 8;   // pairs requested together: one memory round trip per 8192 groups instead of one per 1024
    for (uint32_t g0 = tid; g0 < ngroups; g0 += 1024 * kInFlight) {
      ArgmaxPart p[kInFlight];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) p[u] = parts[min(g0 + u * 1024, ngroups - 1)];
#pragma unroll
      for (int u = 0; u < kInFlight; ++u) {
        const uint32_t g = g0 + u * 1024;
        if (g >= ngroups) break;
        bool listed = false;
        for (uint32_t k = 0; k < n_pen; ++k) listed |= ptok[k] >= 0 && ((uint32_t)ptok[k] >> 3) == g;
        if (!listed) {
          better(p[u].value, p[u].index, best, idx);
        } else {
          for (uint32_t r = g * 8; r < min(n, g * 8 + 8); ++r) better(row_value(r), r, best, idx);
        }
      }
    }
  } else {
    for (uint32_t r = tid; r < n; r += 1024) better(n_pen ? row_value(r) : ld_act(logits, x_f16, (size_t)r), r, best, idx);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float ov = __shfl_xor(best, o);
    uint32_t oi = __shfl_xor(idx, o);
    better(ov, oi, best, idx);
  }
  if ((tid & 63) == 0) {
    bv[tid >> 6] = best;
    bi[tid >> 6] = idx;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w) better(bv[w], bi[w], best, idx);
    out[0] = idx;
  }
}

// ---- RepetitionPenaltyOpNode on a dense factor vector (RepetitionPenalty.cu:19-41) ----
__global__ void __launch_bounds__(256) repetition_penalty_kernel(const float *logits, const float *factors, float *out, uint32_t n) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float l = logits[i], f = factors[i];
  out[i] = l > 0.0f ? l / f : l * f;
}

// ---- EmbeddingCol (operators/impl/memory/EmbeddingCol.cu:16-44): gather from a table kept column-wise ----
// format 0: fp16 table; 1: int8 table with fp16 scales per 32 dims (the loader's separated Q8_0 tensors)
__global__ void __launch_bounds__(256) embedding_col_kernel(const uint32_t *indices, const void *matrix, const uint16_t *scales,
                                                            float *out, uint32_t numIndices, uint32_t embDim,
                                                            uint32_t vocabStride, uint32_t scaleStride, uint32_t outStride,
                                                            uint32_t vocab, int format) {
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  if (gid >= numIndices * embDim) return;
  const uint32_t i = gid / embDim, d = gid % embDim, t = indices[i];
  float v = 0.0f;
  if (t < vocab) {   // an index past the table reads nothing and yields zero
    const size_t idx = (size_t)d * vocabStride + t;
    if (format == 0) {
      v = f16bits_to_f32(reinterpret_cast<const uint16_t *>(matrix)[idx]);
    } else {
      const int b = reinterpret_cast<const int8_t *>(matrix)[idx];
      v = (float)b * f16bits_to_f32(scales[(size_t)(d >> 5) * scaleStride + t]);
    }
  }
  out[(size_t)i * outStride + d] = v;
}

static bool bad_dtype(int d) { return d != CUTHIP_F32 && d != CUTHIP_F16; }

}  // namespace cuthip

using namespace cuthip;

extern "C" {

int cuthip_rmsnorm(const void *x, int x_dtype, const float *weight, void *out, int out_dtype, uint32_t rows, uint32_t dim,
                   uint32_t stride, float eps, void *stream) {
  if (!x || !weight || !out || rows == 0 || dim == 0 || stride < dim || bad_dtype(x_dtype) || bad_dtype(out_dtype)) {
    set_error("cuthip_rmsnorm: bad argument (rows %u, dim %u, stride %u)", rows, dim, stride);
    return CUTHIP_ERR_INVALID;
  }
  const bool xf = x_dtype == CUTHIP_F16, of = out_dtype == CUTHIP_F16;
  // 16-byte loads need rows that start on a 16-byte boundary
  const int aligned = (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (stride % 8 == 0);
  const bool wide = aligned && dim % 8 == 0 && dim <= kNormGroups * 2048 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(weight) % 16 == 0;
  if (wide) {
    auto pick = [&](auto ng) {
      constexpr int NG = decltype(ng)::value;
      return xf ? (of ? rmsnorm8_kernel<true, true, NG> : rmsnorm8_kernel<true, false, NG>)
                : (of ? rmsnorm8_kernel<false, true, NG> : rmsnorm8_kernel<false, false, NG>);
    };
    auto kern = dim <= 2048   ? pick(std::integral_constant<int, 1>{})
                : dim <= 4096 ? pick(std::integral_constant<int, 2>{})
                              : pick(std::integral_constant<int, kNormGroups>{});
    hipLaunchKernelGGL(kern, dim3(rows), dim3(256), 0, (hipStream_t)stream, x, weight, out, dim, stride, eps);
    return check_hip(hipGetLastError(), "rmsnorm launch");
  }
  auto kern = xf ? (of ? rmsnorm_kernel<true, true> : rmsnorm_kernel<true, false>)
                 : (of ? rmsnorm_kernel<false, true> : rmsnorm_kernel<false, false>);
  hipLaunchKernelGGL(kern, dim3(rows), dim3(256), 0, (hipStream_t)stream, x, weight, out, dim, stride, eps, aligned);
  return check_hip(hipGetLastError(), "rmsnorm launch");
}

int cuthip_rope_kv_write(const void *q, const void *k, const void *v, int in_dtype, const uint32_t *runtime_params,
                         const float *cos_table, const float *sin_table, void *k_cache, void *v_cache, void *q_out,
                         int q_out_dtype, uint32_t q_dim, uint32_t kv_dim, uint32_t head_dim, uint32_t aligned_kv_dim,
                         uint32_t max_positions, void *stream) {
  if (!q || !k || !v || !runtime_params || !cos_table || !sin_table || !k_cache || !v_cache || !q_out || head_dim == 0 ||
      head_dim % 2 || q_dim % head_dim || kv_dim % head_dim || aligned_kv_dim < kv_dim || bad_dtype(in_dtype) ||
      bad_dtype(q_out_dtype)) {
    set_error("cuthip_rope_kv_write: bad argument (q_dim %u, kv_dim %u, head_dim %u)", q_dim, kv_dim, head_dim);
    return CUTHIP_ERR_INVALID;
  }
  uint32_t total = q_dim + 2 * kv_dim;
  hipLaunchKernelGGL(rope_kv_kernel, dim3((total + 255) / 256), dim3(256), 0, (hipStream_t)stream, q, k, v,
                     in_dtype == CUTHIP_F16, runtime_params, cos_table, sin_table, (half_t *)k_cache, (half_t *)v_cache, q_out,
                     q_out_dtype == CUTHIP_F16, q_dim, kv_dim, head_dim, aligned_kv_dim, max_positions);
  return check_hip(hipGetLastError(), "rope launch");
}

size_t cuthip_attn_decode_workspace_bytes(uint32_t n_heads, uint32_t head_dim, uint32_t max_seq_len) {
  size_t nsplit = (max_seq_len + kAttnChunk - 1) / kAttnChunk;
  return (size_t)n_heads * nsplit * (2 + head_dim) * sizeof(float);
}

// Argument checks shared by the two attention entry points (the workspace is checked by each).
static int attn_check_args(const char *who, const void *q, int q_dtype, const void *k_cache, const void *v_cache,
                           const uint32_t *runtime_params, const void *out, int out_dtype, uint32_t n_heads,
                           uint32_t n_kv_heads, uint32_t head_dim, uint32_t aligned_kv_dim, uint32_t max_seq_len) {
  if (!q || !k_cache || !v_cache || !runtime_params || !out || n_heads == 0 || n_kv_heads == 0 || n_heads % n_kv_heads ||
      head_dim == 0 || head_dim > kAttnMaxHd || head_dim % 8 || max_seq_len == 0 || aligned_kv_dim < n_kv_heads * head_dim ||
      aligned_kv_dim % 8 || bad_dtype(q_dtype) || bad_dtype(out_dtype)) {
    set_error("%s: bad argument (heads %u/%u, head_dim %u (<= %d, multiple of 8), aligned_kv_dim %u)", who, n_heads, n_kv_heads,
              head_dim, kAttnMaxHd, aligned_kv_dim);
    return CUTHIP_ERR_INVALID;
  }
  if ((max_seq_len + kAttnChunk - 1) / kAttnChunk > (uint32_t)kAttnMaxSplit) {
    set_error("%s: max_seq_len %u exceeds %d", who, max_seq_len, kAttnMaxSplit * kAttnChunk);
    return CUTHIP_ERR_INVALID;
  }
  return CUTHIP_OK;
}

}  // extern "C"

namespace cuthip {
// Splits of the context (records per head): one chunk of 64 positions each while that gives at most kAttnWgs workgroups
// (two per CU; twice as many where a workgroup serves more than four heads; more than eight heads multiply them, not
// counted), several beyond, so that every workgroup is resident and streams.  attn_partial_kernel, when it served these shapes: eight layers of an
// 8B model in all, us, with 8 KV heads of 128 and a context of 16,384 / 8,192 /
// 4,096: one chunk per workgroup 420 / 344 / 300, at most 1024 workgroups 401 / 344 / 298, 512 384 / 332 / 300, 256
// 411 / 340 / 305; 32 KV heads at 8,192: 560 / 512 / 496 / 573; 4 KV heads (eight query heads each) at 16,384: 363 / 363 /
// 372 / 400.  (One chunk each, one group of threads per merge and no prefetch: 464 / 363 / 318; 534; 446.)
constexpr uint32_t kAttnWgs = 512;
static uint32_t attn_splits(uint32_t max_seq_len, uint32_t n_heads, uint32_t n_kv_heads) {
  const uint32_t chunks = (max_seq_len + kAttnChunk - 1) / kAttnChunk, wgs = n_heads / n_kv_heads > 4 ? 2 * kAttnWgs : kAttnWgs;
  const uint32_t per = (uint32_t)(((uint64_t)chunks * n_kv_heads + wgs - 1) / wgs);
  return (chunks + per - 1) / per;
}

// Which kernel: attn_rows_kernel with `heads` query heads of a KV head per workgroup, or (0) attn_partial_kernel.  A group of more than two is
// served in pairs, a chunk each, while these are few: each reads K and V again, from the L2.  Then four heads at a time over several chunks.  (In a
// decode step of twelve layers with 32 / 8 heads, all routes in one library, us a layer, pairs / attn_partial_kernel / four: 1024 positions 43.6 /
// 44.8 / 44.3, 2048 44.6 / 44.9 / 44.7, 3000 45.8 / 46.2 / 46.2, 3500 46.6 / 46.4 / 46.2.)  us by themselves, in
// pairs / four / attn_partial_kernel (query / KV heads, dimension 128; workgroups in pairs): 32 / 8 1500 positions (384) 6.5 / 7.2 / 6.8, 2048 (512) 7.1 /
// 7.4 / 7.4, 3000 (752) 8.4 / 8.4 / 8.7, 4096 (1024) 9.8 / 9.2 / 9.4, 16,384 25.7 / 17.7 / 21.2; 32 / 4 2500 (640) 7.5 / 8.0 / 8.5, 3500 (880) 8.9 /
// 8.2 / 9.1; 64 / 8 1500 (768) 7.3 / 8.1 / 8.4, 2500 (1280) 10.1 / 9.3 / 10.6; more than 32 heads, 71 / 1 30,000: 63 / 60 / 40.
// Dimension 64: four heads 32 / 8 3000 (quads 376) 6.8 against 6.6, 6000 (752) 7.7 / 8.4; 64 / 8 4096 (1024) 7.8 / 8.6; pairs 32 / 4 1500 (384) 5.9 / 6.4,
// 3000 (752) 7.2 / 7.0; 32 / 8 64 (16) 4.8 / 4.9, 1024 (256) 5.4 / 5.5, 1500 (384) 5.9 / 5.6.
// Three, five, six and seven groups of four leave CUs of an XCD idle, which very many heads feel (us, four / attn_partial_kernel): dimension 64,
// 12,000 positions 96 / 8 heads 19.8 / 22.0, 144 / 12 26.3 / 24.1, 288 / 24 45.5 / 40.0; dimension 128 192 / 16 at 20,000 73 / 80, 384 / 32 at 12,000 103 / 91.
struct AttnRoute { uint32_t heads, nsplit; };
AttnRoute attn_route(uint32_t head_dim, uint32_t n_heads, uint32_t n_kv_heads, uint32_t max_seq_len) {
  const uint32_t chunks = (max_seq_len + kAttnChunk - 1) / kAttnChunk, n_rep = n_heads / n_kv_heads;
  const uint64_t work = (uint64_t)chunks * n_kv_heads;
  // as many chunks a workgroup as leave at most one workgroup per CU: its waves stream by themselves, and there is half as much to merge
  // (the kernel with a barrier per chunk wants two).  Counted XCD by XCD: the `groups` workgroups of a (KV head, split) share one, and a CU with
  // two of them ends last.  Counted over the whole chip, three and seven groups put 33 and 35 on the 32 CUs of some XCDs; us, attn_partial_kernel / so
  // (and with the split padded to a multiple of eight workgroups, see the launch) / now, dimension 128: 48 / 4 heads at 32,000 positions 39.0 / 43.0 /
  // 32.2, 56 / 2 at 20,000 28.9 / 33.0 / 25.7, 84 / 7 at 20,000 40.8 / 49.2 / 36.7, 144 / 9 60.7 / 75.2 / 52.0, 40 / 5 27.9 / 27.5 / 20.8.
  auto splits = [&](uint64_t groups) {
    const uint32_t most = (uint32_t)std::max<uint64_t>(1, 8 * (32 / groups) / n_kv_heads), per = (chunks + most - 1) / most;
    return (chunks + per - 1) / per;
  };
  if ((head_dim == 128 || head_dim == 64) && n_kv_heads <= 1u << 16) {   // (65,535 eighths of the pairs)
    if (n_rep <= 2) return {n_rep, work <= 512 ? chunks : splits(1)};
    const uint64_t pairs = work * ((n_rep + 1) / 2), quads = work * ((n_rep + 3) / 4);
    if (pairs <= (head_dim == 128 ? 768u : n_rep <= 4 ? 0u : 512u)) return {2, chunks};
    const uint32_t groups = (n_rep + 3) / 4;
    const bool fills = 32 % groups == 0 || n_heads <= (head_dim == 128 ? 192u : 96u);
    if (n_rep <= 32 && fills && (head_dim == 128 || quads > 512)) return {4, splits(groups)};
  }
  return {0, attn_splits(max_seq_len, n_heads, n_kv_heads)};
}
}  // namespace cuthip

extern "C" {

// The two launches of the split-context attention; `partial` holds cuthip_attn_decode_workspace_bytes() bytes.
static int attn_launch(const void *q, int q_dtype, const void *k_cache, const void *v_cache, const uint32_t *runtime_params,
                       void *out, int out_dtype, uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                       uint32_t aligned_kv_dim, float scale, uint32_t max_seq_len, void *partial, hipStream_t s) {
  const AttnRoute route = attn_route(head_dim, n_heads, n_kv_heads, max_seq_len);
  const uint32_t nsplit = route.nsplit, n_rep = n_heads / n_kv_heads;
  if (route.heads) {
    const bool one = nsplit * (uint64_t)kAttnChunk >= max_seq_len;   // a chunk per workgroup (four heads: only past 1,500 query heads)
    auto of = [&](auto hd, auto o) {
      constexpr int HD = decltype(hd)::value;
      constexpr bool ONE = decltype(o)::value;
      return route.heads == 1 ? attn_rows_kernel<HD, 1, ONE> : route.heads == 2 ? attn_rows_kernel<HD, 2, ONE> : attn_rows_kernel<HD, 4, false>;
    };
    auto kernel = head_dim == 128 ? (one ? of(std::integral_constant<int, 128>{}, std::true_type{}) : of(std::integral_constant<int, 128>{}, std::false_type{}))
                                  : (one ? of(std::integral_constant<int, 64>{}, std::true_type{}) : of(std::integral_constant<int, 64>{}, std::false_type{}));
    // the groups of a (KV head, split) follow each other on one XCD, whose L2 has the chunk by then; only the last eight pairs are padded (empty
    // workgroups between the others, group by group, left CUs with two of them: 84 / 3 heads at 20,000 positions 53.6 us, so 39.2)
    const uint32_t groups = (n_rep - 1) / route.heads + 1, pairs = n_kv_heads * nsplit;
    hipLaunchKernelGGL(kernel, dim3(8, groups, (pairs + 7) / 8), dim3(256), 0, s, q, (const half_t *)k_cache, (const half_t *)v_cache, runtime_params,
                       aligned_kv_dim, max_seq_len, n_rep, n_kv_heads, (int)(q_dtype == CUTHIP_F16), nsplit, (float *)partial, scale);
    if (int rc = check_hip(hipGetLastError(), "attention launch")) return rc;
    return launch_attn_merge(partial, nsplit, n_heads, head_dim, out, out_dtype == CUTHIP_F16, s);
  }
  const bool two = n_rep > 4;
  auto kernel = head_dim == 128  ? attn_partial_kernel<128, 2>   // (more than 32 query heads per KV head, or very many in all)
                : head_dim == 64 ? (two ? attn_partial_kernel<64, 2> : attn_partial_kernel<64, 1>)
                                 : (two ? attn_partial_kernel<0, 2> : attn_partial_kernel<0, 1>);
  hipLaunchKernelGGL(kernel, dim3(n_kv_heads, nsplit, (n_rep + 7) / 8), dim3(256), 0, s, q, (const half_t *)k_cache,
                     (const half_t *)v_cache, runtime_params, aligned_kv_dim, max_seq_len, n_heads, n_kv_heads,
                     (int)(q_dtype == CUTHIP_F16), head_dim, (float *)partial, scale, nsplit);
  if (int rc = check_hip(hipGetLastError(), "attention launch")) return rc;
  return launch_attn_merge(partial, nsplit, n_heads, head_dim, out, out_dtype == CUTHIP_F16, s);
}

int cuthip_attn_decode(const void *q, int q_dtype, const void *k_cache, const void *v_cache, const uint32_t *runtime_params,
                       void *out, int out_dtype, uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                       uint32_t aligned_kv_dim, float scale, uint32_t max_seq_len, void *workspace, size_t workspace_bytes,
                       void *stream) {
  if (int rc = attn_check_args("cuthip_attn_decode", q, q_dtype, k_cache, v_cache, runtime_params, out, out_dtype, n_heads,
                               n_kv_heads, head_dim, aligned_kv_dim, max_seq_len))
    return rc;
  if (!workspace || (uintptr_t)workspace % 4 != 0 ||
      workspace_bytes < cuthip_attn_decode_workspace_bytes(n_heads, head_dim, max_seq_len)) {
    set_error("cuthip_attn_decode: workspace of %zu bytes, need %zu", workspace ? workspace_bytes : (size_t)0,
              cuthip_attn_decode_workspace_bytes(n_heads, head_dim, max_seq_len));
    return CUTHIP_ERR_INVALID;
  }
  return attn_launch(q, q_dtype, k_cache, v_cache, runtime_params, out, out_dtype, n_heads, n_kv_heads, head_dim,
                     aligned_kv_dim, scale, max_seq_len, workspace, (hipStream_t)stream);
}

uint32_t cuthip_attn_partial_splits(uint32_t max_seq_len) {
  const uint32_t chunks = (max_seq_len + kAttnChunk - 1) / kAttnChunk;
  return chunks < (uint32_t)kAttnWideSplits ? chunks : (uint32_t)kAttnWideSplits;
}

size_t cuthip_attn_partial_bytes(uint32_t n_heads, uint32_t head_dim, uint32_t max_seq_len) {
  return (size_t)n_heads * cuthip_attn_partial_splits(max_seq_len) * (2 + head_dim) * sizeof(float);
}

int cuthip_attn_decode_partial(const void *q, int q_dtype, const void *k_cache, const void *v_cache,
                               const uint32_t *runtime_params, uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                               uint32_t aligned_kv_dim, float scale, uint32_t max_seq_len, void *records, size_t records_bytes,
                               void *stream) {
  // (the records stand in for the output in the shared checks)
  if (int rc = attn_check_args("cuthip_attn_decode_partial", q, q_dtype, k_cache, v_cache, runtime_params, records, CUTHIP_F32,
                               n_heads, n_kv_heads, head_dim, aligned_kv_dim, max_seq_len))
    return rc;
  if (head_dim != 128) {
    set_error("cuthip_attn_decode_partial: head_dim %u (the wide-split kernel is built for 128; use cuthip_attn_decode)", head_dim);
    return CUTHIP_ERR_INVALID;
  }
  if ((uintptr_t)records % 8 != 0 || records_bytes < cuthip_attn_partial_bytes(n_heads, head_dim, max_seq_len)) {
    set_error("cuthip_attn_decode_partial: records of %zu bytes, need %zu, 8-byte aligned", records_bytes,
              cuthip_attn_partial_bytes(n_heads, head_dim, max_seq_len));
    return CUTHIP_ERR_INVALID;
  }
  const uint32_t nsplit = cuthip_attn_partial_splits(max_seq_len);
  static std::once_flag lds_once;
  static int lds_rc = CUTHIP_OK;
  std::call_once(lds_once, [] {
    lds_rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(attn_partial_wide_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kAttnWideLds),
                       "hipFuncSetAttribute(attention LDS)");
  });
  if (lds_rc) return lds_rc;
  hipLaunchKernelGGL(attn_partial_wide_kernel, dim3(n_heads * nsplit), dim3(256), kAttnWideLds, (hipStream_t)stream, q,
                     (const half_t *)k_cache, (const half_t *)v_cache, runtime_params, aligned_kv_dim, max_seq_len, n_heads,
                     n_kv_heads, (int)(q_dtype == CUTHIP_F16), nsplit, (float *)records, scale);
  return check_hip(hipGetLastError(), "attention launch");
}

int cuthip_attn_merge(const void *records, uint32_t nsplit, uint32_t n_heads, uint32_t head_dim, void *out, int out_dtype,
                      void *stream) {
  if (!records || !out || nsplit == 0 || nsplit > (uint32_t)kAttnMaxSplit || n_heads == 0 || head_dim == 0 ||
      head_dim > (uint32_t)kAttnMaxHd || (uintptr_t)records % 4 != 0 || bad_dtype(out_dtype)) {
    set_error("cuthip_attn_merge: bad argument (splits %u (<= %d), heads %u, head_dim %u (<= %d))", nsplit, kAttnMaxSplit,
              n_heads, head_dim, kAttnMaxHd);
    return CUTHIP_ERR_INVALID;
  }
  return launch_attn_merge(records, nsplit, n_heads, head_dim, out, out_dtype == CUTHIP_F16, (hipStream_t)stream);
}

}  // extern "C"

// ---- the attention without a caller workspace: partial results in a device array of this library ----
// One copy of the array exists on every GPU the library runs on, at its own address, until the process ends.  The
// array's name is a host-side stand-in; the device address is taken once per device with hipGetSymbolAddress.
namespace cuthip {
constexpr size_t kAttnStaticBytes = 4u << 20;   // 4 MiB: 32 heads of dimension 128 up to a cache capacity of 16,128
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kAttnStaticBytes];
static void *g_scratch_ptr[kMaxDevices];   // per device; written under g_scratch_mu
static std::mutex g_scratch_mu;

// Device address of `scratch` on the device that owns `stream` (the current device for the null stream), looked up
// on first use there with that device current; nullptr after set_error.
static void *attn_static_ptr(hipStream_t stream) {
  int cur = -1, dev = -1;
  if (check_hip(hipGetDevice(&cur), "hipGetDevice")) return nullptr;
  dev = cur;
  if (stream) {
    hipDevice_t sd = 0;
    if (check_hip(hipStreamGetDevice(stream, &sd), "hipStreamGetDevice")) return nullptr;
    dev = (int)sd;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("attention scratch: device index %d beyond %d", dev, kMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    if (dev != cur && check_hip(hipSetDevice(dev), "hipSetDevice")) return nullptr;
    const int rc = check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    if (dev != cur) (void)hipSetDevice(cur);
    if (rc) return nullptr;
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

// called by cuthip_init with the chosen device current
int attn_static_setup() { return attn_static_ptr(nullptr) ? CUTHIP_OK : CUTHIP_ERR_HIP; }
}  // namespace cuthip

extern "C" {

size_t cuthip_attn_decode_static_max_bytes(void) { return kAttnStaticBytes; }


int cuthip_attn_decode_static(const void *q, int q_dtype, const void *k_cache, const void *v_cache,
                              const uint32_t *runtime_params, void *out, int out_dtype, uint32_t n_heads, uint32_t n_kv_heads,
                              uint32_t head_dim, uint32_t aligned_kv_dim, float scale, uint32_t max_seq_len, void *stream) {
  if (int rc = attn_check_args("cuthip_attn_decode_static", q, q_dtype, k_cache, v_cache, runtime_params, out, out_dtype,
                               n_heads, n_kv_heads, head_dim, aligned_kv_dim, max_seq_len))
    return rc;
  const size_t need = cuthip_attn_decode_workspace_bytes(n_heads, head_dim, max_seq_len);
  if (need > kAttnStaticBytes) {
    set_error("cuthip_attn_decode_static: %u heads of dimension %u over a cache of %u positions need %zu bytes of partial "
              "results, the built-in scratch holds %zu; use cuthip_attn_decode with a workspace", n_heads, head_dim,
              max_seq_len, need, kAttnStaticBytes);
    return CUTHIP_ERR_INVALID;
  }
  void *ptr = attn_static_ptr((hipStream_t)stream);
  if (!ptr) return CUTHIP_ERR_HIP;
  // every split record of this call's launch shape is written before the merge reads it, so nothing of an earlier
  // call's contents is read and nothing needs clearing
  return attn_launch(q, q_dtype, k_cache, v_cache, runtime_params, out, out_dtype, n_heads, n_kv_heads, head_dim,
                     aligned_kv_dim, scale, max_seq_len, ptr, (hipStream_t)stream);
}

int cuthip_silu_mul(const void *gate_up, int in_dtype, void *out, int out_dtype, uint32_t n, void *stream) {
  if (!gate_up || !out || n == 0 || bad_dtype(in_dtype) || bad_dtype(out_dtype)) {
    set_error("cuthip_silu_mul: bad argument");
    return CUTHIP_ERR_INVALID;
  }
  const bool in16 = in_dtype == CUTHIP_F16, out16 = out_dtype == CUTHIP_F16;
  if (n % 8 == 0 && n <= 0xFFFFF800u && (uintptr_t)gate_up % 16 == 0 && (uintptr_t)out % 16 == 0) {
    auto kern = in16 ? (out16 ? silu_mul8_kernel<true, true> : silu_mul8_kernel<true, false>)
                     : (out16 ? silu_mul8_kernel<false, true> : silu_mul8_kernel<false, false>);
    hipLaunchKernelGGL(kern, dim3((n / 8 - 1) / 256 + 1), dim3(256), 0, (hipStream_t)stream, gate_up, out, n);
  } else {
    hipLaunchKernelGGL(silu_mul_kernel, dim3((n - 1) / 256 + 1), dim3(256), 0, (hipStream_t)stream, gate_up, in16, out, out16, n);
  }
  return check_hip(hipGetLastError(), "silu_mul launch");
}

int cuthip_argmax(const void *x, int x_dtype, uint32_t n, uint32_t *out_index, void *stream) {
  if (!x || !out_index || n == 0 || bad_dtype(x_dtype)) {
    set_error("cuthip_argmax: bad argument");
    return CUTHIP_ERR_INVALID;
  }
  hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, x, x_dtype == CUTHIP_F16, n, out_index);
  return check_hip(hipGetLastError(), "argmax launch");
}

}  // extern "C"

extern "C" {

int cuthip_argmax_penalized(void *logits, int x_dtype, uint32_t n, const int32_t *pen_tokens, const float *pen_factors,
                            uint32_t n_pen, uint32_t *out_index, void *stream) {
  if (!logits || !out_index || n == 0 || bad_dtype(x_dtype) || n_pen > kMaxPenalized || (n_pen && (!pen_tokens || !pen_factors))) {
    set_error("cuthip_argmax_penalized: bad argument (n %u, %u penalised tokens, at most %u)", n, n_pen, kMaxPenalized);
    return CUTHIP_ERR_INVALID;
  }
  hipLaunchKernelGGL(argmax_finish_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const ArgmaxPart *)nullptr, logits,
                     x_dtype == CUTHIP_F16, n, pen_tokens, pen_factors, n_pen, out_index);
  return check_hip(hipGetLastError(), "argmax launch");
}

int cuthip_repetition_penalty(const float *logits, const float *factors, float *out, uint32_t n, void *stream) {
  if (!logits || !factors || !out) {
    set_error("cuthip_repetition_penalty: null argument");
    return CUTHIP_ERR_INVALID;
  }
  if (n == 0) return CUTHIP_OK;
  hipLaunchKernelGGL(repetition_penalty_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, logits, factors, out, n);
  return check_hip(hipGetLastError(), "repetition penalty launch");
}

int cuthip_embedding_col(const uint32_t *indices, const void *matrix, const uint16_t *scales, float *out, uint32_t num_indices,
                         uint32_t emb_dim, uint32_t vocab_stride, uint32_t scale_stride, uint32_t out_stride, uint32_t vocab,
                         int format, void *stream) {
  if (!indices || !matrix || !out || (format != 0 && format != 1) || (format == 1 && !scales) || out_stride < emb_dim ||
      vocab > vocab_stride || (format == 1 && vocab > scale_stride) || (uint64_t)num_indices * emb_dim > 0xFFFFFFFFull) {
    set_error("cuthip_embedding_col: bad argument (format %d, emb_dim %u, vocab %u, strides %u %u %u)", format, emb_dim, vocab,
              vocab_stride, scale_stride, out_stride);
    return CUTHIP_ERR_INVALID;
  }
  const uint32_t total = num_indices * emb_dim;
  if (total == 0) return CUTHIP_OK;
  hipLaunchKernelGGL(embedding_col_kernel, dim3((total + 255) / 256), dim3(256), 0, (hipStream_t)stream, indices, matrix, scales,
                     out, num_indices, emb_dim, vocab_stride, scale_stride, out_stride, vocab, format);
  return check_hip(hipGetLastError(), "embedding launch");
}

}  // extern "C"

namespace cuthip {
// second launch of cuthip_matmul_gguf_argmax (gemv.hip): arguments validated there
int launch_argmax_finish(const ArgmaxPart *parts, void *logits, int x_f16, uint32_t n, const int32_t *pen_tokens,
                         const float *pen_factors, uint32_t n_pen, uint32_t *out_index, hipStream_t stream) {
  hipLaunchKernelGGL(argmax_finish_kernel, dim3(1), dim3(1024), 0, stream, parts, logits, x_f16, n, pen_tokens, pen_factors,
                     n_pen, out_index);
  return check_hip(hipGetLastError(), "argmax launch");
}
uint32_t max_penalized() { return kMaxPenalized; }
}  // namespace cuthip
