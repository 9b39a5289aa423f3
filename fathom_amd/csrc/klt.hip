// Query side of the KLT-rotated bit-plane store (scripts/R_ruler.py:63-64,
// 82-84, the "planesK" method): the store holds bit planes of (K - mu) @ Vt,
// so each decode step rotates the query the same way, qr = q @ Vt, and plans
// from the gains g_e = sum_g qr_ge^2 * lam_e of the rotated coordinates.
//
// A workgroup owns 16 output coordinates of one (batch, KV head) row, with the
// G query heads staged in LDS: thread (c, p) sums q_g[d] * Vt[d, e0 + c] over
// the p-th of 16 d ranges (fp32 FMAs, ascending d, every load in flight at
// once), and the range sums are added in order; the gain follows in head order.
#include "common.hpp"

namespace fathom {
namespace {

constexpr int kKltThreads = 256;
constexpr int kKltMaxG = 32;                     // query heads per (batch, KV head) row
constexpr int kKltMaxD = 256;
constexpr int kKltCols = 16;                     // output coordinates per workgroup
constexpr int kKltParts = kKltThreads / kKltCols;  // d ranges per coordinate

// MAXG: the heads the workgroup holds (8 for GQA groups of up to 8, else 32).
template <int MAXG>
__global__ __launch_bounds__(kKltThreads) void klt_query_kernel(const float *__restrict__ q,
                                                                 const float *__restrict__ Vt,
                                                                 const float *__restrict__ lam, int G, int D,
                                                                 float *__restrict__ qr, float *__restrict__ gain) {
  __shared__ float qs[MAXG][kKltMaxD];
  __shared__ float part[kKltParts][MAXG][kKltCols];
  const int tid = threadIdx.x;
  const int64_t bh = blockIdx.y;
  const int e0 = blockIdx.x * kKltCols;
  for (int e = tid; e < G * D; e += kKltThreads) qs[e / D][e % D] = q[bh * G * D + e];
  __syncthreads();
  const float *V = Vt + bh * (int64_t)D * D;
  const int c = tid % kKltCols, pt = tid / kKltCols, e = e0 + c;
  const int per = (D + kKltParts - 1) / kKltParts;
  float acc[MAXG];
#pragma unroll
  for (int g = 0; g < MAXG; ++g) acc[g] = 0.0f;
  if (e < D) {
    for (int i = 0; i < per; ++i) {
      const int d = pt * per + i;
      if (d < D) {
        const float v = V[(int64_t)d * D + e];
#pragma unroll
        for (int g = 0; g < MAXG; ++g)
          if (g < G) acc[g] = fmaf(qs[g][d], v, acc[g]);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < MAXG; ++g) part[pt][g][c] = acc[g];
  __syncthreads();
  if (tid < kKltCols && e0 + tid < D) {
    const int eo = e0 + tid;
    const float l = lam[bh * D + eo];
    float s = 0.0f;
    for (int g = 0; g < G; ++g) {
      float r = 0.0f;
      for (int p = 0; p < kKltParts; ++p) r += part[p][g][tid];  // the d ranges in order
      qr[(bh * G + g) * D + eo] = r;
      s += (r * r) * l;  // ((qr ** 2) * lam).sum over heads, in head order
    }
    gain[bh * D + eo] = s;
  }
}

// float(K) - mu of key rows [BH, n, D], the store build's input to the rotation: one
// pass where a conversion and a subtraction took two (a conversion's float32 copy
// written and read again).  V elements per thread and step: 8 16-bit or 4 32-bit keys
// (16-byte loads and stores), 1 where a pointer or D is not aligned to that.  Bound:
// HBM, 6 bytes per 16-bit key, 8 per 32-bit one: 8 x 20011 f16 keys 47 -> 20.4 us; 8 x
// 131072 f32 keys 174 us (329 an element at a time, 177 torch's subtraction).
template <int KDT, int V>
__global__ __launch_bounds__(256) void klt_center_kernel(const void *__restrict__ K, const float *__restrict__ mu, int64_t n,
                                                         int64_t D, float *__restrict__ out) {
  const int64_t bh = blockIdx.y, per = n * D, step = (int64_t)gridDim.x * 256 * V;
  const bool small = per <= 0xFFFFFFFFll;  // uniform: a 32-bit remainder
  const float *m = mu + bh * D;
  float *o = out + bh * per;
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V; i < per; i += step) {
    const int64_t j = small ? (int64_t)((uint32_t)i % (uint32_t)D) : i % D;  // V divides D
    if constexpr (V == 1) {
      o[i] = load_elem<KDT>(K, bh * per + i) - m[j];
    } else {
      float x[V];
      if constexpr (KDT == FATHOM_DT_F32) {
        const float4 r = *reinterpret_cast<const float4 *>(static_cast<const float *>(K) + bh * per + i);
        x[0] = r.x, x[1] = r.y, x[2] = r.z, x[3] = r.w;
      } else {
        const uint4 r = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(K) + bh * per + i);
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const uint16_t h = (uint16_t)(e & 1 ? w[e / 2] >> 16 : w[e / 2]);
          x[e] = KDT == FATHOM_DT_BF16 ? bf16_bits_to_float(h) : f16_bits_to_float(h);
        }
      }
#pragma unroll
      for (int e = 0; e < V; e += 4) {
        const float4 a = *reinterpret_cast<const float4 *>(m + j + e);
        *reinterpret_cast<float4 *>(o + i + e) = make_float4(x[e] - a.x, x[e + 1] - a.y, x[e + 2] - a.z, x[e + 3] - a.w);
      }
    }
  }
}

template <int KDT>
void launch_center(const void *K, const float *mu, int64_t BH, int64_t n, int64_t D, float *out, hipStream_t st) {
  constexpr int V = KDT == FATHOM_DT_F32 ? 4 : 8;
  const bool vec = D % V == 0 &&
                   ((reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(mu) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  const dim3 grid((unsigned)min(cdiv(n * D, vec ? 256 * V : 256), (int64_t)65535), (unsigned)BH);
  if (vec) klt_center_kernel<KDT, V><<<grid, 256, 0, st>>>(K, mu, n, D, out);
  else klt_center_kernel<KDT, 1><<<grid, 256, 0, st>>>(K, mu, n, D, out);
}

}  // namespace
}  // namespace fathom

using namespace fathom;

extern "C" int fathom_klt_center(const void *K, int k_dtype, const float *mu, int64_t BH, int64_t n, int64_t D, float *out,
                                 void *stream) {
  if (!K || !mu || !out) return fail(FATHOM_ERR_INVALID, "klt_center: null pointer");
  if (BH < 1 || BH > 65535 || n < 1 || D < 1)
    return fail(FATHOM_ERR_INVALID, "klt_center: BH=%lld n=%lld D=%lld", (long long)BH, (long long)n, (long long)D);
  hipStream_t st = (hipStream_t)stream;
  switch (k_dtype) {
    case FATHOM_DT_F32: launch_center<FATHOM_DT_F32>(K, mu, BH, n, D, out, st); break;
    case FATHOM_DT_F16: launch_center<FATHOM_DT_F16>(K, mu, BH, n, D, out, st); break;
    case FATHOM_DT_BF16: launch_center<FATHOM_DT_BF16>(K, mu, BH, n, D, out, st); break;
    default: return fail(FATHOM_ERR_INVALID, "klt_center: bad dtype %d", k_dtype);
  }
  return launch_status("klt_center_kernel");
}

extern "C" int fathom_klt_query(const float *q, const float *Vt, const float *lam, int64_t BH, int64_t G, int64_t D,
                                float *qr, float *gain, void *stream) {
  if (!q || !Vt || !lam || !qr || !gain) return fail(FATHOM_ERR_INVALID, "klt_query: null pointer");
  if (BH < 1 || BH > 0x7FFFFFFF) return fail(FATHOM_ERR_INVALID, "klt_query: BH=%lld", (long long)BH);
  if (G < 1 || G > kKltMaxG) return fail(FATHOM_ERR_INVALID, "klt_query: G=%lld outside [1, %d]", (long long)G, kKltMaxG);
  if (D < 1 || D > kKltMaxD) return fail(FATHOM_ERR_INVALID, "klt_query: D=%lld outside [1, %d]", (long long)D, kKltMaxD);
  const dim3 grid((unsigned)cdiv(D, kKltCols), (unsigned)BH);
  if (BH > 65535) return fail(FATHOM_ERR_INVALID, "klt_query: BH=%lld above 65535", (long long)BH);
  if (G <= 8)
    klt_query_kernel<8><<<grid, kKltThreads, 0, (hipStream_t)stream>>>(q, Vt, lam, (int)G, (int)D, qr, gain);
  else
    klt_query_kernel<kKltMaxG><<<grid, kKltThreads, 0, (hipStream_t)stream>>>(q, Vt, lam, (int)G, (int)D, qr, gain);
  return launch_status("klt_query_kernel");
}
