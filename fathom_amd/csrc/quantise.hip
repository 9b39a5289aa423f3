// Store build of D = 128 rows: 4-bit quantiser and bit-plane packer in one pass
// over the keys (kernels/bitplane.py:23-32, 44-50, 60-65).
//
// A wave owns one 64-token block, lane l channels 2l and 2l + 1 (CPL = 2; one
// channel and half a block row with CPL = 1).  Its 64 row loads are all in
// flight at once.
//
// The code floor(x / s), s = amax / 8, without a division per element.  rs is
// the correctly rounded 1 / s, so p = x * rs is within 2^-23 of x / s.
//   16-bit keys: x has at most 11 significant bits and so has s, so a quotient
//     that is no integer is at least 2^-14 (relative) from every nonzero one.
//     Adding 2^-19 |p| -- away from zero above, towards it below -- therefore
//     lifts an exact multiple back over its integer and moves no other quotient
//     across one.
//   32-bit keys: m = rint(p), r = x - m s is exact (fma), and fma(r, rs, m) falls
//     on the same side of m as the correctly rounded quotient: r = -s ulp(m) / 2
//     exactly needs s a power of two (where rs is exact), and any other r is
//     further from it than the error of rs, as s has at most 11 significant bits.
// Both hold for scales between 2^-14 and 65504 and finite keys (32-bit: no
// denormal key); a wave with another channel divides.
//
// Bit packing: v_cvt_pk_u8_f32 drops a code into a byte, two byte words make one
// of eight nibbles, nibble k of word m being token 4k + m of a 32-token half, so
// plane p of the half is the OR over m of (W_m >> (3 - p) & 0x11111111) << m with
// no permutation of bits: 0.9 operations per element instead of 8.
//
// Bound: HBM.  8 x 131072 bf16 keys with codes kept (268 MB in, 207 MB out): 98 us,
// 4.8 TB/s, against 384 us for pack.hip's kernel (a division and about 30
// operations per element, 2-byte loads); 1 x 16384 f32 keys 37 -> 6.8 us.
#include <type_traits>

#include "pack_internal.hpp"

namespace fathom {
namespace pack {
namespace {

constexpr int kD = 128;
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The raw keys of a lane: CPL channels of one token.
template <int KDT, int CPL>
struct RawOf {
  typedef uint32_t type;  // two 16-bit keys
};
template <>
struct RawOf<FATHOM_DT_F32, 2> {
  typedef float2 type;
};
template <>
struct RawOf<FATHOM_DT_F32, 1> {
  typedef float type;
};
template <>
struct RawOf<FATHOM_DT_F16, 1> {
  typedef uint16_t type;
};
template <>
struct RawOf<FATHOM_DT_BF16, 1> {
  typedef uint16_t type;
};

template <int KDT, int CPL>
__device__ __forceinline__ float key_of(const typename RawOf<KDT, CPL>::type &r, int c) {
  if constexpr (KDT == FATHOM_DT_F32) {
    if constexpr (CPL == 2) return c ? r.y : r.x;
    else return r;
  } else if constexpr (KDT == FATHOM_DT_BF16) {
    return __uint_as_float(c ? ((uint32_t)r & 0xFFFF0000u) : ((uint32_t)r << 16));
  } else {
    return f16_bits_to_float((uint16_t)(c ? ((uint32_t)r >> 16) : (uint32_t)r));
  }
}

template <int KDT, int CPL>
__device__ __forceinline__ typename RawOf<KDT, CPL>::type zero_raw() {
  typename RawOf<KDT, CPL>::type z;
  if constexpr (KDT == FATHOM_DT_F32 && CPL == 2) z.x = z.y = 0.0f;
  else z = 0;
  return z;
}

// Plane words of one 32-token half from its byte words B[m][h], byte k of which
// is the code of token 4 (2k + h) + m.
__device__ __forceinline__ void half_planes(const uint32_t (&B)[4][2], uint32_t (&w)[4]) {
  uint32_t W[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) W[m] = B[m][0] | (B[m][1] << 4);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int b = 3 - p;
    uint32_t x = 0u;
#pragma unroll
    for (int m = 0; m < 4; ++m) x |= (m >= b ? W[m] << (m - b) : W[m] >> (b - m)) & (0x11111111u << m);
    w[p] = x;
  }
}

// Codes and plane words of a wave's block.  FAST: the quotient forms above, else
// one IEEE division per element.
template <int KDT, int CPL, bool FAST>
__device__ __forceinline__ void quantise_block(const typename RawOf<KDT, CPL>::type (&raw)[kBlk], const float (&s)[CPL],
                                               int real, uint8_t *code, uint32_t (&w)[CPL][2][4]) {
#pragma clang fp contract(off)
  float rs[CPL], e2[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    rs[c] = FAST ? 1.0f / s[c] : 0.0f;
    e2[c] = rs[c] * 0x1p-19f;
  }
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    uint32_t B[CPL][4][2];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          uint32_t q = 0u;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float x = key_of<KDT, CPL>(raw[32 * half + 4 * (2 * k + h) + m], c);
            float f;
            if constexpr (FAST) {
              const float p = x * rs[c];
              float v;
              if constexpr (KDT == FATHOM_DT_F32) {
                const float mi = rintf(p);
                v = floorf(fmaf(fmaf(-mi, s[c], x), rs[c], mi));
              } else {
                v = floorf(fmaf(fabsf(x), e2[c], p));
              }
              f = __builtin_amdgcn_fmed3f(v, -8.0f, 7.0f) + 8.0f;
            } else {
              // kernels/bitplane.py:31: clamp(floor(x / s), -8, 7) + 8; NaN -> 0.
              const float v = floorf(x / s[c]);
              f = v != v ? 0.0f : fminf(fmaxf(v, -8.0f), 7.0f) + 8.0f;
            }
            q = __builtin_amdgcn_cvt_pk_u8_f32(f, k, q);
          }
          B[c][m][h] = q;
        }
        if (code) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int i = 32 * half + 4 * (2 * k + h) + m;
            if (i < real) {  // uniform
              if constexpr (CPL == 2) {
                const uint32_t two = __builtin_amdgcn_perm(B[1][m][h], B[0][m][h], (uint32_t)k | ((uint32_t)(4 + k) << 8));
                *reinterpret_cast<uint16_t *>(code + i * kD) = (uint16_t)two;
              } else {
                code[i * kD] = (uint8_t)(B[0][m][h] >> (8 * k));
              }
            }
          }
        }
        if (real < kBlk) {  // pack_planes pads the tail of the last block with code 0
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (32 * half + 4 * (2 * k + h) + m >= real) {
#pragma unroll
              for (int c = 0; c < CPL; ++c) B[c][m][h] &= ~(0xFFu << (8 * k));
            }
        }
      }
#pragma unroll
    for (int c = 0; c < CPL; ++c) half_planes(B[c], w[c][half]);
  }
}

// Loads a wave's block, quantises it and writes its logical outputs; the plane
// words (all zero past the row's blocks) and fp16 scale bits come back.
template <int KDT, int CPL>
__device__ __forceinline__ void block_words(const QuantArgs &a, int64_t bh, int64_t b, int j0, uint32_t (&w)[CPL][2][4],
                                            uint16_t (&s16)[CPL]) {
  typedef typename RawOf<KDT, CPL>::type raw_t;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    s16[c] = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 4; ++p) w[c][h][p] = 0u;
  }
  if (b >= a.nblk) return;  // uniform per wave
  const int64_t tok0 = b * kBlk;
  const int real = (int)min((int64_t)kBlk, a.n - tok0);
  const int64_t base = (bh * a.n + tok0) * kD + j0;
  constexpr int kElt = KDT == FATHOM_DT_F32 ? 4 : 2;
  const char *src = static_cast<const char *>(a.K) + base * kElt;
  raw_t raw[kBlk];
  if (real == kBlk) {
#pragma unroll
    for (int i = 0; i < kBlk; ++i) raw[i] = *reinterpret_cast<const raw_t *>(src + (int64_t)i * kD * kElt);
  } else {
#pragma unroll
    for (int i = 0; i < kBlk; ++i) {
      raw[i] = *reinterpret_cast<const raw_t *>(src + (int64_t)min(i, real - 1) * kD * kElt);
      if (i >= real) raw[i] = zero_raw<KDT, CPL>();
    }
  }
  // block absmax, NaN propagating: magnitudes order as their bits
  float af[CPL], s[CPL];
  bool sane = true;
  float amax[CPL];
  bool nan[CPL];
  if constexpr (KDT != FATHOM_DT_F32) {
    constexpr uint32_t kInf = KDT == FATHOM_DT_BF16 ? 0x7F80u : 0x7C00u;
    u16x2 mx = {0, 0};
#pragma unroll
    for (int i = 0; i < kBlk; ++i) {
      const uint32_t m = (uint32_t)raw[i] & 0x7FFF7FFFu;
      u16x2 v;
      __builtin_memcpy(&v, &m, 4);
      mx = __builtin_elementwise_max(mx, v);
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const uint32_t m = c ? mx.y : mx.x;
      amax[c] = KDT == FATHOM_DT_BF16 ? bf16_bits_to_float((uint16_t)m) : f16_bits_to_float((uint16_t)m);
      nan[c] = m > kInf;
    }
  } else {
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      uint32_t mx = 0u, mn = ~0u;
#pragma unroll
      for (int i = 0; i < kBlk; ++i) {
        const uint32_t m = __float_as_uint(key_of<KDT, CPL>(raw[i], c)) & 0x7FFFFFFFu;
        mx = max(mx, m);
        mn = min(mn, m - 1u);  // zero wraps to the top
      }
      amax[c] = __uint_as_float(mx);
      nan[c] = mx > 0x7F800000u;
      sane = sane && mn >= 0x007FFFFFu && a.sdt != FATHOM_DT_F32;
    }
  }
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    // kernels/bitplane.py:29: amax.clamp_min(1e-8).to(scale_dtype).float()
    const float v = nan[c] ? __uint_as_float(0x7FC00000u) : fmaxf(amax[c], 1e-8f);
    uint16_t blk16 = 0;
    if (a.sdt == FATHOM_DT_F16) {
      blk16 = float_to_f16_bits(v);
      af[c] = f16_bits_to_float(blk16);
    } else if (a.sdt == FATHOM_DT_BF16) {
      blk16 = float_to_bf16_bits(v);
      af[c] = bf16_bits_to_float(blk16);
    } else {
      af[c] = v;
    }
    s16[c] = a.sdt == FATHOM_DT_F16 ? blk16 : float_to_f16_bits(af[c]);
    if (a.scales_blk) {
      const int64_t o = (bh * a.nblk + b) * kD + j0 + c;
      if (a.sdt == FATHOM_DT_F32) static_cast<float *>(a.scales_blk)[o] = af[c];
      else static_cast<uint16_t *>(a.scales_blk)[o] = blk16;
    }
    sane = sane && af[c] >= 0x1p-14f && af[c] <= 65504.0f;
    s[c] = af[c] / 8.0f;
  }
  uint8_t *code = a.code ? a.code + base : nullptr;
  if (__all(sane)) quantise_block<KDT, CPL, true>(raw, s, real, code, w);
  else quantise_block<KDT, CPL, false>(raw, s, real, code, w);
  if (a.planes_log) {
    uint4 *P = reinterpret_cast<uint4 *>(a.planes_log + ((bh * a.nblk + b) * kD + j0) * 4);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      P[2 * c] = make_uint4(w[c][0][0], w[c][1][0], w[c][0][1], w[c][1][1]);
      P[2 * c + 1] = make_uint4(w[c][0][2], w[c][1][2], w[c][0][3], w[c][1][3]);
    }
  }
}

// Slot of block bi's word in its unit's run of NB words: the pair of blocks 2i,
// 2i + 1 of channel j sits at pair i ^ (j >> 1 & (NB / 2 - 1)).  A lane's units
// are 32 NB bytes apart and would share banks.
template <int NB>
__device__ __forceinline__ int tile_slot(int j, int bi) {
  return ((bi >> 1) ^ ((j >> 1) & (NB / 2 - 1))) * 2 + (bi & 1);
}

// Writes NB consecutive blocks b0, ... of row bh from LDS (tile [128 * 4][NB] in
// slots, scales stile [128][NB]) to the superblock store, blocks past cover
// dropped.  A (channel, plane) unit leaves in 16-byte pieces where the blocks lie
// in one superblock of even size, else word by word.
template <int NB, int NT>
__device__ __forceinline__ void store_tile(const uint64_t *tile, const uint16_t *stile, int64_t bh, int64_t b0,
                                           int64_t cover, int64_t sub, int64_t nsb, uint64_t *planes_sb,
                                           uint16_t *scales_sb) {
  const int64_t sb0 = b0 / sub, bs0 = b0 - sb0 * sub;
  if ((sub & 1) == 0 && bs0 + NB <= sub) {  // cover is a multiple of sub: all NB blocks are within it
    uint64_t *P = planes_sb + (bh * nsb + sb0) * kD * 4 * sub + bs0;
    for (int e = threadIdx.x; e < kD * 4 * (NB / 2); e += NT) {
      const int u = e / (NB / 2), i = e % (NB / 2);
      *reinterpret_cast<ulonglong2 *>(P + (int64_t)u * sub + 2 * i) =
          *reinterpret_cast<const ulonglong2 *>(&tile[u * NB + tile_slot<NB>(u >> 2, 2 * i)]);
    }
  } else {
    const int bi = threadIdx.x % NB;  // a thread keeps its block: one division
    const int64_t b = b0 + bi, sb = b / sub;
    if (b < cover) {
      uint64_t *P = planes_sb + (bh * nsb + sb) * kD * 4 * sub + (b - sb * sub);
      for (int u = threadIdx.x / NB; u < kD * 4; u += NT / NB)
        P[(int64_t)u * sub] = tile[u * NB + tile_slot<NB>(u >> 2, bi)];
    }
  }
  const int bi = threadIdx.x % NB;
  const int64_t b = b0 + bi, sb = b / sub;
  if (b >= cover) return;
  uint16_t *S = scales_sb + (bh * nsb + sb) * kD * sub + (b - sb * sub);
  for (int j = threadIdx.x / NB; j < kD; j += NT / NB) S[(int64_t)j * sub] = stile[j * NB + bi];
}

// 4 R consecutive blocks per workgroup (CPL = 2: four waves; CPL = 1: eight, two
// per block), R of them per wave: their plane words meet in LDS so that a
// (channel, plane) unit leaves as one run of 32 R bytes (a whole 128-byte line
// with R = 4) in 16-byte stores, where a wave alone writes 8-byte pieces of 512
// lines.
template <int KDT, int CPL, int R>
__global__ __launch_bounds__(512 / CPL, 2) void quantise_tile_kernel(QuantArgs a) {
  constexpr int NB = 4 * R, NT = 512 / CPL;
  __shared__ __align__(16) uint64_t tile[kD * 4 * NB];
  __shared__ __align__(16) uint16_t stile[kD * NB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t bh = blockIdx.y, b0 = (int64_t)blockIdx.x * NB;
  const int j0 = CPL == 2 ? 2 * lane : 64 * (wave & 1) + lane;
  for (int r = 0; r < R; ++r) {
    const int bi = 4 * r + (CPL == 2 ? wave : wave >> 1);
    uint32_t w[CPL][2][4];
    uint16_t s16[CPL];
    block_words<KDT, CPL>(a, bh, b0 + bi, j0, w, s16);
    if (!a.planes_sb) continue;
    const int at = tile_slot<NB>(j0, bi);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
#pragma unroll
      for (int p = 0; p < 4; ++p)
        tile[((j0 + c) * 4 + p) * NB + at] = ((uint64_t)w[c][1][p] << 32) | w[c][0][p];
      stile[(j0 + c) * NB + bi] = s16[c];
    }
  }
  if (!a.planes_sb) return;
  __syncthreads();
  store_tile<NB, NT>(tile, stile, bh, b0, a.cover, a.sub, a.nsb, a.planes_sb, a.scales_sb);
}

// Few blocks: two waves per block, one channel per lane, plane words stored as
// they are made.
template <int KDT>
__global__ __launch_bounds__(256) void quantise_small_kernel(QuantArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t bh = blockIdx.y, b = (int64_t)blockIdx.x * 2 + (wave >> 1);
  if (b >= a.cover) return;
  const int j = 64 * (wave & 1) + lane;
  uint32_t w[1][2][4];
  uint16_t s16[1];
  block_words<KDT, 1>(a, bh, b, j, w, s16);
  if (!a.planes_sb) return;
  const int64_t sb = b / a.sub, bs = b - sb * a.sub;
  uint64_t *P = a.planes_sb + ((bh * a.nsb + sb) * kD + j) * 4 * a.sub + bs;
#pragma unroll
  for (int p = 0; p < 4; ++p) P[p * a.sub] = ((uint64_t)w[0][1][p] << 32) | w[0][0][p];
  a.scales_sb[((bh * a.nsb + sb) * kD + j) * a.sub + bs] = s16[0];
}

// Codes -> logical planes (kernels/bitplane.py:44-50), the quantiser's bit packing
// on loaded codes: CPL channels per lane, 3 - CPL waves per block.  Bound: latency
// of one round of 64 loads below about 1000 blocks (1 x 16384 codes 13.7 -> 3.7
// us), then HBM (8 x 32768: 21 -> 12 us, 5.6 TB/s).
template <int CPL>
__global__ __launch_bounds__(256) void pack128_kernel(const uint8_t *__restrict__ code, int64_t n, int64_t nblk,
                                                      uint64_t *__restrict__ planes) {
  typedef typename std::conditional<CPL == 2, uint16_t, uint8_t>::type raw_t;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t bh = blockIdx.y;
  const int64_t b = CPL == 2 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x * 2 + (wave >> 1);
  if (b >= nblk) return;
  const int j = CPL == 2 ? 2 * lane : 64 * (wave & 1) + lane;
  const int real = (int)min((int64_t)kBlk, n - b * kBlk);
  const uint8_t *src = code + (bh * n + b * kBlk) * kD + j;
  uint32_t raw[kBlk];
#pragma unroll
  for (int i = 0; i < kBlk; ++i) raw[i] = *reinterpret_cast<const raw_t *>(src + min(i, real - 1) * kD);
  uint32_t w[CPL][2][4];
#pragma unroll
  for (int c = 0; c < CPL; ++c)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      uint32_t B[4][2];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint32_t q = 0u;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int i = 32 * half + 4 * (2 * k + h) + m;
            const uint32_t v = i < real ? (raw[i] >> (8 * c)) & 15u : 0u;
            q |= v << (8 * k);
          }
          B[m][h] = q;
        }
      half_planes(B, w[c][half]);
    }
  uint4 *P = reinterpret_cast<uint4 *>(planes + ((bh * nblk + b) * kD + j) * 4);
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    P[2 * c] = make_uint4(w[c][0][0], w[c][1][0], w[c][0][1], w[c][1][1]);
    P[2 * c + 1] = make_uint4(w[c][0][2], w[c][1][2], w[c][0][3], w[c][1][3]);
  }
}

// Workgroup shapes by the number of 64-token blocks, us measured (bf16 keys with
// codes kept / without; f32 keys with codes / without):
//   blocks     small        R = 1        R = 2        R = 4
//     256   8.7/6.8 8.7/6.6   9.5/7.3 9.2/7.7   15/11 15/10   26/18 26/18
//     632   10.9/8.7 12/9.3   10.7/8.3 10.7/9.0   16/12 16/11   27/19 27/19
//    2504   21/19 29/25   23/18 34/27   22/17 33/24   30/21 32/23
//   16384   132/148 182/158   117/80 183/148   108/72 167/127   100/77 165/130
// A wave works its R blocks off one after the other, so few blocks want few per
// wave; the long runs of a whole tile pay once every CU has several workgroups.
// f32 keys take one channel per lane: two would need 128 registers for the keys
// alone (203 us against 127 at 16384 blocks).
template <int KDT>
int launch128(const QuantArgs &a, int64_t lead, hipStream_t st) {
  constexpr int CPL = KDT == FATHOM_DT_F32 ? 1 : 2;
  const int64_t blocks = a.cover * lead;
  const unsigned y = (unsigned)lead;
  if (blocks < 512)
    quantise_small_kernel<KDT><<<dim3((unsigned)cdiv(a.cover, 2), y), 256, 0, st>>>(a);
  else if (blocks < 2048)
    quantise_tile_kernel<KDT, CPL, 1><<<dim3((unsigned)cdiv(a.cover, 4), y), 512 / CPL, 0, st>>>(a);
  else if (blocks < 12288 || !a.code || KDT == FATHOM_DT_F32)
    quantise_tile_kernel<KDT, CPL, 2><<<dim3((unsigned)cdiv(a.cover, 8), y), 512 / CPL, 0, st>>>(a);
  else if constexpr (KDT != FATHOM_DT_F32)
    quantise_tile_kernel<KDT, CPL, 4><<<dim3((unsigned)cdiv(a.cover, 16), y), 512 / CPL, 0, st>>>(a);
  return launch_status("quantise128");
}

bool aligned(const void *p, uintptr_t to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; }

}  // namespace

bool quantise128_accepts(const QuantArgs &a, int k_dtype, int64_t D) {
  return D == kD && aligned(a.K, k_dtype == FATHOM_DT_F32 ? 8 : 4) && aligned(a.code, 2) && aligned(a.planes_log, 16) &&
         aligned(a.planes_sb, 16) && aligned(a.scales_sb, 4);
}

int quantise128(const QuantArgs &a, int k_dtype, int64_t lead, hipStream_t st) {
  switch (k_dtype) {
    case FATHOM_DT_F16: return launch128<FATHOM_DT_F16>(a, lead, st);
    case FATHOM_DT_BF16: return launch128<FATHOM_DT_BF16>(a, lead, st);
    default: return launch128<FATHOM_DT_F32>(a, lead, st);
  }
}

bool pack128_accepts(const uint8_t *code, int64_t D, const uint64_t *planes) {
  return D == kD && aligned(code, 2) && aligned(planes, 16);
}

int pack128(const uint8_t *code, int64_t lead, int64_t n, uint64_t *planes, hipStream_t st) {
  const int64_t nblk = cdiv(n, kBlk);
  const unsigned y = (unsigned)lead;
  if (nblk * lead < 1024)
    pack128_kernel<1><<<dim3((unsigned)cdiv(nblk, 2), y), 256, 0, st>>>(code, n, nblk, planes);
  else
    pack128_kernel<2><<<dim3((unsigned)cdiv(nblk, 4), y), 256, 0, st>>>(code, n, nblk, planes);
  return launch_status("pack128_kernel");
}

}  // namespace pack
}  // namespace fathom
