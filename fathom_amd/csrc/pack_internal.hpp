// Store builders shared between pack.hip (general shapes) and quantise.hip
// (D = 128 rows).
#pragma once
#include "common.hpp"

namespace fathom {
namespace pack {

// One quantise call: keys [lead, n, 128] in, every output optional (null).
struct QuantArgs {
  const void *K;
  int64_t n, nblk, cover, sub, nsb;  // cover: blocks written per row (nsb * sub with a superblock store)
  int sdt;                           // FATHOM_DT_* of the block scale
  uint8_t *code;
  void *scales_blk;
  uint64_t *planes_log, *planes_sb;
  uint16_t *scales_sb;
};

// Whether quantise128 takes the call: D = 128 and every pointer aligned to its
// loads and stores.
bool quantise128_accepts(const QuantArgs &a, int k_dtype, int64_t D);
int quantise128(const QuantArgs &a, int k_dtype, int64_t lead, hipStream_t st);

// The logical planes of D = 128 codes.
bool pack128_accepts(const uint8_t *code, int64_t D, const uint64_t *planes);
int pack128(const uint8_t *code, int64_t lead, int64_t n, uint64_t *planes, hipStream_t st);

}  // namespace pack
}  // namespace fathom
