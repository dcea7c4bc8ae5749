// dsa_dropout.h — attention dropout of the fused kernels (gfx950): the keep
// bit of every (query, key) pair, generated by one small kernel before the
// forward and read by the forward and dkdv kernels.
//
// The reference drops attention probabilities with nn.Dropout
// (deberta_v2_native.py:222, 636): probs * keep / (1 - p), keep ~
// Bernoulli(1 - p) per element.  Here keep comes from Philox4x32-10
// (J. K. Salmon, M. A. Moraes, R. O. Dror, D. E. Shaw, "Parallel random
// numbers: as easy as 1, 2, 3", SC 2011), a counter-based generator: the
// bits of a pair are a function of the pair's coordinates and the call's
// 64-bit seed, so the backward regenerates exactly the forward's mask.
//
// Contract (restated on the CPU in oracle/dropout.py).  For pair (i, j) of
// head h, batch row b, with r = j % 64, jb = r / 16, g = (r % 16) / 4, e = r % 4:
//   counter = ((j / 64) * 8 + g * 2 + jb / 2,  i,  h,  b)
//   key     = (seed & 0xffffffff, seed >> 32)
//   x       = Philox4x32-10(counter, key)          (four 32-bit words)
//   u       = (jb % 2) * 4 + e;   v = (x[u / 2] >> (16 * (u % 2))) & 0xffff
//   keep    = v >= t
// where t in [1, 65535] is the call's threshold: a pair is dropped with
// probability t / 65536 exactly, and kept probabilities are scaled by
// 65536 / (65536 - t).  One Philox call covers the eight keys of one query
// that a lane of the forward holds in two of its 16 x 16 score tiles.
//
// Bit layout: one 32-bit word per (b, h, 32-query block qb, 64-key tile kt,
// lane), word index ((((b H + h) NQB + qb) NKT + kt) 64 + lane) with NQB =
// LqP / 32, NKT = LkP / 64, in the order the forward's lanes hold the pairs
// (lane = 16 g + c16, query column c16, key group g): bit 16 ib + 4 jb + e
// is the pair (32 qb + 16 ib + c16, 64 kt + 16 jb + 4 g + e).  A forward
// lane reads one word per key tile; a dkdv lane (keys down) reads the four
// words of lanes 16 (c16' / 4) + 4 g' .. + 3, 16 contiguous bytes.
#pragma once

#include "dsa_common.h"

namespace dsa {

// Philox4x32 round constants: the multipliers and the Weyl increments of the
// key schedule, from the paper above.
constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u;
constexpr uint32_t kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;

// a ^ b ^ k in one VALU instruction, k uniform: gfx950's three-input
// bitwise operation with truth table 0x96 (the parity of its three inputs;
// the compiler emits two XORs for the expression)
DSA_DEV uint32_t xor3_uniform(uint32_t a, uint32_t b, uint32_t k) {
  uint32_t r;
  asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(r) : "v"(a), "v"(b), "s"(k));
  return r;
}

// Ten rounds of Philox4x32 on counter (c0, c1, c2, c3) with key (k0, k1),
// the key uniform over the wave.  Each round: (hi0, lo0) = M0 * c0, (hi1,
// lo1) = M1 * c2 (64-bit products, one v_mad_u64_u32 each), c <- (hi1 ^ c1
// ^ k0, lo1, hi0 ^ c3 ^ k1, lo0); the key is bumped by the Weyl increments
// between rounds.
DSA_DEV uint4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)kPhiloxM0 * c0;
    const uint64_t p1 = (uint64_t)kPhiloxM1 * c2;
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    c0 = xor3_uniform(hi1, c1, k0);
    c1 = lo1;
    c2 = xor3_uniform(hi0, c3, k1);
    c3 = lo0;
    k0 += kPhiloxW0;
    k1 += kPhiloxW1;
  }
  return make_uint4(c0, c1, c2, c3);
}

// The eight keep bits of one Philox output (bit u: 16-bit value u >= t).
DSA_DEV uint32_t keep8(uint4 x, uint32_t t) {
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
  uint32_t m = 0;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const uint32_t v = (u & 1) ? (w[u >> 1] >> 16) : (w[u >> 1] & 0xffffu);
    m |= (v >= t ? 1u : 0u) << u;
  }
  return m;
}

struct DropParams {
  uint32_t* bits;   // the words, laid out as above
  int B, H, NQB, NKT;
  uint32_t t;       // threshold in [1, 65535]
  uint32_t k0, k1;  // the seed's low and high words
};

// Index of the word of (b, h, 32-query block qb, 64-key tile kt, lane 0).
DSA_DEV int64_t drop_word0(int b, int h, int H, int NQB, int NKT, int qb, int kt) {
  return ((((int64_t)b * H + h) * NQB + qb) * NKT + kt) * 64;
}

// Bytes of the keep bits for these extents (LqP, LkP multiples of 128).
inline size_t dropout_bits_bytes(int B, int H, int LqP, int LkP) {
  return (size_t)B * H * (size_t)(LqP / 32) * (size_t)(LkP / 64) * 64 * sizeof(uint32_t);
}

// One thread per word: four Philox calls (two query rows, two halves of the
// key group's 16 keys).  Grid (ceil(NKT / 4) * NQB, H, B): a workgroup takes
// four 64-key tiles of one 32-query block, one wave per tile (a wave past
// NKT ends at once); consecutive threads write consecutive words.
static __global__ __launch_bounds__(256) void dsa_dropout_bits_kernel(DropParams d) {
  const int nx = (d.NKT + 3) / 4;
  const int qb = blockIdx.x / nx;
  const int kt = (blockIdx.x % nx) * 4 + (threadIdx.x >> 6);
  if (kt >= d.NKT) return;
  const int h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int64_t w = drop_word0(b, h, d.H, d.NQB, d.NKT, qb, kt) + lane;
  const int g = lane >> 4, c16 = lane & 15;
  uint32_t word = 0;
#pragma unroll
  for (int ib = 0; ib < 2; ++ib) {
    const uint32_t i = (uint32_t)(32 * qb + 16 * ib + c16);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t c0 = (uint32_t)(kt * 8 + g * 2 + half);
      word |= keep8(philox4x32_10(c0, i, (uint32_t)h, (uint32_t)b, d.k0, d.k1), d.t) << (16 * ib + 8 * half);
    }
  }
  d.bits[w] = word;
}

}  // namespace dsa
