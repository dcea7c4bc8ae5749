// dsa_pair.h — dense pair masks as bits (gfx950): one pass over the byte mask
// [B or 1, H or 1, Lq, Lk] into one bit a pair, in the order the forward's
// lanes hold the pairs, and two flags per tile of 32 queries x 64 keys.
//
// The kernels that apply the mask then read one word a lane and tile (the
// layout of dropout's keep bits, dsa_dropout.h) instead of testing bytes, skip
// the tiles without a kept pair and leave the tiles whose pairs are all kept
// unmasked, as they do under segment masks.  A bit is set iff the pair is
// kept, its query's diagonal is set (a live row) and both tokens lie inside
// the sequence.
//
// Bound by the read of the mask (16-byte loads, 2 KB a wave): one wave per
// tile, the two 32-key halves of a row in neighbouring lanes, turned into the
// forward's lane order with four shuffles.
//
// A window with a global token, [4, 12, 1000, 64] bf16 (4 MB of mask, one pass
// in the forward's preparation and one in the backward's): forward 112 -> 66
// us, dkdv 194 -> 83, dq and tables 76 -> 48, preparation 12 -> 19.  The bits
// are used wherever there is room for them, since they also pay where no tile
// can be skipped: half of the pairs kept at random, training pass, bytes ->
// bits: [16, 12, 512] 416 -> 284 us, [4, 12, 1000] 405 -> 292 (dropout 469 ->
// 317), [2, 12, 2048] 760 -> 429, float32 [4, 12, 512] 420 -> 387; causal
// 412 -> 250, 408 -> 293, 781 -> 346.
#pragma once

#include "dsa_tiles.h"

namespace dsa {

// Masks held: one per (batch row, head) that differs (a stride of 0 broadcasts).
inline int64_t pair_masks(int B, int H, int64_t pkb, int64_t pkh) { return (pkb ? B : 1) * (int64_t)(pkh ? H : 1); }

// Bits of the four bytes of v (bit k: byte k is nonzero).
DSA_DEV uint32_t nonzero_bytes(uint32_t v) {
  v |= v >> 4;
  v |= v >> 2;
  v |= v >> 1;
  return ((v & 0x01010101u) * 0x10204080u) >> 28;
}

struct PairBits {
  const uint8_t* pk;
  int64_t pkb, pkq, pkh;  // byte strides of batch row, query and head
  uint32_t* bits;         // FwdParams::pbits
  uint8_t* flags;         // FwdParams::pflag
  int B, H, Lq, Lk, LqP, LkP;
};

// Waves (tiles) of a call; a block of 256 threads takes four.
inline int64_t pair_tiles(const PairBits& t) {
  return pair_masks(t.B, t.H, t.pkb, t.pkh) * (t.LqP / 32) * (t.LkP / 64);
}

DSA_DEV void pair_bits_block(const PairBits& t, int64_t blk) {
  const int nqb = t.LqP / 32, nkt = t.LkP / 64, nh = t.pkh ? t.H : 1;
  const int64_t tile = blk * 4 + (threadIdx.x >> 6);
  const int64_t n = (int64_t)(t.pkb ? t.B : 1) * nh * nqb * nkt;
  if (tile >= n) return;
  const int lane = threadIdx.x & 63;
  const int kt = (int)(tile % nkt), qb = (int)(tile / nkt % nqb);
  const int64_t m = tile / ((int64_t)nkt * nqb);
  const uint8_t* base = t.pk + (m / nh) * t.pkb + (m % nh) * t.pkh;
  // lane: row lane / 2, keys [64 kt + 32 (lane % 2), + 32)
  const int i = 32 * qb + (lane >> 1), j = 64 * kt + 32 * (lane & 1);
  uint32_t bits = 0;
  if (i < t.Lq) {
    const uint8_t* row = base + (int64_t)i * t.pkq;
    if (row[i]) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // (a 16-key chunk that starts below Lk lies in the row's allocation)
        if (j + 16 * u < t.Lk) {
          const uint4 v = *reinterpret_cast<const uint4*>(row + j + 16 * u);
          bits |= (nonzero_bytes(v.x) | nonzero_bytes(v.y) << 4 | nonzero_bytes(v.z) << 8 | nonzero_bytes(v.w) << 12)
                  << (16 * u);
        }
      }
      if (j + 32 > t.Lk) bits &= j < t.Lk ? (1u << (t.Lk - j)) - 1u : 0u;
    }
  }
  const bool any = __ballot(bits != 0) != 0, all = __ballot(bits == 0xffffffffu) == ~0ull;
  // lane (g, c16): bit 16 ib + 4 jb + e is the pair (16 ib + c16, 16 jb + 4 g + e)
  const int g = lane >> 4, c16 = lane & 15;
  uint32_t word = 0;
#pragma unroll
  for (int ib = 0; ib < 2; ++ib)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t src = (uint32_t)__shfl((int)bits, 2 * (16 * ib + c16) + half);
      word |= ((src >> (4 * g)) & 0xfu) << (16 * ib + 8 * half);
      word |= ((src >> (16 + 4 * g)) & 0xfu) << (16 * ib + 8 * half + 4);
    }
  t.bits[tile * 64 + lane] = word;
  if (lane == 0) t.flags[tile] = (any ? 1 : 0) | (all ? 2 : 0);
}

// Index of (batch row, head)'s mask among the masks held.
DSA_DEV int64_t pair_index(const FwdParams& p, int b, int h) {
  return (p.pkb ? b : 0) * (int64_t)(p.pkh ? p.H : 1) + (p.pkh ? h : 0);
}
// Flags of query block qb (32 queries): one byte per 64-key tile.
DSA_DEV const uint8_t* pair_flags(const FwdParams& p, int64_t m, int qb) {
  return p.pflag + (m * (p.LqP / 32) + qb) * (p.LkP / 64);
}
// Whether query chunk c (32 queries) and key tile k (128 keys) hold a kept
// pair: the tiles the dkdv kernel computes and writes (ChunkRange's part
// under a pair mask).
DSA_DEV bool pair_active(const FwdParams& p, int64_t m, int c, int k) {
  return (*reinterpret_cast<const uint16_t*>(pair_flags(p, m, c) + 2 * k) & 0x0101u) != 0;
}

}  // namespace dsa
