// dsa_bwd_dkdv.h — dK, dV and dS of the fused disentangled attention
// (gfx950).
//
// One workgroup = 4 waves = one (batch b, head h, 128-key tile); wave w owns
// keys [j0 + 32w, j0 + 32w + 32) and streams 32-query tiles.  The tiles (Q,
// dO, the saved relative term, lse and Delta, and a 32-offset block of
// qrgt) are double-buffered in LDS and filled by direct global-to-LDS copies
// issued one tile ahead; K and V of the wave's keys stay in registers.  Per
// tile:
//   scores        y = Q K^T + bias (unscaled), queries down / keys across,
//                 where bias = c2p + p2c is the relative term the forward
//                 saved (read transposed from the LDS tile)
//   P, dP, dS     P = exp2(y * scale*log2e - lse*log2e), dP = dO V^T,
//                 dS = P (dP - Delta)
//   dS            staged transposed in the wave's LDS tile (rows j), then
//                 stored to the workspace in rows i (4 consecutive keys per
//                 lane, read back transposed): the dq and table kernels
//                 read it
//   dV^T         += dO^T P,  dK^T += Q^T dS        (dO^T, Q^T read transposed)
//   p2c          dK^T[d][j] += sum_x qrgt[d][t0 + x] F[x][j], F[x][j] =
//                dS(i0 + x + (j - jw) - 31, j): x = (i - i0) - (j - jw) + 31 is
//                the wave's offset index and qrgt holds the Qr rows gathered
//                per offset and transposed.  The wave's dS^T tile in LDS
//                (rows j, 32 zero columns before each row) makes F's
//                operand eight consecutive elements of one row; the
//                qrgt window (160 offsets of the workgroup) is a ring of
//                32-offset blocks, one new block per tile.
// Every query tile of the padded extent is visited, so dS is fully written
// (zeros for masked pairs, dead rows and padding), or, under a mask, the
// listed tiles are and the others are neither written nor read.
#pragma once

#include "dsa_bwd.h"
#include "dsa_dropout.h"

namespace dsa {

namespace kvcfg {
constexpr int NW = 4, WK = 32, BKW = 128, BQ = 32;
}  // namespace kvcfg

// DROP: attention dropout with the forward's keep bits p.drop
// (dsa_dropout.h): dV sums the kept probabilities, scaled by p.drop_scale,
// and dP keeps the kept pairs' dO . v, scaled the same way.
// FAR: calls that look for far blocks (FarSpan, p.far); kept out of the others'
// code, whose registers are all taken (250 of 256).  Its near tiles are slower
// than the others' (49 to 90 scalar registers spill to vector lanes): at B=4,
// L=2048, H=12 with 52% of the blocks far, 286 -> 292 us where the forward goes
// from 274 to 230 and DQ|TABLE from 326 to 224 (far_call has the rule).
template <typename T, int D, int MASK, bool DROP, bool FAR>
__global__ __launch_bounds__(256, 2) void dsa_bwd_dkdv_kernel(BwdParams bp) {
  using namespace kvcfg;
  using M = Mfma<T>;
  typedef typename M::frag frag;
  typedef typename BandType<T>::type BT;
  using SQ = Swz<T, D>;
  constexpr int NS = D / M::KSTEP;
  constexpr int ND = D / 16;
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int QCH = BQ * D * (int)sizeof(T) / 16;   // 16-byte chunks of a Q (or dO) tile
  constexpr int QCW = QCH / NW;                         // ... per wave
  constexpr int BE = 2 * 2048;                          // saved-bias elements of a tile
  constexpr int BCW = BE * (int)sizeof(BT) / 16 / NW;   // bias chunks per wave
  constexpr int FE = M::FRAG_ELEMS;
  // dS^T tile of a wave: rows j (32 + 1), ZL zero columns, 32 data columns,
  // the rest of the stride zero; a row's right-hand zeros continue into the
  // next row's leading ones.
  constexpr int ZL = 32;
  constexpr int SROW = sizeof(T) == 2 ? 72 : 76;         // few bank conflicts for 16-byte row reads
  // (the last row's right-hand zeros: the walk reads up to 26 elements past it)
  constexpr int SW = WK * SROW + 32;
  // qrgt ring: NRB blocks of 32 offsets, each stored [chunk c][d][VEC] so that
  // a fragment read (one chunk of 16 consecutive d rows) is contiguous.
  constexpr int NRB = 6, RBE = 32 * D;
  constexpr int RCPB = RBE / VEC;                        // 16-byte chunks per block
  const FwdParams& p = bp.f;

  // Double-buffered tiles, filled by LDS copies issued one tile ahead.  The
  // two buffers are distinct arrays and the loop is unrolled by two, so the
  // compiler sees that a tile's reads do not touch the buffer the next
  // tile's copies are landing in (it would otherwise wait for those copies
  // before every read).
  __shared__ __align__(16) T Qs0[BQ * D], Qs1[BQ * D];
  __shared__ __align__(16) T dOs0[BQ * D], dOs1[BQ * D];
  __shared__ __align__(16) BT Bs0[BE], Bs1[BE];
  __shared__ __align__(16) float Rs0[2 * BQ], Rs1[2 * BQ];  // per query: lse*log2e (inf: no probabilities), Delta
  __shared__ __align__(16) T Ring[NRB * RBE];     // qrgt window (p2c)
  __shared__ __align__(16) T Stg[NW * SW];        // each wave's dS^T tile
  // dropout: each wave's keep words of the tile (one per lane), double-buffered
  __shared__ __align__(16) uint32_t Dk0[DROP ? NW * 64 : 1], Dk1[DROP ? NW * 64 : 1];
  static_assert(MASK != MASK_PAIR, "pair masks come as bits");
  constexpr bool SEGM = seg_mode(MASK);
  constexpr bool BITS = MASK == MASK_BITS;
  constexpr bool LIST = SEGM || BITS;  // the query tiles to visit are listed
  constexpr int MAXQT = 1024;  // query tiles (Lq <= 32768)
  // segment masks: the active query tiles in order (tile | 0x4000 if it
  // needs no masking), FAR: the far ones of either side, then the near ones;
  // query segments of MASK_SEG tiles
  __shared__ short qlist[LIST ? MAXQT : 1];
  __shared__ int qlen[3];
  __shared__ __align__(16) int qsg[MASK == MASK_SEG ? 2 : 1][MASK == MASK_SEG ? BQ : 1];
  // pair bits: each wave's words of the tile, as dropout's keep words (with
  // dropout, whose words fill the LDS of two workgroups a CU, each lane holds
  // its four in registers)
  constexpr bool PLDS = BITS && !DROP;
  __shared__ __align__(16) uint32_t Pk0[PLDS ? NW * 64 : 1], Pk1[PLDS ? NW * 64 : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  // SCAL: the wave index is known to the compiler as uniform, and the copies'
  // addresses are scalar bases and small per-lane offsets: 20 to 30 vector
  // registers fewer, which the far loops (with 64-bit addresses a lane they
  // spilled in the near loop: 339 against 276 us at B=4, L=2048, H=16) and the
  // kernels with per-element mask tests need, for more scalar ones, which
  // spill to vector lanes and cost the others up to 6% (dropout at B=12,
  // L=512: 85.7 against 80.8 us; documents with dropout at B=32, whose kernel
  // fits without: 71.1 against 69.0).
  constexpr bool SCAL = FAR || (MASK == MASK_SEG && !DROP) || BITS;
  const int w = SCAL ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
  const int g = (tid & 63) >> 4, c16 = tid & 15;
  // one 16-byte LDS copy: byte offset off (lane part) from the uniform base
  auto copy16 = [&](const void* base, unsigned off, void* lds_wave) {
    if constexpr (SCAL) lds_dma16_s(base, off, lds_wave);
    else lds_dma16((const char*)base + off, lds_wave);
  };
  const int Lq = p.Lq, Lk = p.Lk;
  const int NKT = p.LkP / BKW;
  // (b, h, kt), kt fastest; with an order (masks), item order[r / H] and
  // head r % H, heaviest first
  int kt, h, b;
  if (bp.korder) {
    const int it = __builtin_amdgcn_readfirstlane(bp.korder[blockIdx.x / p.H]);
    h = blockIdx.x % p.H, kt = it % NKT, b = it / NKT;
  } else {
    const int m = xcd_remap(blockIdx.x, gridDim.x);
    kt = m % NKT, h = (m / NKT) % p.H, b = m / (NKT * p.H);
  }
  const bool p2c = (p.flags & 2) != 0;
  const float sl2 = p.scale * kLog2e;
  const int nqt = p.LqP / BQ;

  const int j0 = kt * BKW;
  const int jw = j0 + w * WK;
  const T* qbase = (const T*)p.q + (int64_t)b * p.qs[0] + (int64_t)h * p.qs[2];
  const T* kbase = (const T*)p.k + (int64_t)b * p.ks[0] + (int64_t)h * p.ks[2];
  const T* vbase = (const T*)p.v + (int64_t)b * p.vs[0] + (int64_t)h * p.vs[2];
  const T* dobase = (const T*)bp.dout + (int64_t)b * bp.dos[0] + (int64_t)h * bp.dos[2];
  const BT* biasb = (const BT*)p.bias;
  const float* rib = bp.rowinfo + (int64_t)(b * p.H + h) * p.LqP * 2;
  const int64_t riplane = (int64_t)p.B * p.H * p.LqP * 2;  // far blocks: the planes of the two sides follow
  FarSpan fs{kNoFar, -kNoFar};
  if constexpr (FAR) fs = far_span_of(bp);
  int64_t pmask = 0;  // pair bits: the mask of (b, h)
  if constexpr (BITS) pmask = pair_index(p, b, h);
  const SegView<MASK> sv(p, b);
  T* dsw = (T*)bp.ds + (int64_t)(b * p.H + h) * p.LqP * p.LkP + jw;  // dS column jw, row 0
  const T* qrg = p2c ? (const T*)bp.qrgt + (int64_t)h * D * bp.TGP : nullptr;
  // qrgt column of the workgroup window's first offset at query tile 0
  // (a multiple of 32: t = d + OFF with d = -j0 - 127)
  const int tw0 = -j0 - (BKW - 1) + bp.OFF;
  T* stg = Stg + w * SW;

  int jcol[2], jseg[2] = {0, 0};
  bool jkeep[2];
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
    const int j = jw + 16 * jb + c16;
    jcol[jb] = j;
    if (SEGM && j < Lk) jseg[jb] = sv(j);
    jkeep[jb] = j < Lk && (!SEGM || jseg[jb] != 0);
  }
  // Segment masks and pair bits: the query tiles that meet this key tile (ChunkRange; the tile flags),
  // listed by wave 0 (one chunk per lane); the others are neither computed
  // nor written.
  // FAR: the far tiles past neg (queries before the keys) come first, then
  // the far ones past pos, then the near ones: n1, n2 and nlist end the three
  // parts, each a loop of its own.  The near loop's registers are all taken
  // (a spill in it waits for the next tile's copies), and last it carries
  // nothing of the others.
  bool any_key;
  int nlist = nqt, n1 = 0, n2 = 0, qhi = 0;
  if constexpr (FAR) {
    // far: the tiles below n1 and from qhi on
    n1 = min(max((128 / BQ) * (kt + fs.neg + 1), 0), nqt);
    qhi = min(max((128 / BQ) * (kt + fs.pos), 0), nqt);
    n2 = n1 + nqt - qhi;
  }
  if constexpr (LIST) {
    ChunkRange kr{0, 0, 0};
    if constexpr (SEGM) kr = key_tile_range(bp.cinfo + (int64_t)b * nqt, kt, nqt);
    if (w == 0) {
      int n = 0;
#pragma unroll 1
      for (int part = 0; part < (FAR ? 3 : 1); ++part) {
        const int from = part == 0 ? 0 : part == 1 ? qhi : n1;
        const int to = !FAR || part == 1 ? nqt : part == 0 ? n1 : qhi;
        for (int c0 = from; c0 < to; c0 += 64) {
          const int c = c0 + lane;
          bool act = false, full = false;
          if (c < to) {
            if constexpr (SEGM) {
              const ChunkRange x = chunk_range(bp.cinfo + (int64_t)b * nqt, c);
              act = x.meets(kr);
              full = act && x.all && kr.all && x.lo == x.hi && kr.lo == kr.hi && x.lo == kr.lo;
            } else {
              const unsigned f = *reinterpret_cast<const uint16_t*>(pair_flags(p, pmask, c) + 2 * kt);
              act = (f & 0x0101u) != 0;
              full = (f & 0x0202u) == 0x0202u;
            }
          }
          n = wave_append(act, (short)(c | (full ? 0x4000 : 0)), qlist, n);
        }
        if (lane == 0) qlen[part] = n;
      }
    }
    __syncthreads();
    if constexpr (FAR) {
      n1 = __builtin_amdgcn_readfirstlane(qlen[0]);
      n2 = __builtin_amdgcn_readfirstlane(qlen[1]);
    }
    nlist = __builtin_amdgcn_readfirstlane(qlen[FAR ? 2 : 0]);
    any_key = nlist > 0;
  } else {
    any_key = __syncthreads_or(tid < BKW && j0 + tid < Lk);
  }

  f32x4 dka[ND][2], dva[ND][2];
#pragma unroll
  for (int db = 0; db < ND; ++db) dka[db][0] = dka[db][1] = dva[db][0] = dva[db][1] = zero4();

  // Issues the LDS copies of qrgt block rb (columns [32 rb, 32 rb + 32)) into
  // ring slot rb % NRB: chunk c of row d at ((c * D) + d) * VEC.
  typedef T vecT __attribute__((ext_vector_type(VEC)));
  auto issue_ring = [&](int rb) {
    T* slot = Ring + (rb % NRB) * RBE;
#pragma unroll
    for (int k = 0; k < (RCPB + 255) / 256; ++k) {
      if (256 * k + w * 64 < RCPB) {
        char* dst = (char*)(slot + (256 * k + w * 64) * VEC);
        if constexpr (SCAL) {
          const int c = (256 * k + w * 64) / D + lane / D, d = lane % D;  // D divides 64
          lds_dma16_s(qrg + 32 * rb, (unsigned)((d * bp.TGP + c * VEC) * (int)sizeof(T)), dst);
        } else {
          const int pc = 256 * k + w * 64 + lane;
          lds_dma16(qrg + (int64_t)(pc % D) * bp.TGP + 32 * rb + (pc / D) * VEC, dst);
        }
      }
    }
  };

  // Dropout: the forward's 64 keep words of the 32-query block qi and the
  // 64-key tile of the wave's keys (dsa_dropout.h), copied to LDS with the
  // tile (16 lanes x 16 bytes).  The pair (query i0 + 16 ib + 4 g + e, key
  // jw + 16 jb + c16) is bit 16 ib + 4 (2 (w % 2) + jb) + c16 % 4 of the word
  // of forward lane 16 (c16 / 4) + 4 g + e: a lane's four words are 16
  // contiguous bytes.
  const uint32_t *dropw = nullptr, *pairw = nullptr;
  const int NKT64 = p.LkP / 64;
  if constexpr (BITS) pairw = p.pbits + (pmask * nqt * NKT64 + jw / 64) * 64;
  if constexpr (DROP) dropw = p.drop + drop_word0(b, h, p.H, p.LqP / 32, NKT64, 0, jw / 64);
  // Issues the LDS copies of query tile qi into the given buffers (lane
  // order = physical chunk order; Q and dO rows are clamped to Lq - 1, where
  // probabilities are zero anyway) and the last nring blocks of its qrgt
  // window (one from the tile before, whose ring slot was last read two tiles
  // earlier; five for the first near tile after far ones); with dropout, the
  // wave's keep words, under a pair mask its bits.  side: the far side of a
  // far tile, or -1.
  uint4 pnext = {0, 0, 0, 0};  // pair bits in registers: the lane's words of the next tile
  int qseg_next = 0;  // MASK_SEG: query segment of lane (w = 1, lane < 32) in the next tile
  auto issue = [&](int qi, int nring, int side, T* Qd, T* dOd, BT* Bd, float* Rd, uint32_t* Dd, uint32_t* Pd) {
    const int i0 = qi * BQ;
    if (MASK == MASK_SEG && w == 1 && lane < BQ) qseg_next = (i0 + lane < Lq) ? sv(i0 + lane) : 0;
#pragma unroll
    for (int k = 0; k < (QCW + 63) / 64; ++k) {
      const int pc = w * QCW + 64 * k + lane;  // physical chunk
      if (64 * k + lane < QCW) {
        const int r = pc / SQ::CPR, lc = (pc % SQ::CPR) ^ (r & (SQ::CPR - 1));
        const int64_t i = min(i0 + r, Lq - 1);
        lds_dma16(qbase + i * p.qs[1] + lc * SQ::VEC, (char*)Qd + (w * QCW + 64 * k) * 16);
        lds_dma16(dobase + i * bp.dos[1] + lc * SQ::VEC, (char*)dOd + (w * QCW + 64 * k) * 16);
      }
    }
    if (p.flags && side < 0) {
      // two 2048-element blocks of the saved term: forward wave block
      // (i0 % 128) / 32 of forward key tiles j0/64 and j0/64 + 1
      constexpr int CPB = 2048 * (int)sizeof(BT) / 16;
#pragma unroll
      for (int k = 0; k < BCW / 64; ++k) {
        // of lane 0 (SCAL; a wave's 64 chunks lie in one block) or the lane
        const int pc = w * BCW + 64 * k + (SCAL ? 0 : lane);
        const BT* src = biasb + bias_tile_offset(b, h, p.H, i0 / 128, j0 / 64 + pc / CPB, p.LqP, p.LkP) +
                        ((i0 % 128) / 32) * 2048 + (pc % CPB) * (16 / (int)sizeof(BT));
        char* dst = (char*)Bd + (w * BCW + 64 * k) * 16;
        if constexpr (SCAL) lds_dma16_s_nt(src, lane * 16, dst);  // read once: non-temporal
        else lds_dma16_nt(src, dst);
      }
    }
    if (w == 0 && lane < 2 * BQ * 4 / 16)
      copy16(rib + (FAR ? (1 + side) * riplane : 0) + 2 * i0, lane * 16, (char*)Rd);
    if (p2c) {
      if constexpr (FAR) {
        for (int r = 5 - nring; r < 5; ++r) issue_ring(tw0 / 32 + qi + r);
      } else {
        if (nring) issue_ring(tw0 / 32 + qi + 4);
      }
    }
    if (BITS && !PLDS) pnext = *reinterpret_cast<const uint4*>(pairw + (int64_t)qi * NKT64 * 64 + 16 * (c16 >> 2) + 4 * g);
    if (PLDS && lane < 16) copy16(pairw + (int64_t)qi * NKT64 * 64, lane * 16, (char*)(Pd + w * 64));
    if (DROP && lane < 16) copy16(dropw + (int64_t)qi * NKT64 * 64, lane * 16, (char*)(Dd + w * 64));
  };

  typedef T vec4 __attribute__((ext_vector_type(4)));
  // dS rows i of the wave's 32 keys: lane (g, c16) writes keys jw + 8g +
  // [0, 8) of query i0 + 16 mi + c16, one 16-byte store (bf16; two for
  // fp32): NST store instructions per tile.
  typedef T vec8 __attribute__((ext_vector_type(8)));
  constexpr int NST = (BQ / 16) * (int)(sizeof(vec8) / 16);
  auto store_ds = [&](int i0, int mi, const vec8& v) {
    *reinterpret_cast<vec8*>(dsw + (int64_t)(i0 + 16 * mi + c16) * p.LkP + 8 * g) = v;
  };
  if (!any_key) {
    if (!LIST)
      for (int qi = 0; qi < nqt; ++qi)
#pragma unroll
        for (int mi = 0; mi < BQ / 16; ++mi) store_ds(qi * BQ, mi, vec8{});
  } else {
    // K and V rows of the wave's keys stay in registers (B operands)
    frag kf[2][NS], vf[2][NS];
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      const int j = jcol[jb];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        kf[jb][s] = (j < Lk) ? M::load_contig(kbase + (int64_t)j * p.ks[1], s, g) : M::zero();
        vf[jb][s] = (j < Lk) ? M::load_contig(vbase + (int64_t)j * p.vs[1], s, g) : M::zero();
      }
    }
    {
      // zero the wave's dS^T tile (its zero columns are never written)
      vecT z;
#pragma unroll
      for (int e = 0; e < VEC; ++e) z[e] = (T)0.0f;
      static_assert(SW % VEC == 0, "whole chunks");
      for (int c = lane; c < SW / VEC; c += 64) reinterpret_cast<vecT*>(stg)[c] = z;
      // without relative terms no saved term is copied in: the bias buffers
      // hold zeros, so the scores add them unconditionally (no branch per
      // product block)
      if (!p.flags) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        constexpr int NCH = BE * (int)sizeof(BT) / 16;
        for (int c = tid; c < NCH; c += 256) {
          reinterpret_cast<u4*>(Bs0)[c] = u4{0u, 0u, 0u, 0u};
          reinterpret_cast<u4*>(Bs1)[c] = u4{0u, 0u, 0u, 0u};
        }
      }
    }
    // Unmasked workgroups whose 128 keys all lie below Lk: on query tiles
    // below Lq every row is live and every pair kept, so P needs no keep
    // test per element.
    const bool keys_in = MASK == MASK_NONE && j0 + BKW <= Lk;
    // The qrgt ring holds blocks [qi, qi + 4] of the window (relative to
    // tw0 / 32) while tile qi is computed; block qi + 5 lands in the sixth
    // slot meanwhile when the next tile is qi + 1.  The first window:
    auto entry = [&](int n) {
      if constexpr (LIST) return __builtin_amdgcn_readfirstlane(qlist[n]);
      if constexpr (!FAR) return n;
      return n < n1 ? n : n < n2 ? qhi + n - n1 : n1 + n - n2;
    };
    // the tile of an entry: a list entry has its flag above 10 bits; a call
    // without a list may have more tiles, below 2^18 (the padded dS slice, at
    // least 128 keys wide, is below 2 GiB; the compiler is told, since without
    // a bound the unmasked kernel spills 13 registers)
    auto tile_of = [&](int ent) { return ent & (LIST ? 0x3ff : 0x3ffff); };
    const int qfirst = tile_of(entry(0));
    if (!FAR || n2 == 0) {
      if (p2c)
        for (int r = 0; r < 4; ++r) issue_ring(tw0 / 32 + qfirst + r);
      issue(qfirst, 1, -1, Qs0, dOs0, Bs0, Rs0, Dk0, Pk0);
    } else {
      // the near part's first tile is to find its buffers first
      if (n2 & 1) issue(qfirst, 0, n1 > 0 ? 1 : 0, Qs1, dOs1, Bs1, Rs1, Dk1, Pk1);
      else issue(qfirst, 0, n1 > 0 ? 1 : 0, Qs0, dOs0, Bs0, Rs0, Dk0, Pk0);
    }
    lds_dma_wait();
    // Far tiles, one side at a time: the p2c term of the lane's keys and the
    // column sums of dS (every row of the A operand is ones).
    float fb[2] = {0.f, 0.f};
    f32x4 fcs[2] = {zero4(), zero4()};
    auto tile = [&](auto farkind, int n, const T* Q, const T* dO, const BT* Bt, const float* R, const uint32_t* Dw,
                    const uint32_t* Pw, T* nQ, T* ndO, BT* nBt, float* nR, uint32_t* nDw, uint32_t* nPw) {
      constexpr bool far = decltype(farkind)::value;
      const int ent = entry(n);
      const int qi = tile_of(ent), i0 = qi * BQ;
      // This wave's copies of tile qi have landed: they were issued before
      // the previous tile's NST dS stores, its last vector-memory
      // instructions (tile 0 was waited for before the loop).
      vm_wait<NST>();
      if (MASK == MASK_SEG && w == 1 && lane < BQ) qsg[n & 1][lane] = qseg_next;
      __syncthreads();  // ... every wave's, and the previous tile is no longer read
      if (LIST && !far && p2c && n > n2) {
        // after skipped tiles: the blocks of this tile's window not in the
        // ring yet (their slots hold blocks no longer needed)
        const int pv = __builtin_amdgcn_readfirstlane(qlist[n - 1]) & 0x3ff;
        if (qi > pv + 1) {
          for (int x = max(qi, pv + 5); x <= qi + 4; ++x) issue_ring(tw0 / 32 + x);
          vm_wait<0>();
          __syncthreads();
        }
      }
      const uint4 pcur = pnext;
      if (n + 1 < nlist) {
        const int qn = tile_of(entry(n + 1));
        if constexpr (far) issue(qn, n + 1 == n2 ? 5 : 0, n + 1 < n1 ? 1 : n + 1 < n2 ? 0 : -1, nQ, ndO, nBt, nR, nDw, nPw);
        else issue(qn, qn == qi + 1, -1, nQ, ndO, nBt, nR, nDw, nPw);
      }
      // A listed tile marked full needs no masking.  Without a list, a tile
      // past Lq stores zeros.
      const bool full = LIST && (ent & 0x4000);
      const bool skip = !LIST && i0 >= Lq;
      if (skip) {
#pragma unroll
          for (int mi = 0; mi < BQ / 16; ++mi) store_ds(i0, mi, vec8{});
        return;
      }

      // ---- scores (queries down, keys across): Q K^T + saved bias (unscaled) --------------------
      // The products run at a raised wave priority and the P / dS arithmetic
      // at the normal one, so that the SIMD's other wave fills in (dkdv
      // 158.2 -> 156.8 us in one process).
      __builtin_amdgcn_s_setprio(1);
      const float one = opaque_one();
      f32x4 sc[2][BQ / 16];
#pragma unroll
      for (int ib = 0; ib < BQ / 16; ++ib) {
        frag qa[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) qa[s] = SQ::row_frag(Q, 16 * ib + c16, s, g);
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) {
          // a far tile: the p2c term of the lane's keys starts the products
          // (the c2p term is in the plane of rowinfo that the tile reads)
          f32x4 acc = far ? f32x4{fb[jb], fb[jb], fb[jb], fb[jb]} : zero4();
#pragma unroll
          for (int s = 0; s < NS; ++s)
            acc = M::mma(qa[s], kf[jb][s], acc);
          if constexpr (!far) {
            // rows 16*ib + 4*g + e of key column 32w + 16*jb + c16 (forward
            // tile order); without relative terms the buffer holds zeros
            const int jl = WK * w + 16 * jb;
            const int o = (jl / 64) * 2048 + ib * 1024 + ((jl % 64) / 16) * 256;
            if constexpr (sizeof(BT) == 2) {
              // one mixed-precision FMA per element adds the fp16 term
              typedef _Float16 h4 __attribute__((ext_vector_type(4)));
              const h4 v = __builtin_bit_cast(
                  h4, tr4_at(reinterpret_cast<const bf16*>(Bt) + o + (4 * g + (c16 >> 2)) * 16 + (c16 & 3) * 4));
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf((float)v[e], one, acc[e]);
            } else {
              float v[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = Bt[o + (4 * g + e) * 16 + c16];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[e] += v[e];
            }
          }
          sc[jb][ib] = acc;
        }
      }

      __builtin_amdgcn_s_setprio(0);
      // ---- P, dP, dS -----------------------------------------------------------------------------
      f32x4 pp[2][BQ / 16], dsh[2][BQ / 16];
      // this lane's 16 bits of a tile's words, bit 8 ib + 4 jb + e: word e,
      // shifted by 8 (w % 2) + c16 % 4, holds the pair (ib, jb) at bit 16 ib +
      // 4 jb: bits 0 and 4 stay, bits 16 and 20 move to 8 and 12, then the
      // word's four bits go to 8 ib + 4 jb + e
      auto lane_words = [&](const uint32_t* W) {
        return *reinterpret_cast<const uint4*>(W + w * 64 + 16 * (c16 >> 2) + 4 * g);
      };
      auto lane_bits = [&](const uint4& f4) {
        const uint32_t f[4] = {f4.x, f4.y, f4.z, f4.w};
        const int sh = 8 * (w & 1) + (c16 & 3);
        uint32_t m = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t t = f[e] >> sh;
          m |= ((t & 0x11u) | ((t >> 8) & 0x1100u)) << e;
        }
        return m;
      };
      uint32_t dm = 0, pm = 0;  // dropout's keep bits, the pair mask's
      if constexpr (DROP) dm = lane_bits(lane_words(Dw));
      if constexpr (BITS) pm = lane_bits(PLDS ? lane_words(Pw) : pcur);
      auto probs = [&](auto plain) {
        // segment masks: the lane's query segments, four consecutive rows
        // of each 16-row block in one 16-byte LDS read (read per element,
        // they cost segment-masked steps 4 to 13%)
        int4 qv[BQ / 16];
        if constexpr (MASK == MASK_SEG && !decltype(plain)::value) {
#pragma unroll
          for (int ib = 0; ib < BQ / 16; ++ib) qv[ib] = *reinterpret_cast<const int4*>(&qsg[n & 1][16 * ib + 4 * g]);
        }
#pragma unroll
        for (int ib = 0; ib < BQ / 16; ++ib) {
          frag dof[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) dof[s] = SQ::row_frag(dO, 16 * ib + c16, s, g);
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) {
            f32x4 dp = zero4();
#pragma unroll
            for (int s = 0; s < NS; ++s)
              dp = M::mma(dof[s], vf[jb][s], dp);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int il = 16 * ib + 4 * g + e;
              const float lr = R[2 * il];
              float pe;
              if constexpr (decltype(plain)::value) {
                pe = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[jb][ib][e], sl2, -lr));
              } else {
                // rows without probabilities (dead, padding) have lr = inf and may hold an
                // unwritten saved term: they are never exponentiated
                bool keep = jkeep[jb] && lr != INFINITY;
                if (MASK == MASK_SEG && !full)
                  keep = keep && (e == 0 ? qv[ib].x : e == 1 ? qv[ib].y : e == 2 ? qv[ib].z : qv[ib].w) == jseg[jb];
                if constexpr (BITS) keep = keep && (full || ((pm >> (8 * ib + 4 * jb + e)) & 1u));
                pe = keep ? __builtin_amdgcn_exp2f(__builtin_fmaf(sc[jb][ib][e], sl2, -lr)) : 0.f;
              }
              if constexpr (DROP) {
                const bool kept = (dm >> (8 * ib + 4 * jb + e)) & 1u;
                pp[jb][ib][e] = kept ? pe : 0.f;
                dsh[jb][ib][e] = pe * ((kept ? dp[e] * p.drop_scale : 0.f) - R[2 * il + 1]);
              } else {
                pp[jb][ib][e] = pe;
                dsh[jb][ib][e] = pe * (dp[e] - R[2 * il + 1]);
              }
            }
          }
        }
      };
      // without masking: unmasked tiles inside the sequence, and segment
      // tiles listed as full (every query and key of the tile active and in
      // one segment, so every pair is kept and every row has probabilities)
      if (!DROP && ((keys_in && i0 + BQ <= Lq) || ((MASK == MASK_SEG || BITS) && full)))
        probs(std::true_type{});
      else
        probs(std::false_type{});
      // dS^T of the tile into the wave's LDS tile (rows j), then dS rows to
      // the workspace, four consecutive keys per lane read transposed
#pragma unroll
      for (int jb = 0; jb < 2; ++jb)
#pragma unroll
        for (int ib = 0; ib < BQ / 16; ++ib) {
          vec4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (T)dsh[jb][ib][e];
          *reinterpret_cast<vec4*>(stg + (16 * jb + c16) * SROW + ZL + 16 * ib + 4 * g) = v;
        }
#pragma unroll
      for (int mi = 0; mi < BQ / 16; ++mi)
        store_ds(i0, mi, join_halves<T>(tr4(stg + ZL, SROW, 8 * g, 16 * mi, c16), tr4(stg + ZL, SROW, 8 * g + 4, 16 * mi, c16)));

      // ---- dV^T += dO^T P,  dK^T += Q^T dS (dO^T, Q^T read transposed) -----------------------
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < BQ / M::KSTEP; ++s) {
        frag pf[2], df[2];
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) {
          pf[jb] = M::from_acc(pp[jb], s);
          df[jb] = M::from_acc(dsh[jb], s);
          if constexpr (far) {
            frag ones;
#pragma unroll
            for (int e = 0; e < FE; ++e) ones[e] = (T)1.0f;
            fcs[jb] = M::mma(ones, df[jb], fcs[jb]);
          }
        }
#pragma unroll
        for (int db = 0; db < ND; ++db) {
          const frag dotf = SQ::col_acc(dO, s * M::KSTEP, 16 * db, g, c16);
          const frag qtf = SQ::col_acc(Q, s * M::KSTEP, 16 * db, g, c16);
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) {
            dva[db][jb] = M::mma(dotf, pf[jb], dva[db][jb]);
            dka[db][jb] = M::mma(qtf, df[jb], dka[db][jb]);
          }
        }
      }

      // ---- p2c: dK^T += qrgt[t0 + x]^T F[x] ------------------------------------------------
      if (!far && p2c) {
        // qrgt column of x = 0 for this wave: i0 - jw - 31 + OFF (a multiple of 32)
        const int t0 = tw0 + i0 + BKW - WK - WK * w;
#pragma unroll
        for (int s = 0; s < 2 * WK / M::KSTEP; ++s) {
          frag bfr[2];
#pragma unroll
          for (int jb = 0; jb < 2; ++jb) {
            // k = x = KSTEP*s + FE*g + e  ->  staged column (i - i0) = x + (j - jw) - 31
            const int jl = 16 * jb + c16;
            const T* row = stg + jl * SROW + ZL + M::KSTEP * s + FE * g + jl - 31;
            lds_read_elems<T, FE>(bfr[jb], row);
          }
          const int t = t0 + M::KSTEP * s + FE * g;  // this lane's first k column
          const T* blk = Ring + ((t >> 5) % NRB) * RBE + ((t & 31) / VEC) * D * VEC;
#pragma unroll
          for (int db = 0; db < ND; ++db) {
            const frag af = *reinterpret_cast<const frag*>(blk + (16 * db + c16) * VEC);
#pragma unroll
            for (int jb = 0; jb < 2; ++jb) dka[db][jb] = M::mma(af, bfr[jb], dka[db][jb]);
          }
        }
      }
      __builtin_amdgcn_s_setprio(0);
    };
    if constexpr (FAR) {
      float cs[2][2] = {{0.f, 0.f}, {0.f, 0.f}};  // column sums of dS per side
      int n = 0;
#pragma unroll
      for (int side = 1; side >= 0; --side) {
        const int hi = side ? n1 : n2;
        if (n >= hi) continue;
        const T* row = (const T*)p.qr + (int64_t)h * p.qrs[0] +
                       (p2c ? (int64_t)offset_row(p.rel, far_offset(p, side), Lq, Lk, p.A, true) * p.qrs[1] : 0);
        fcs[0] = fcs[1] = zero4();
        if (p2c) {
          f32x4 acc[2] = {zero4(), zero4()};
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const frag af = M::load_contig(row, s, g);  // every row of the A operand
#pragma unroll
            for (int jb = 0; jb < 2; ++jb) acc[jb] = M::mma(af, kf[jb][s], acc[jb]);
          }
          fb[0] = acc[0][0], fb[1] = acc[1][0];
        }
#pragma unroll 1
        for (; n < hi; ++n) {
          // the parity picks the buffers at run time (the copies are issued
          // from assembly, so the compiler waits for none of them)
          const bool o = (n ^ n2) & 1;
          tile(std::true_type{}, n, o ? Qs1 : Qs0, o ? dOs1 : dOs0, o ? Bs1 : Bs0, o ? Rs1 : Rs0, o ? Dk1 : Dk0, o ? Pk1 : Pk0,
               o ? Qs0 : Qs1, o ? dOs0 : dOs1, o ? Bs0 : Bs1, o ? Rs0 : Rs1, o ? Dk0 : Dk1, o ? Pk0 : Pk1);
        }
        if (p2c) {
          cs[side][0] = fcs[0][0], cs[side][1] = fcs[1][0];
#pragma unroll
          for (int db = 0; db < ND; ++db)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float r = (float)row[16 * db + 4 * g + e];
#pragma unroll
              for (int jb = 0; jb < 2; ++jb) dka[db][jb][e] = __builtin_fmaf(r, cs[side][jb], dka[db][jb][e]);
            }
        }
      }
      if (p2c && n2 > 0) {
        // and to the table gradient row: the waves' sums meet in their dS^T
        // tiles' space, which the near tiles then need zeroed again
        float* red = reinterpret_cast<float*>(stg);
        static_assert(SW * sizeof(T) >= 2 * D * sizeof(float), "both sides' sums in a wave's tile");
        wave_lds_sync();
#pragma unroll
        for (int side = 0; side < 2; ++side) far_row_sum<T, NS>(red + side * D, cs[side], kf, g, c16);
        __syncthreads();
        if (tid < 2 * D) {
          const int side = tid / D, d = tid % D;
          float v = 0.f;
#pragma unroll
          for (int u = 0; u < NW; ++u) v += reinterpret_cast<const float*>(Stg + u * SW)[side * D + d];
          far_part(bp.farpart, p, h, 1, side, D)[((int64_t)b * NKT + kt) * D + d] = v;
        }
        __syncthreads();
        for (int c = lane; c < 2 * D * (int)sizeof(float) / 16; c += 64)
          reinterpret_cast<f32x4*>(stg)[c] = zero4();
        wave_lds_sync();
      }
    }
    using near_t = std::false_type;
    for (int n = n2; n < nlist; n += 2) {
      tile(near_t{}, n, Qs0, dOs0, Bs0, Rs0, Dk0, Pk0, Qs1, dOs1, Bs1, Rs1, Dk1, Pk1);
      if (n + 1 < nlist) tile(near_t{}, n + 1, Qs1, dOs1, Bs1, Rs1, Dk1, Pk1, Qs0, dOs0, Bs0, Rs0, Dk0, Pk0);
    }
  }

  // ---- dK, dV ------------------------------------------------------------------------------
  T* dkbase = (T*)bp.dk + (int64_t)b * bp.dks[0] + (int64_t)h * bp.dks[2];
  T* dvbase = (T*)bp.dv + (int64_t)b * bp.dvs[0] + (int64_t)h * bp.dvs[2];
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
    const int j = jcol[jb];
    if (j < Lk) {
      T* krow = dkbase + (int64_t)j * bp.dks[1];
      T* vrow = dvbase + (int64_t)j * bp.dvs[1];
#pragma unroll
      for (int db = 0; db < ND; ++db) {
        typedef T vec4 __attribute__((ext_vector_type(4)));
        vec4 kv, vv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          kv[e] = (T)(dka[db][jb][e] * p.scale);
          vv[e] = (T)(DROP ? dva[db][jb][e] * p.drop_scale : dva[db][jb][e]);
        }
        *reinterpret_cast<vec4*>(krow + 16 * db + 4 * g) = kv;
        *reinterpret_cast<vec4*>(vrow + 16 * db + 4 * g) = vv;
      }
    }
  }
}

}  // namespace dsa
