// dsa_launch.h — host side of the attention kernels: launch parameters,
// workspace layouts and kernel selection (the C ABI over it: dsa_capi.hip).
//
// fwd_mask<T, D> and launch_bwd<T, D> hold every kernel of one element type
// and head dim.  Each pair is compiled in a translation unit of its own
// (dsa_inst.hip with DSA_T and DSA_D), so that the library builds in
// parallel; dsa_capi.hip only declares them.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../include/dsa.h"
#include "dsa_bwd.h"
#include "dsa_bwd_dkdv.h"
#include "dsa_bwd_dq.h"
#include "dsa_bwd_dqtab.h"
#include "dsa_bwd_table.h"
#include "dsa_dropout.h"
#include "dsa_fwd.h"
#include "dsa_order.h"

namespace dsa {
namespace host {

// description of the calling thread's last error (dsa_last_error)
inline thread_local std::string g_err;

static int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
static int fail(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return 1;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

static size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

static int round_up(int x, int a) { return (x + a - 1) / a * a; }

static int elem_bytes(int dtype) { return dtype == DSA_BF16 ? 2 : 4; }

// Whether the call's kernels look for far blocks (FarSpan): where at least
// `need` percent of its blocks lie past the saturation.  A far block saves its
// bands, but the FAR kernels' near tiles are the slower ones (in bf16 dkdv's
// scalar registers spill, and its query rows are read once more for the far
// planes), so that calls with few far blocks lose.  Training step at 12 heads,
// buckets 256 / max_position 512, 8192 tokens, plain -> FAR in us:
//   L (share)     1024 (19%)  1152 (25%)  1408 (35%)  1536 (39%)  2048 (52%)
//   no mask       489 -> 503  565 -> 555  616 -> 581  707 -> 643  930 -> 791
//   ... p2p       482 -> 503  542 -> 539  600 -> 579  674 -> 630  921 -> 766
//   ... and drop  537 -> 566  605 -> 615  662 -> 664  761 -> 722  1002 -> 868
//   padded rows   392 -> 395  311 -> 308  358 -> 339  467 -> 387  474 -> 410
//   causal, bits  389 -> 378  400 -> 394  430 -> 398  532 -> 473  689 -> 565
//   window, bits  204 -> 214  226 -> 237  224 -> 235  236 -> 246  260 -> 265
// Documents know no share: those of 2/3 of a row gain from half of the blocks
// on (434 -> 439 at 39%, 646 -> 591 at 52%, 632 -> 546 at L = 3072), those of
// 250 tokens hold no far pair and lose 2 to 4% at any length (288 -> 295, 265
// -> 270), more with dropout (dkdv's registers again: 331 -> 346 for 748 ->
// 653): they take long rows.  In float32 (4096 tokens) the registers fit: 6%
// 1013 -> 1022, 12% 1148 -> 1112, 30% 1605 -> 1467; documents 30% 1244 -> 1193
// and 606 -> 618.
static bool far_call(const dsa_fwd_args* a) {
  if (!a->flags) return false;
  const int nq = round_up(a->Lq, 128) / 128, nk = round_up(a->Lk, 128) / 128;
  const int64_t far = dsa::far_blocks(nq, nk, a->rel_saturated > 0 ? a->rel_saturated : 2 * a->att_span);
  const bool bf = a->dtype == DSA_BF16, drop = a->dropout_threshold != 0;
  const int need = a->seg ? (!bf ? 30 : drop ? 60 : 50) : !bf ? 10 : a->qc ? 34 : 25;
  return far > 0 && far * 100 >= (int64_t)nq * nk * need;
}

static dsa::FwdParams to_params(const dsa_fwd_args* a) {
  dsa::FwdParams p;
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.kr = a->kr;
  p.qr = a->qr;
  p.rel = a->rel_table;
  p.kk = a->key_keep;
  p.pk = a->pair_keep;
  p.out = a->out;
  p.lse = a->lse;
  p.bias = a->bias;
  for (int s = 0; s < 3; ++s) {
    p.qs[s] = a->q_strides[s];
    p.ks[s] = a->k_strides[s];
    p.vs[s] = a->v_strides[s];
    p.os[s] = a->o_strides[s];
  }
  for (int s = 0; s < 2; ++s) {
    p.krs[s] = a->kr_strides[s];
    p.qrs[s] = a->qr_strides[s];
  }
  p.krk = p.qrk = 64 / elem_bytes(a->dtype);  // rows contiguous: k-steps adjacent
  p.kkb = a->key_keep_stride_b;
  p.pkb = a->pair_keep_strides[0];
  p.pkq = a->pair_keep_strides[1];
  p.pkh = a->pair_keep ? a->pair_keep_stride_h : 0;
  p.seg = a->seg;
  p.segb = a->seg_stride_b;
  p.order = nullptr;
  p.qc = a->qc;
  for (int s = 0; s < 3; ++s) p.qcs[s] = a->qc ? a->qc_strides[s] : 0;
  p.B = a->B;
  p.H = a->H;
  p.Lq = a->Lq;
  p.Lk = a->Lk;
  p.A = a->flags ? a->att_span : 1;
  p.flags = a->flags;
  p.LqP = round_up(a->Lq, 128);
  p.LkP = round_up(a->Lk, 128);
  p.scale = a->scale;
  p.drop = nullptr;  // set where the keep bits are generated
  p.drop_scale = 1.f;
  p.olo = a->dtype == DSA_BF16 ? a->out_lo : nullptr;
  p.far = far_call(a);
  p.span = nullptr;  // set where the span is found before the kernel
  p.pbits = nullptr;  // set where the pair mask's bits are made
  p.pflag = nullptr;
  return p;
}

// ---- pair masks as bits (dsa_pair.h) ----
// Bytes of a pair mask's bits and of its tile flags (0 without one).
static size_t pair_words_bytes(const dsa_fwd_args* a) {
  if (!a->pair_keep) return 0;
  const int64_t m = dsa::pair_masks(a->B, a->H, a->pair_keep_strides[0], a->pair_keep_stride_h);
  return (size_t)m * (round_up(a->Lq, 128) / 32) * (round_up(a->Lk, 128) / 64) * 64 * sizeof(uint32_t);
}
static size_t pair_bytes(const dsa_fwd_args* a) {
  return align_up(pair_words_bytes(a), 256) + align_up(pair_words_bytes(a) / 256, 256);
}
// Bytes of them in the forward's workspace: none past the length of its tile
// lists in LDS (the kernels then read the mask's bytes; the backward's
// extents end below it).
constexpr int kMaxPairL = 32768;
static size_t fwd_pair_bytes(const dsa_fwd_args* a) { return a->Lk <= kMaxPairL ? pair_bytes(a) : 0; }
// Bytes of the far blocks' span in the forward's workspace.
static size_t fwd_span_bytes(const dsa_fwd_args* a) { return far_call(a) ? 256 : 0; }
// Points the kernels' parameters at the bits in buf and sets up their block.
static dsa::PairBits fill_pair(const dsa_fwd_args* a, void* buf, dsa::FwdParams& p) {
  dsa::PairBits t{};
  t.pk = a->pair_keep;
  t.pkb = p.pkb, t.pkq = p.pkq, t.pkh = p.pkh;
  t.bits = static_cast<uint32_t*>(buf);
  t.flags = static_cast<uint8_t*>(buf) + align_up(pair_words_bytes(a), 256);
  t.B = p.B, t.H = p.H, t.Lq = p.Lq, t.Lk = p.Lk, t.LqP = p.LqP, t.LkP = p.LkP;
  p.pbits = t.bits;
  p.pflag = t.flags;
  return t;
}
static int pair_blocks(const dsa::PairBits& t) { return (int)((dsa::pair_tiles(t) + 3) / 4); }

static int mask_mode(const dsa_fwd_args* a) {
  return a->pair_keep ? dsa::MASK_PAIR : a->key_keep ? dsa::MASK_KEY : a->seg ? dsa::MASK_SEG : dsa::MASK_NONE;
}

static int launch_check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail("dsa: %s launch failed: %s", what, hipGetErrorString(e));
  return 0;
}

// Heaviest-first order (dsa_order.h) of B * ntiles items: cost and order
// arrays of that many ints each.  Used under key_keep / seg masks only, and
// for at most this many items (one block sorts them).
constexpr int64_t kMaxOrderItems = 65536;

static size_t order_bytes(const dsa_fwd_args* a, int ntiles) {
  const int64_t n = (int64_t)a->B * ntiles;
  if (!(a->key_keep || a->seg) || n > kMaxOrderItems) return 0;
  return align_up((size_t)2 * n * sizeof(int), 256);
}

// Up to two heaviest-first orders (dsa_order.h): each job a buffer of cost
// then order (B * ntiles ints each), its tiles per row and its cost kind.
// fill_orders sets up the launches' parameters and the number of cost
// blocks (batch row fastest, then the tile group, then the job);
// launch_orders runs the cost and sort kernels, a caller that runs the cost
// blocks inside another launch only the sort (launch_order_sort).
static int fill_orders(const dsa::FwdParams& p, int njobs, int* const* bufs, const int* ntiles, const bool* fwd,
                dsa::OrderParams2& op, int& ny) {
  op.f = p;
  op.njobs = njobs;
  int maxt = 0;
  for (int j = 0; j < 2; ++j) {
    const int jj = j < njobs ? j : 0;
    op.job[j].cost = bufs[jj];
    op.job[j].order = bufs[jj] + (int64_t)p.B * ntiles[jj];
    op.job[j].ntiles = ntiles[jj];
    op.job[j].fwd = fwd[jj] ? 1 : 0;
    maxt = std::max(maxt, ntiles[jj]);
  }
  ny = (maxt + dsa::ORDER_TPB - 1) / dsa::ORDER_TPB;
  return p.B * ny * njobs;
}

static int launch_order_sort(const dsa::OrderParams2& op, hipStream_t st) {
  hipLaunchKernelGGL(dsa::dsa_order_sort_kernel, dim3(1), dim3(1024), 0, st, op);
  return launch_check("dsa_order_sort_kernel");
}

static int launch_orders(const dsa::FwdParams& p, int njobs, int* const* bufs, const int* ntiles, const bool* fwd,
                  hipStream_t st) {
  dsa::OrderParams2 op;
  int ny = 0;
  fill_orders(p, njobs, bufs, ntiles, fwd, op, ny);
  const dim3 grid((unsigned)p.B, (unsigned)ny, (unsigned)njobs);
  hipLaunchKernelGGL(dsa::dsa_order_cost_kernel, grid, dim3(256), 0, st, op);
  if (launch_check("dsa_order_cost_kernel")) return 1;
  return launch_order_sort(op, st);
}

static int fwd_tiles(const dsa_fwd_args* a) { return (a->Lq + dsa::dcfg::BQ - 1) / dsa::dcfg::BQ; }

// ---- attention dropout (dsa_dropout.h) ----
// Bytes of the keep bits (0 without dropout).
static size_t drop_bits_bytes(const dsa_fwd_args* a) {
  if (!a->dropout_threshold) return 0;
  return dsa::dropout_bits_bytes(a->B, a->H, round_up(a->Lq, 128), round_up(a->Lk, 128));
}
// Bytes of them in the forward's or the backward's workspace: none when the
// caller keeps them (dropout_bits).
static size_t drop_bytes(const dsa_fwd_args* a) {
  return a->dropout_bits ? 0 : align_up(drop_bits_bytes(a), 256);
}
static float drop_scale(const dsa_fwd_args* a) { return 65536.f / (float)(65536u - a->dropout_threshold); }

// Generates the call's keep bits into `bits` and points the kernels'
// parameters at them.
static int launch_dropout_bits(const dsa_fwd_args* a, uint32_t* bits, dsa::FwdParams& p, hipStream_t st) {
  dsa::DropParams d;
  d.bits = bits;
  d.B = a->B;
  d.H = a->H;
  d.NQB = round_up(a->Lq, 128) / 32;
  d.NKT = round_up(a->Lk, 128) / 64;
  d.t = a->dropout_threshold;
  d.k0 = (uint32_t)(a->dropout_seed & 0xffffffffu);
  d.k1 = (uint32_t)(a->dropout_seed >> 32);
  const dim3 grid((unsigned)((d.NKT + 3) / 4 * d.NQB), (unsigned)d.H, (unsigned)d.B);
  hipLaunchKernelGGL(dsa::dsa_dropout_bits_kernel, grid, dim3(256), 0, st, d);
  if (launch_check("dsa_dropout_bits_kernel")) return 1;
  p.drop = bits;
  p.drop_scale = drop_scale(a);
  return 0;
}


template <typename T, int D, int MASK, bool DROP, bool FAR>
int launch_fwd(const dsa::FwdParams& p, hipStream_t st) {
  dim3 grid((unsigned)((p.Lq + dsa::dcfg::BQ - 1) / dsa::dcfg::BQ * p.H * p.B));
  if (p.qc)
    hipLaunchKernelGGL((dsa::dsa_fwd_kernel<T, D, MASK, true, DROP, FAR>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((dsa::dsa_fwd_kernel<T, D, MASK, false, DROP, FAR>), grid, dim3(256), 0, st, p);
  return launch_check("dsa_fwd_kernel");
}

template <typename T, int D, int MASK>
int launch_fwd(const dsa::FwdParams& p, hipStream_t st) {
  if constexpr (MASK != dsa::MASK_PAIR) {
    if (p.far) return p.drop ? launch_fwd<T, D, MASK, true, true>(p, st) : launch_fwd<T, D, MASK, false, true>(p, st);
  }
  return p.drop ? launch_fwd<T, D, MASK, true, false>(p, st) : launch_fwd<T, D, MASK, false, false>(p, st);
}

template <typename T, int D>
int fwd_mask(const dsa::FwdParams& p, int mode, hipStream_t st) {
  switch (mode) {
    case dsa::MASK_KEY: return launch_fwd<T, D, dsa::MASK_KEY>(p, st);
    case dsa::MASK_PAIR:  // the bits wherever there is room for them (dsa_pair.h has both sides' times)
      if (p.pflag) return launch_fwd<T, D, dsa::MASK_BITS>(p, st);
      return launch_fwd<T, D, dsa::MASK_PAIR>(p, st);
    case dsa::MASK_SEG: return launch_fwd<T, D, dsa::MASK_SEG>(p, st);
    default: return launch_fwd<T, D, dsa::MASK_NONE>(p, st);
  }
}

// Compute units of the current device (queried once per device).
static int device_cus() {
  static std::atomic<int> cached[16] = {};
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  if (dev >= 0 && dev < 16 && (cus = cached[dev].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 256;
  if (dev >= 0 && dev < 16) cached[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// Workspace of the backward (offsets 256-byte aligned) and the padded
// extents the kernels share.
struct WsLayout {
  int LqP, LkP, TGP, OFF, NDB, NPG;
  size_t rowinfo, krgt, qrgt, ds, gpart, farpart, farspan, seg, cinfo, pair, korder, qorder, drop, total;
};

// fp32 elements of the far blocks' table gradient partials (far_part),
// rounded up to 256 bytes; 0 for calls without far blocks.
static size_t far_floats(const dsa_fwd_args& f) {
  const int LqP = round_up(f.Lq, 128), LkP = round_up(f.Lk, 128);
  if (!far_call(&f)) return 0;
  return align_up((size_t)f.H * 4 * f.B * (std::max(LqP, LkP) / 128) * f.D, 64);
}

static WsLayout ws_layout(const dsa_bwd_args* a) {
  const dsa_fwd_args& f = a->fwd;
  const size_t es = (size_t)elem_bytes(f.dtype);
  WsLayout w;
  w.LqP = round_up(f.Lq, 128);
  w.LkP = round_up(f.Lk, 128);
  w.OFF = w.LkP - 1;            // offset origin: t = d + OFF, 32-aligned tile starts
  w.TGP = w.LqP + w.LkP;        // offsets [-(LkP - 1), LqP] of every band window
  w.NDB = (w.LqP + w.LkP) / dsa::tbcfg::DBW;
  // Partial groups of the table kernel (ranges of an offset block's items
  // of one kind; a central block has about B * L / 32): about one and a
  // half workgroups per CU, whose fp32 atomics into the block accumulators
  // stay few and which leave room for dq beside them (B=32, L=512, the two
  // in one launch: backward 312 us with one workgroup per CU, 305 with one
  // and a half, 307 with two, 319 with three).  Long sequences and masks concentrate the work in the
  // central blocks, whose workgroups then bound the launch: those get at
  // most 64 items of a kind each.
  const int per = f.H * w.NDB;
  const int64_t items = (int64_t)f.B * ((w.LqP > w.LkP ? w.LqP : w.LkP) / 32);
  int64_t groups = (3 * device_cus() / 2 + per - 1) / per;
  if (w.NDB > 16 || f.key_keep || f.seg || f.pair_keep) groups = std::max<int64_t>(groups, (items + 63) / 64);
  w.NPG = (int)std::min<int64_t>(std::max<int64_t>(groups, 1), items);
  size_t off = 0;
  w.rowinfo = off;
  // one plane, with far blocks (FarSpan) one more per side
  const int planes = far_call(&f) ? 3 : 1;
  off = align_up(off + (size_t)f.B * f.H * w.LqP * 2 * planes * sizeof(float), 256);
  w.krgt = off;
  if (f.flags & DSA_C2P) off = align_up(off + (size_t)f.H * f.D * w.TGP * es, 256);
  w.qrgt = off;
  if (f.flags & DSA_P2C) off = align_up(off + (size_t)f.H * f.D * w.TGP * es, 256);
  w.ds = off;
  off = align_up(off + (size_t)f.B * f.H * w.LkP * w.LqP * es, 256);
  w.gpart = off;
  if (f.flags) off = align_up(off + (size_t)f.H * w.NDB * 2 * dsa::tbcfg::DBW * f.D * sizeof(float), 256);
  w.farpart = off;  // right after gpart: PREP zeroes both at once
  off += far_floats(f) * sizeof(float);
  w.farspan = off;
  if (planes > 1) off += 256;
  w.seg = off;
  if (f.flags) off = align_up(off + (size_t)2 * 2 * (2 * f.att_span) * sizeof(int), 256);
  w.cinfo = off;
  if (f.key_keep || f.seg) off = align_up(off + (size_t)f.B * (w.LqP / 32) * 4 * sizeof(int), 256);
  w.pair = off;
  off += pair_bytes(&f);
  w.korder = off;  // dkdv launch order (cost, order), under key_keep / seg
  off += order_bytes(&f, w.LkP / dsa::kvcfg::BKW);
  w.qorder = off;  // dq launch order
  off += order_bytes(&f, w.LqP / dsa::dqcfg::BQ);
  w.drop = off;  // attention dropout's keep bits, regenerated by PREP
  off += drop_bytes(&f);
  w.total = off;
  return w;
}

template <typename T, int D, bool DROP, bool FAR>
int launch_dkdv(const dsa::BwdParams& bp, const WsLayout& ws, int mode, hipStream_t st) {
  const dsa::FwdParams& f = bp.f;
  dim3 grid((unsigned)(ws.LkP / dsa::kvcfg::BKW * f.H * f.B));
  switch (mode) {
    case dsa::MASK_KEY:
      hipLaunchKernelGGL((dsa::dsa_bwd_dkdv_kernel<T, D, dsa::MASK_KEY, DROP, FAR>), grid, dim3(256), 0, st, bp);
      break;
    case dsa::MASK_PAIR:
      hipLaunchKernelGGL((dsa::dsa_bwd_dkdv_kernel<T, D, dsa::MASK_BITS, DROP, FAR>), grid, dim3(256), 0, st, bp);
      break;
    case dsa::MASK_SEG:
      hipLaunchKernelGGL((dsa::dsa_bwd_dkdv_kernel<T, D, dsa::MASK_SEG, DROP, FAR>), grid, dim3(256), 0, st, bp);
      break;
    default:
      hipLaunchKernelGGL((dsa::dsa_bwd_dkdv_kernel<T, D, dsa::MASK_NONE, DROP, FAR>), grid, dim3(256), 0, st, bp);
  }
  return launch_check("dsa_bwd_dkdv_kernel");
}

template <typename T, int D>
int launch_dkdv(const dsa::BwdParams& bp, const WsLayout& ws, int mode, hipStream_t st) {
  if (bp.f.far)
    return bp.f.drop ? launch_dkdv<T, D, true, true>(bp, ws, mode, st) : launch_dkdv<T, D, false, true>(bp, ws, mode, st);
  return bp.f.drop ? launch_dkdv<T, D, true, false>(bp, ws, mode, st) : launch_dkdv<T, D, false, false>(bp, ws, mode, st);
}

// The dq and table kernels: one launch for both, or either alone.
template <typename T, int D, bool FAR>
int launch_dq_fold(const dsa::BwdParams& bp, const dsa::BwdParams& tp, int ntab, int ndq, bool dq, bool fold,
                   hipStream_t st) {
  const bool listed = bp.cinfo != nullptr || bp.f.pflag != nullptr, qc = bp.f.qc != nullptr;
  if (fold && dq) {
    const int nt8 = (ntab + 7) / 8 * 8;
    const dim3 grid((unsigned)(nt8 + ndq));
    if (listed && qc)
      hipLaunchKernelGGL((dsa::dsa_bwd_dqtab_kernel<T, D, true, true, FAR>), grid, dim3(256), 0, st, bp, tp, ntab, nt8, ndq);
    else if (listed)
      hipLaunchKernelGGL((dsa::dsa_bwd_dqtab_kernel<T, D, true, false, FAR>), grid, dim3(256), 0, st, bp, tp, ntab, nt8, ndq);
    else if (qc)
      hipLaunchKernelGGL((dsa::dsa_bwd_dqtab_kernel<T, D, false, true, FAR>), grid, dim3(256), 0, st, bp, tp, ntab, nt8, ndq);
    else
      hipLaunchKernelGGL((dsa::dsa_bwd_dqtab_kernel<T, D, false, false, FAR>), grid, dim3(256), 0, st, bp, tp, ntab, nt8, ndq);
    return launch_check("dsa_bwd_dqtab_kernel");
  }
  if (fold) {
    if (listed)
      hipLaunchKernelGGL((dsa::dsa_bwd_table_kernel<T, D, true, FAR>), dim3(ntab), dim3(256), 0, st, tp);
    else
      hipLaunchKernelGGL((dsa::dsa_bwd_table_kernel<T, D, false, FAR>), dim3(ntab), dim3(256), 0, st, tp);
    return launch_check("dsa_bwd_table_kernel");
  }
  if (dq) {
    if (listed && qc)
      hipLaunchKernelGGL((dsa::dsa_bwd_dq_kernel<T, D, true, true, FAR>), dim3(ndq), dim3(256), 0, st, bp);
    else if (listed)
      hipLaunchKernelGGL((dsa::dsa_bwd_dq_kernel<T, D, true, false, FAR>), dim3(ndq), dim3(256), 0, st, bp);
    else if (qc)
      hipLaunchKernelGGL((dsa::dsa_bwd_dq_kernel<T, D, false, true, FAR>), dim3(ndq), dim3(256), 0, st, bp);
    else
      hipLaunchKernelGGL((dsa::dsa_bwd_dq_kernel<T, D, false, false, FAR>), dim3(ndq), dim3(256), 0, st, bp);
    return launch_check("dsa_bwd_dq_kernel");
  }
  return 0;
}

template <typename T, int D>
int launch_bwd(const dsa_bwd_args* a, const WsLayout& ws, int mode, hipStream_t st) {
  const dsa_fwd_args& f = a->fwd;
  dsa::BwdParams bp;
  bp.f = to_params(&f);
  bp.dout = a->dout;
  for (int s = 0; s < 3; ++s) {
    bp.dos[s] = a->do_strides[s];
    bp.dqs[s] = a->dq_strides[s];
    bp.dks[s] = a->dk_strides[s];
    bp.dvs[s] = a->dv_strides[s];
  }
  bp.dq = a->dq;
  bp.dk = a->dk;
  bp.dv = a->dv;
  bp.dqc = f.qc ? a->dqc : nullptr;
  for (int s = 0; s < 3; ++s) bp.dqcs[s] = f.qc ? a->dqc_strides[s] : 0;
  bp.dkr = a->dkr;
  bp.dqr = a->dqr;
  bp.dtab_bf16 = a->dtab_dtype == DSA_BF16;
  bp.dtab_overwrite = a->dtab_overwrite != 0;
  bp.dtab_rows = a->dtab_rows_first != 0;
  char* base = static_cast<char*>(a->workspace);
  bp.rowinfo = reinterpret_cast<float*>(base + ws.rowinfo);
  bp.krgt = base + ws.krgt;
  bp.qrgt = base + ws.qrgt;
  bp.ds = base + ws.ds;
  bp.gpart = reinterpret_cast<float*>(base + ws.gpart);
  bp.farpart = reinterpret_cast<float*>(base + ws.farpart);
  bp.farspan = reinterpret_cast<int*>(base + ws.farspan);
  bp.rowseg = reinterpret_cast<int*>(base + ws.seg);
  bp.cinfo = (f.key_keep || f.seg) ? reinterpret_cast<int4*>(base + ws.cinfo) : nullptr;
  dsa::PairBits pairs{};
  if (f.pair_keep) pairs = fill_pair(&f, base + ws.pair, bp.f);
  const int nkt = ws.LkP / dsa::kvcfg::BKW;
  int* kbuf = order_bytes(&f, nkt) ? reinterpret_cast<int*>(base + ws.korder) : nullptr;
  bp.korder = kbuf ? kbuf + (int64_t)f.B * nkt : nullptr;
  const int nqt = ws.LqP / dsa::dqcfg::BQ;
  int* qbuf = order_bytes(&f, nqt) ? reinterpret_cast<int*>(base + ws.qorder) : nullptr;
  bp.qorder = qbuf ? qbuf + (int64_t)f.B * nqt : nullptr;
  bp.TGP = ws.TGP;
  bp.OFF = ws.OFF;
  bp.NDB = ws.NDB;
  bp.NPG = ws.NPG;
  bp.fardq = 0;
  const int stages =
      a->stages ? a->stages : (DSA_STAGE_PREP | DSA_STAGE_DQ | DSA_STAGE_DKDV | DSA_STAGE_FOLD);
  if (f.dropout_threshold) {
    if (f.dropout_bits) {
      // the forward's keep bits, kept by the caller
      bp.f.drop = static_cast<const uint32_t*>(f.dropout_bits);
      bp.f.drop_scale = drop_scale(&f);
    } else {
      // PREP regenerates them (same seed, same bits) into the workspace; a
      // DKDV run in a later call reads the ones an earlier PREP left
      uint32_t* dbits = reinterpret_cast<uint32_t*>(base + ws.drop);
      if (stages & DSA_STAGE_PREP) {
        if (launch_dropout_bits(&f, dbits, bp.f, st)) return 1;
      } else {
        bp.f.drop = dbits;
        bp.f.drop_scale = drop_scale(&f);
      }
    }
  }

  if (stages & DSA_STAGE_PREP) {
    // dkdv's key tiles against 32-query chunks; dq's tiles (128 queries
    // against 64-key tiles) weigh as the forward's.  Their cost blocks run
    // first in the prep launch, the sort after it.
    int* bufs[2];
    int nts[2];
    bool kinds[2];
    int nj = 0;
    if (kbuf) bufs[nj] = kbuf, nts[nj] = nkt, kinds[nj++] = false;
    if (qbuf) bufs[nj] = qbuf, nts[nj] = nqt, kinds[nj++] = true;
    dsa::OrderParams2 op;
    op.f = bp.f;
    op.njobs = 0;
    dsa::PrepBlocks nb;
    nb.span = bp.f.far ? 1 : 0;
    nb.order = 0;
    nb.order_ny = 1;
    if (nj) nb.order = fill_orders(bp.f, nj, bufs, nts, kinds, op, nb.order_ny);
    const int64_t n = (int64_t)f.B * f.H * ws.LqP * (D / (16 / (int)sizeof(T)));
    nb.delta = (int)((n + 255) / 256);
    nb.gather = nb.seg = nb.chunk = nb.zero = 0;
    nb.pair = f.pair_keep ? pair_blocks(pairs) : 0;
    nb.gacc_floats = 0;
    if (f.key_keep || f.seg) nb.chunk = (int)(((int64_t)f.B * (ws.LqP / 32) + 255) / 256);
    if (f.flags) {
      const int64_t m = 2 * (int64_t)f.H * D * (ws.TGP / (16 / (int)sizeof(T)));
      nb.gather = (int)((m + 255) / 256);
      const int64_t ns = 2 * (int64_t)(f.Lq + f.Lk);
      nb.seg = (int)((ns + 255) / 256);
      // the table kernel's block accumulators, added to in FOLD
      nb.gacc_floats = (int64_t)f.H * ws.NDB * 2 * dsa::tbcfg::DBW * D + (int64_t)far_floats(f);
      nb.zero = (int)((nb.gacc_floats / 4 + 255) / 256);
    }
    hipLaunchKernelGGL((dsa::dsa_bwd_prep_kernel<T, D>),
                       dim3((unsigned)(nb.order + nb.span + nb.gather + nb.seg + nb.chunk + nb.zero + nb.pair + nb.delta)),
                       dim3(256), 0, st, bp, nb, op, pairs);
    if (launch_check("dsa_bwd_prep_kernel")) return 1;
    if (nj && launch_order_sort(op, st)) return 1;
  }
  if (stages & DSA_STAGE_DKDV) {
    if (launch_dkdv<T, D>(bp, ws, mode, st)) return 1;
  }
  // DQ and FOLD both only read dS: with both requested, the dq and table
  // workgroups run in one launch (dsa_bwd_dqtab.h) and share the GPU.
  // FOLD is TABLE (the table kernel) followed by SUM (the fold kernel).
  const bool fold = (stages & (DSA_STAGE_FOLD | DSA_STAGE_TABLE)) && f.flags;
  const bool sum = (stages & (DSA_STAGE_FOLD | DSA_STAGE_SUM)) && f.flags;
  const bool dq = (stages & DSA_STAGE_DQ) != 0;
  // In one launch the dq workgroups add the far blocks' dKr sums and the
  // table workgroups leave those blocks out; apart, the table kernel does
  // all of dKr, so that a caller may ask for either stage alone.
  bp.fardq = fold && dq;
  // dKr sums dS_ij times the c2p term's query rows: qc when it is given
  dsa::BwdParams tp = bp;
  if (f.qc) {
    tp.f.q = f.qc;
    for (int s = 0; s < 3; ++s) tp.f.qs[s] = f.qc_strides[s];
  }
  const int ntab = ws.NDB * f.H * ws.NPG;
  const int ndq = ws.LqP / dsa::dqcfg::BQ * f.H * f.B;
  if (bp.f.far) {
    if (launch_dq_fold<T, D, true>(bp, tp, ntab, ndq, dq, fold, st)) return 1;
  } else {
    if (launch_dq_fold<T, D, false>(bp, tp, ntab, ndq, dq, fold, st)) return 1;
  }
  if (sum) {
    const int rows = 2 * f.H * (2 * f.att_span);
    if (f.Lq + f.Lk > 2048)  // long rows of saturated relative positions: two waves a row
      hipLaunchKernelGGL((dsa::dsa_bwd_fold_kernel<D, 2>), dim3((unsigned)((rows + 1) / 2)), dim3(256), 0, st, bp);
    else  // one wave a row, four rows a workgroup
      hipLaunchKernelGGL((dsa::dsa_bwd_fold_kernel<D, 1>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, bp);
    if (launch_check("dsa_bwd_fold_kernel")) return 1;
  }
  return 0;
}

}  // namespace host
}  // namespace dsa
