// pl_kernels.hip — gfx950 kernels of the pileup path.
//
//   k_prep           per read (a wave for a long one), once per resident
//                    read set: alignment end, validity/adjMq, touched span,
//                    fragment, outliers
//   k_scan_*         exclusive scans (keep-read prefix, radix histograms)
//   k_begin          the batch's counters; per region: readCount
//                    (BamFile.process), P ops, errors
//   k_plan           per window: the sorted read range it must scan
//   k_heads          the windows in cost order, for the work queue
//   k_window         the hot kernel: one workgroup owns a window of W
//                    positions, accumulates every counter in LDS, scans
//                    physCov, and writes counters + BaseCall once
//   k_spill_place    evidence records beyond a window's LDS buffer, put with
//                    the window's others
//   k_indel_pass     BaseCall of columns whose indel strings matter
//   k_cand_*         the change candidates in position order
//   k_finalize       Pass 1 per region: minDepth, deletion pass
//   k_after          columns changed by the deletion pass called again;
//                    exact confirmed counts of very deep regions
//   k_final_flags    final dispositions for export
//   k_rs_*           LSD radix sort (the assembler's K-mers)
//
// Reference: broadinstitute/pilon v1.24, src/main/scala/org/broadinstitute/pilon/
#include <hip/hip_runtime.h>
#include "pl_core.h"
#include "pl_kernels.h"

namespace {

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane ? ((~0ull) >> (64 - lane)) : 0ull;
}

template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    T o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

// slot of this lane in a list grown by the lanes of the wave whose pred is
// set: one atomic on the list counter per wave
__device__ __forceinline__ uint32_t wave_append(uint32_t* ctr, bool pred) {
  const uint64_t m = __ballot(pred);
  if (!m) return 0u;
  const int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0u;
  if ((int)(threadIdx.x & 63) == leader) base = atomicAdd(ctr, (uint32_t)__popcll(m));
  base = __shfl(base, leader, 64);
  return base + (uint32_t)__popcll(m & lanemask_lt());
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Wave-wide integer scans through DPP lane moves (no LDS round trips): a
// Hillis-Steele scan inside each row of 16 lanes (row_shr 1, 2, 4, 8, lanes
// shifted in from outside the row read 0), then the last lane of row 0 added
// into row 1 and of row 2 into row 3 (row_bcast:15), and the last lane of
// row 1 into rows 2 and 3 (row_bcast:31).  Integer adds only, so the result
// equals the shuffle scan's; all 64 lanes must be active.
template <int CTRL, int ROW = 0xf>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW, 0xf, true);
}
template <class T>
__device__ __forceinline__ T wave_scan_dpp(T v) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32- or 64-bit integers");
  if constexpr (sizeof(T) == 4) {
    uint32_t x = (uint32_t)v;
    x += dpp_move<0x111>(x);
    x += dpp_move<0x112>(x);
    x += dpp_move<0x114>(x);
    x += dpp_move<0x118>(x);
    x += dpp_move<0x142, 0xa>(x);
    x += dpp_move<0x143, 0xc>(x);
    return (T)x;
  } else {
    uint64_t x = (uint64_t)v;
    auto mv = [](auto ctrl, auto row, uint64_t y) {
      return (uint64_t)dpp_move<decltype(ctrl)::value, decltype(row)::value>((uint32_t)y) |
             ((uint64_t)dpp_move<decltype(ctrl)::value, decltype(row)::value>((uint32_t)(y >> 32)) << 32);
    };
    using std::integral_constant;
    x += mv(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{}, x);
    x += mv(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{}, x);
    x += mv(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{}, x);
    x += mv(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{}, x);
    x += mv(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{}, x);
    x += mv(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{}, x);
    return (T)x;
  }
}
// lane 63's value in every lane (wave-uniform)
template <class T>
__device__ __forceinline__ T lane63(T v) {
  if constexpr (sizeof(T) == 4) return (T)__builtin_amdgcn_readlane((int)v, 63);
  else
    return (T)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), 63) << 32) |
               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, 63));
}
template <class T>
__device__ __forceinline__ T wave_total_dpp(T v) { return lane63(wave_scan_dpp(v)); }

}  // namespace

// ------------------------------------------------------------------ k_prep
// the read set's scalars (scal[0], [1], [2], [6]: maxima, -1 = none;
// flags: scal[4], scal[5], scal[7]) gathered over a thread's reads, then over its
// wave, so one wave gives one atomic per scalar
struct PrepAcc {
  int32_t back = -1, lead = -1, span = -1, fp = -1;
  uint32_t flags = 0;
};
__device__ __forceinline__ void prep_flush(PrepAcc a, int32_t* scal) {
  for (int d = 32; d >= 1; d >>= 1) {
    a.back = max(a.back, __shfl_xor(a.back, d, 64));
    a.lead = max(a.lead, __shfl_xor(a.lead, d, 64));
    a.span = max(a.span, __shfl_xor(a.span, d, 64));
    a.fp = max(a.fp, __shfl_xor(a.fp, d, 64));
    a.flags |= (uint32_t)__shfl_xor((int)a.flags, d, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (a.back >= 0) atomicMax(&scal[0], a.back);
    if (a.lead >= 0) atomicMax(&scal[1], a.lead);
    if (a.span >= 0) atomicMax(&scal[2], a.span);
    if (a.fp >= 0) atomicMax(&scal[6], a.fp);
    if (a.flags & 1u) atomicOr(&scal[4], 1);
    if (a.flags & 2u) atomicOr(&scal[5], 1);
    if (a.flags & 4u) atomicOr(&scal[7], 1);
  }
}

// the facts of read r of set R, whose segments take `slots` table entries
__device__ __forceinline__ void prep_put(const RSDev& R, int64_t r, const PrepOut& o, uint32_t slots,
                                         uint32_t* keepflag, uint32_t* segcount, int32_t* scal, int64_t* outliers,
                                         int64_t out_cap, PrepAcc& acc) {
  RMeta m = o.m;
  segcount[r] = slots;
  const bool keep = (m.info & RI_KEEP) != 0;
  if (keep) {
    int64_t lo = INT64_MAX, hi = INT64_MIN;
    if (m.fp_lo <= m.fp_hi) { lo = m.fp_lo; hi = m.fp_hi; }
    if (m.fr_lo < m.fr_hi) {
      lo = lo < m.fr_lo ? lo : m.fr_lo;
      hi = hi > (int64_t)m.fr_hi - 1 ? hi : (int64_t)m.fr_hi - 1;
    }
    if (lo <= hi) {
      const int64_t lead = m.pos - lo, back = hi - m.pos;
      if (lead > PL_MAX_LEAD || back > (R.all_long ? PL_MAX_BACK_LONG : PL_MAX_BACK) || R.seq_off[r + 1] - R.seq_off[r] >= PL_MAX_SEQ) {
        m.info |= RI_OUTLIER;
        int k = atomicAdd(&scal[3], 1);
        if (k < out_cap) outliers[k] = r;
      } else {
        acc.back = max(acc.back, (int32_t)(back > 0 ? back : 0));
        acc.lead = max(acc.lead, (int32_t)(lead > 0 ? lead : 0));
        if (m.fp_lo <= m.fp_hi && m.fp_hi > m.pos) acc.fp = max(acc.fp, m.fp_hi - m.pos);
      }
    }
    const int32_t spanEnd = m.aend != 0 ? m.aend : m.pos;
    acc.span = max(acc.span, spanEnd - m.pos > 0 ? spanEnd - m.pos : 0);
    if (m.info & RI_UNK_MASK) acc.flags |= 1u;
    if (m.info & (RI_BAD | RI_EDGE_CLIP)) acc.flags |= 2u;
    if (o.clips) acc.flags |= 4u;
  }
  R.meta[r] = m;
  R.ftail[r] = frag_tail(m);
  keepflag[r] = keep ? 1u : 0u;
}

// A read without QUAL piles defaultQual at every base (PileUpRegion.scala:114-115):
// written into its quality bytes once, so the window kernel reads quals unconditionally.
__device__ __forceinline__ void fill_quals(const RSDev& R, int64_t r, const KConf& cf, int first, int step) {
  int8_t* qd = (int8_t*)R.quals + R.seq_off[r];
  const int64_t L = R.seq_off[r + 1] - R.seq_off[r];
  for (int64_t k = first; k < L; k += step) qd[k] = (int8_t)cf.default_qual;
}

// k_prep's work on read r of set R (long reads are prep_long's)
__device__ __forceinline__ void prep_one(const RSDev& R, int64_t r, const KConf& cf, uint32_t* keepflag,
                                         uint32_t* segcount, int32_t* scal, int64_t* outliers, int64_t out_cap,
                                         PrepAcc& acc) {
  const PrepOut o = prep_read(R, r, cf);
  if (o.m.info & RI_NOQUAL) fill_quals(R, r, cf, 0, 1);
  const uint32_t slots = wants_segs(o.m.info) ? (uint32_t)build_segs(R, r, o.m.info, cf, nullptr) : 0u;
  prep_put(R, r, o, slots, keepflag, segcount, scal, outliers, out_cap, acc);
}

// Calls f(w, locus, readOffset, k) for the ops of read r, 64 of them side by
// side (w = 0, an empty M, in lanes past the last).
template <class F>
__device__ __forceinline__ void wave_ops(const RSDev& R, int64_t r, F&& f) {
  const int lane = threadIdx.x & 63;
  const int64_t c0 = R.cigar_off[r], c1 = R.cigar_off[r + 1];
  int32_t ro = 0, locus = R.pos[r];
  for (int64_t k0 = c0; k0 < c1; k0 += 64) {
    const uint32_t w = k0 + lane < c1 ? R.cigar[k0 + lane] : 0u;
    const int op = (int)(w & 15);
    const int32_t rd = consumes_read(op) ? (int32_t)(w >> 4) : 0, rf = consumes_ref(op) ? (int32_t)(w >> 4) : 0;
    const int32_t ir = wave_scan_dpp(rd), il = wave_scan_dpp(rf);
    f(w, locus + il - rf, ro + ir - rd, (int32_t)(k0 - c0) + lane);
    ro += lane63(ir);
    locus += lane63(il);
  }
}

// prep_one for a long read, by a wave, an op a lane: its hundreds of ops, one
// after the other in a thread, are as many slides along the reference, each a
// chain of loads.  2,668 reads of 6,001 bases: k_prep 2.2 ms and k_segfill
// 2.9 with a thread a read, 117 and 116 us so.
__device__ __forceinline__ void prep_long(const RSDev& R, int64_t r, const KConf& cf, uint32_t* keepflag,
                                          uint32_t* segcount, int32_t* scal, int64_t* outliers, int64_t out_cap,
                                          PrepAcc& acc) {
  const int lane = threadIdx.x & 63;
  const ReadHead h = read_head(R, r);
  const int32_t L = h.L;
  ReadSums sums;
  for (int64_t k = h.c0 + lane; k < h.c1; k += 64) add_op(sums, R.cigar[k]);
  sums.refLen = wave_sum(sums.refLen);
  sums.readLen = wave_sum(sums.readLen);
  sums.clipped = (int32_t)wave_sum((uint32_t)sums.clipped);          // (Int sums wrap)
  sums.nP = wave_sum(sums.nP);
  sums.nS = wave_sum(sums.nS);
  sums.bad = __ballot(sums.bad) != 0;
  const uint32_t op0 = h.c1 > h.c0 ? R.cigar[h.c0] : 0u;
  int32_t aend;
  const uint32_t info = read_info(R, r, h, sums, op0, cf, &aend);
  OpSpan span;
  LongOps lo;
  int64_t n = 0;
  if (!(info & RI_BAD)) {
    const ReadAcc a = read_acc(R, r, info, cf.default_qual);
    const bool segs = wants_segs(info);
    wave_ops(R, r, [&](uint32_t w, int32_t locus, int32_t readOffset, int32_t k) {
      span = op_span(R, a, info, cf, w, locus, readOffset, L, span);
      if (!segs) return;
      lo = add_long_op(lo, w, k, readOffset);
      n += op_segs(R, a, info, cf, w, locus, readOffset, L, nullptr);
    });
    for (int d = 32; d >= 1; d >>= 1) {
      span.lo = min(span.lo, __shfl_xor(span.lo, d, 64));
      span.hi = max(span.hi, __shfl_xor(span.hi, d, 64));
      lo.clip = min(lo.clip, __shfl_xor(lo.clip, d, 64));
      lo.last = max(lo.last, __shfl_xor(lo.last, d, 64));
    }
    span.events = wave_sum(span.events);
    lo.lead = __ballot(lo.lead) != 0;
    n = wave_sum(n);
  }
  if (info & RI_NOQUAL) fill_quals(R, r, cf, lane, 64);
  if (lane == 0)
    prep_put(R, r, prep_result(h, op0, info, aend, sums, span), wants_segs(info) ? long_seg_slots(lo, L, n, h.c1 - h.c0) : 0u,
             keepflag, segcount, scal, outliers, out_cap, acc);
}

__global__ void k_prep(RSDev R, KConf cf, uint32_t* keepflag, uint32_t* segcount, int32_t* scal, int64_t* outliers,
                       int64_t out_cap) {
  const int64_t n = R.n;
  PrepAcc acc;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
    if (!R.lrt || !R.lrt[r]) prep_one(R, r, cf, keepflag, segcount, scal, outliers, out_cap, acc);
  prep_flush(acc, scal);
}
// ... and its long reads, a wave each
__global__ void __launch_bounds__(256) k_prep_long(RSDev R, KConf cf, uint32_t* keepflag, uint32_t* segcount,
                                                   int32_t* scal, int64_t* outliers, int64_t out_cap) {
  PrepAcc acc;
  for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < R.n; r += (int64_t)gridDim.x * 4)
    if (R.lrt[r]) prep_long(R, r, cf, keepflag, segcount, scal, outliers, out_cap, acc);
  prep_flush(acc, scal);
}

// the set of block b when set s has blocks [blk[s], blk[s + 1])
__device__ __forceinline__ int32_t set_of_block(const int64_t* blk, int32_t n_sets, int64_t b) {
  int32_t lo = 0, hi = n_sets;
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) / 2;
    if (blk[mid] <= b) lo = mid; else hi = mid;
  }
  return lo;
}

// k_prep over many sets in one launch: set s's reads on blocks [blk[s],
// blk[s + 1]), a wave a read in the sets of long reads (a set has only those
// or none), its flags at keep + at[s], its outlier list outl[s] of ocap[s]
// entries
__global__ void k_prep_sets(const RSDev* sets, const int64_t* blk, int32_t n_sets, KConf cf, uint32_t* keep,
                            uint32_t* segc, const int64_t* at, int64_t* const* outl, const int64_t* ocap) {
  const int32_t s = set_of_block(blk, n_sets, blockIdx.x);
  const RSDev& R = sets[s];
  if (R.lrt) return;
  const int64_t nb = blk[s + 1] - blk[s];
  PrepAcc acc;
  for (int64_t r = (blockIdx.x - blk[s]) * blockDim.x + threadIdx.x; r < R.n; r += nb * blockDim.x)
    prep_one(R, r, cf, keep + at[s], segc + at[s], R.scal, outl[s], ocap[s], acc);
  prep_flush(acc, R.scal);   // every wave of a block is in set s
}
__global__ void __launch_bounds__(256) k_prep_long_sets(const RSDev* sets, const int64_t* blk, int32_t n_sets, KConf cf,
                                                        uint32_t* keep, uint32_t* segc, const int64_t* at,
                                                        int64_t* const* outl, const int64_t* ocap) {
  const int32_t s = set_of_block(blk, n_sets, blockIdx.x);
  const RSDev& R = sets[s];
  if (!R.lrt) return;
  const int64_t nb = blk[s + 1] - blk[s];
  PrepAcc acc;
  for (int64_t r = (blockIdx.x - blk[s]) * 4 + (threadIdx.x >> 6); r < R.n; r += nb * 4)
    prep_long(R, r, cf, keep + at[s], segc + at[s], R.scal, outl[s], ocap[s], acc);
  prep_flush(acc, R.scal);
}

// fills the segment table; RMeta.op0 of a multi-op read becomes its first
// entry and the info word carries the count (RI_SEG_MAX = too many: walked)
__device__ __forceinline__ void segfill_one(const RSDev& R, int64_t r, const KConf& cf, const uint32_t* segoff,
                                            Seg* segs) {
  RMeta m = R.meta[r];
  if (!wants_segs(m.info)) return;
  const uint32_t o = segoff[r], c = segoff[r + 1] - o;
  m.info = seg_fill(R, r, m.info, cf, segs, o, c);
  m.op0 = o;
  R.meta[r] = m;
}
// ... for a long read by a wave, an op a lane
__device__ __forceinline__ void segfill_long(const RSDev& R, int64_t r, const KConf& cf, const uint32_t* segoff,
                                             Seg* segs) {
  const int lane = threadIdx.x & 63;
  RMeta m = R.meta[r];
  if (!wants_segs(m.info)) return;
  const uint32_t o = segoff[r], c = segoff[r + 1] - o;
  int32_t reach = 0;
  if (c) {
    const int32_t L = (int32_t)(R.seq_off[r + 1] - R.seq_off[r]);
    const ReadAcc a = read_acc(R, r, m.info, cf.default_qual);
    uint32_t at = o + 1;
    wave_ops(R, r, [&](uint32_t w, int32_t locus, int32_t readOffset, int32_t) {
      const int n = op_segs(R, a, m.info, cf, w, locus, readOffset, L, nullptr);
      const int inc = wave_scan_dpp(n);
      Seg* out = segs + at + (inc - n);
      if (n) op_segs(R, a, m.info, cf, w, locus, readOffset, L, out);
      for (int i = 0; i < n; i++) reach = max(reach, seg_reach(out[i]));
      at += (uint32_t)lane63(inc);
    });
    for (int d = 32; d >= 1; d >>= 1) reach = max(reach, __shfl_xor(reach, d, 64));
  }
  if (lane != 0) return;
  if (c) put_seg_header(segs[o], m.pos, c, reach);
  m.info = seg_info(m.info, c);
  m.op0 = o;
  R.meta[r] = m;
}

__global__ void k_segfill(RSDev R, KConf cf, const uint32_t* segoff, Seg* segs) {
  const int64_t n = R.n;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
    if (!R.lrt || !R.lrt[r]) segfill_one(R, r, cf, segoff, segs);
}
__global__ void __launch_bounds__(256) k_segfill_long(RSDev R, KConf cf, const uint32_t* segoff, Seg* segs) {
  for (int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < R.n; r += (int64_t)gridDim.x * 4)
    if (R.lrt[r]) segfill_long(R, r, cf, segoff, segs);
}

// k_segfill over many sets in one launch: set s's segment offsets at
// segoff + at[s], its table segs[s]
__global__ void k_segfill_sets(const RSDev* sets, const int64_t* blk, int32_t n_sets, KConf cf, const uint32_t* segoff,
                               const int64_t* at, Seg* const* segs) {
  const int32_t s = set_of_block(blk, n_sets, blockIdx.x);
  const RSDev& R = sets[s];
  if (R.lrt) return;
  const int64_t nb = blk[s + 1] - blk[s];
  for (int64_t r = (blockIdx.x - blk[s]) * blockDim.x + threadIdx.x; r < R.n; r += nb * blockDim.x)
    segfill_one(R, r, cf, segoff + at[s], segs[s]);
}
__global__ void __launch_bounds__(256) k_segfill_long_sets(const RSDev* sets, const int64_t* blk, int32_t n_sets, KConf cf,
                                                           const uint32_t* segoff, const int64_t* at, Seg* const* segs) {
  const int32_t s = set_of_block(blk, n_sets, blockIdx.x);
  const RSDev& R = sets[s];
  if (!R.lrt) return;
  const int64_t nb = blk[s + 1] - blk[s];
  for (int64_t r = (blockIdx.x - blk[s]) * 4 + (threadIdx.x >> 6); r < R.n; r += nb * 4)
    segfill_long(R, r, cf, segoff + at[s], segs[s]);
}

// ------------------------------------------------------------------ scans
// Exclusive scan of n uint32 in tiles of SCAN_TILE; out has n+1 entries.
__global__ void __launch_bounds__(256) k_scan_tiles(const uint32_t* in, int64_t n, uint32_t* tile_sums) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
  uint32_t s = 0;
  for (int i = threadIdx.x; i < SCAN_TILE; i += 256) {
    const int64_t k = base + i;
    if (k < n) s += in[k];
  }
  s = wave_sum(s);
  __shared__ uint32_t ws[4];
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ void __launch_bounds__(1024) k_scan_top(uint32_t* tile_sums, int64_t nt) {
  __shared__ uint32_t ws[16];
  __shared__ uint32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t b0 = 0; b0 < nt; b0 += 1024) {
    const int64_t k = b0 + threadIdx.x;
    uint32_t v = k < nt ? tile_sums[k] : 0;
    uint32_t inc = wave_incl_scan(v);
    if ((threadIdx.x & 63) == 63) ws[threadIdx.x >> 6] = inc;
    __syncthreads();
    uint32_t add = carry;
    for (int w = 0; w < (int)(threadIdx.x >> 6); w++) add += ws[w];
    if (k < nt) tile_sums[k] = add + inc - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = add + inc;
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) k_scan_apply(const uint32_t* in, int64_t n, const uint32_t* tile_sums, uint32_t* out) {
  // each thread owns SCAN_TILE/256 consecutive items
  constexpr int PER = SCAN_TILE / 256;
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * PER;
  uint32_t v[PER];
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < PER; i++) {
    v[i] = (base + i < n) ? in[base + i] : 0u;
    s += v[i];
  }
  uint32_t inc = wave_incl_scan(s);
  __shared__ uint32_t ws[4];
  if ((threadIdx.x & 63) == 63) ws[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t acc = tile_sums[blockIdx.x] + inc - s;
  for (int w = 0; w < (int)(threadIdx.x >> 6); w++) acc += ws[w];
#pragma unroll
  for (int i = 0; i < PER; i++) {
    if (base + i < n) out[base + i] = acc;
    if (base + i == n - 1) out[n] = acc + v[i];
    acc += v[i];
  }
  if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
}

// ------------------------------------------------------------------ plan
namespace {

// first index in pos[lo, hi) whose position is >= x, by an aligned group of
// GL lanes (all 64 lanes of the wave active): GL probes a round cut the
// range GL+1-fold, so 16 lanes take 5 dependent loads for a million reads
// where one lane takes 20.
template <int GL>
__device__ __forceinline__ int64_t group_lower_pos(const int32_t* pos, int64_t lo, int64_t hi, int64_t x) {
  const int lane = threadIdx.x & 63, gl = lane & (GL - 1), g0 = lane & ~(GL - 1);
  const uint64_t gm = GL == 64 ? ~0ull : (1ull << (GL & 63)) - 1ull;
  while (__ballot(hi - lo > GL)) {
    const int64_t m = hi - lo;
    const bool more = m > GL;
    const bool less = more && (int64_t)pos[lo + (gl + 1) * m / (GL + 1)] < x;
    const int k = __popcll((__ballot(less) >> g0) & gm);      // probes ascend: a prefix of the group
    if (more) {
      const int64_t a = lo;
      if (k > 0) lo = a + k * m / (GL + 1) + 1;
      if (k < GL) hi = a + (k + 1) * m / (GL + 1);
    }
  }
  const bool less = lo + gl < hi && (int64_t)pos[lo + gl] < x;
  return lo + __popcll((__ballot(less) >> g0) & gm);
}

// the same for an answer expected near lo: one round of probes 16, 32, 64, ...
// beyond it bounds the search (a window's reads end a few hundred on, and a
// search of the whole set takes six rounds of scattered loads)
template <int GL>
__device__ __forceinline__ int64_t group_lower_pos_near(const int32_t* pos, int64_t lo, int64_t n, int64_t x) {
  const int lane = threadIdx.x & 63, gl = lane & (GL - 1), g0 = lane & ~(GL - 1);
  const uint64_t gm = GL == 64 ? ~0ull : (1ull << (GL & 63)) - 1ull;
  const int64_t at = lo + (16ll << gl);
  const bool less = at < n && (int64_t)pos[at] < x;
  const int k = __popcll((__ballot(less) >> g0) & gm);
  int64_t hi = n;
  if (k < GL && lo + (16ll << k) < n) hi = lo + (16ll << k);
  if (k > 0) lo += (16ll << (k - 1)) + 1;
  return group_lower_pos<GL>(pos, lo, hi, x);
}

__device__ __forceinline__ void put_head(WinHead* heads, int32_t slot, int32_t wi, const WinDev& w, const JobDev& J,
                                         int32_t m0) {
  WinHead h;
  h.wi = wi; h.job = w.job; h.p0 = w.p0; h.p1 = w.p1;
  h.lo = w.lo; h.hi = w.hi; h.plo = w.plo; h.out = J.out;
  h.rs = J.rs; h.start = J.start; h.stop = J.stop; h.qs = J.qs; h.qe = J.qe;
  h.m0 = m0;
  h.pad[0] = h.pad[1] = 0;
  heads[slot] = h;
}

// The read ranges of the windows of a block, one per group of 16 lanes;
// returns this lane's window's cost bin (-1: past the last window).
// Windows are few and short, so the three searches are all latency: a lane
// per window took 27 us for 47,000 windows and 14 us for 400.
__device__ int plan_windows(const EngineArgs& A, int32_t blk, WinDev* wins, bool heads) {
  const int32_t w0 = blk * (int32_t)(blockDim.x >> 4) + (int32_t)(threadIdx.x >> 4);
  const bool in = w0 < A.n_wins;
  const int32_t w = in ? w0 : A.n_wins - 1;                 // idle groups repeat the last window
  WinDev win = wins[w];
  const JobDev& J = A.jobs[win.job];
  const RSDev& R = A.rs[J.rs];
  const int64_t L0 = (int64_t)J.start + win.p0, L1 = (int64_t)J.start + win.p1;
  const int32_t back = R.scal[0], lead = R.scal[1], fp = R.scal[6];
  win.lo = group_lower_pos<16>(R.pos, 0, R.n, L0 - back);
  win.hi = group_lower_pos_near<16>(R.pos, win.lo, R.n, L1 + lead);
  // the end of the fragment-only reads: fragment_only_end with the group's search
  const bool all = fragment_all(J, (int32_t)L0, back, fp);
  const int64_t plo = group_lower_pos<16>(R.pos, win.lo, win.hi, L0 - fp);
  win.plo = all ? win.lo : plo;
  // adjMq + 1 of most of 16 reads spread over the window's (1 when none is valid)
  uint32_t mq1 = 0;
  {
    const int gl = threadIdx.x & 15, nr = (int)(win.hi - win.plo < 16 ? win.hi - win.plo : 16);
    if (gl < nr) {
      const uint32_t info = R.meta[win.plo + (win.hi - win.plo) * gl / nr].info;
      if (info & RI_VALID) mq1 = (info & RI_ADJMQ_MASK) + 1u;
    }
    uint32_t same = 0;
#pragma unroll
    for (int d = 0; d < 16; d++) same += (uint32_t)__shfl_xor((int)mq1, d, 64) == mq1;
    uint32_t best = mq1 ? same << 16 | mq1 : 1u;
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) best = max(best, (uint32_t)__shfl_xor((int)best, d, 64));
    win.m0 = (int32_t)(best & 0xffffu);
  }
  const int bin = (int)cost_bin((win.hi - win.plo) + (win.plo - win.lo) / 8 + (int64_t)(win.p1 - win.p0) / 16);
  if (in && (threadIdx.x & 15) == 0) {
    wins[w] = win;
    A.cost[w] = (uint8_t)bin;
    if (heads) put_head((WinHead*)A.heads, w, w, win, J, win.m0);
  }
  if (in)
    for (int q = threadIdx.x & 15; q < A.W >> 6; q += 16) A.dmask[(int64_t)w * (A.W >> 6) + q] = 0;   // for the indel pass
  return in ? bin : -1;
}

// readCount of BamFile.process (BamFile.scala:118-139): kept reads whose span
// overlaps [qs, qe], from the keep-prefix plus the reads straddling qs.  One
// wave per region, which also clears the region's counters.
__device__ void job_begin(const EngineArgs& A, const uint32_t* const* keep_prefix, int32_t j) {
  const JobDev& J = A.jobs[j];
  const RSDev& R = A.rs[J.rs];
  const uint32_t* kp = keep_prefix[J.rs];
  const int lane = threadIdx.x & 63;
  for (int d = lane; d < PL_HIST; d += 64) A.hist[(int64_t)j * PL_HIST + d] = 0;
  const int64_t a = group_lower_pos<64>(R.pos, 0, R.n, J.qs);
  const int64_t b = group_lower_pos<64>(R.pos, a, R.n, (int64_t)J.qe + 1);
  const int64_t a1 = group_lower_pos<64>(R.pos, a, b, (int64_t)J.qs + 1);
  const int64_t a2 = group_lower_pos<64>(R.pos, 0, a, (int64_t)J.qs - R.scal[2]);
  int64_t adj = 0;
  // reads at pos == qs whose span ends before it (no reference-consuming op)
  for (int64_t r = a + lane; r < a1; r += 64) {
    const RMeta m = R.meta[r];
    if ((m.info & RI_KEEP) && m.aend != 0 && m.aend < J.qs) adj--;
  }
  // reads that start before qs and reach it
  for (int64_t r = a2 + lane; r < a; r += 64) {
    const RMeta m = R.meta[r];
    const int32_t se = m.aend != 0 ? m.aend : m.pos;
    if ((m.info & RI_KEEP) && se >= J.qs) adj++;
  }
  adj = wave_sum(adj);
  // P ops and malformed/edge reads: only scanned when the set has any
  int64_t unk = 0, bad_r = INT64_MAX, edge_r = INT64_MAX;
  if (R.scal[4] || R.scal[5]) {
    for (int64_t r = a2 + lane; r < b; r += 64) {
      const RMeta m = R.meta[r];
      if (!(m.info & RI_KEEP)) continue;
      const int32_t se = m.aend != 0 ? m.aend : m.pos;
      if (!(m.pos <= J.qe && se >= J.qs)) continue;
      unk += (m.info & RI_UNK_MASK) >> RI_UNK_SHIFT;
      if ((m.info & RI_BAD) && r < bad_r) bad_r = r;
      if ((m.info & RI_EDGE_CLIP) && r < edge_r) edge_r = r;
    }
    unk = wave_sum(unk);
    for (int d = 32; d >= 1; d >>= 1) {
      int64_t o1 = __shfl_xor(bad_r, d, 64), o2 = __shfl_xor(edge_r, d, 64);
      bad_r = o1 < bad_r ? o1 : bad_r;
      edge_r = o2 < edge_r ? o2 : edge_r;
    }
  }
  if (lane == 0) {
    JobStat S;
    S.read_count = (int64_t)kp[b] - (int64_t)kp[a] + adj;
    S.base_count = 0;
    S.aligned = 0;
    S.unknown_ops = unk;
    S.err_read_edge = edge_r;
    S.err_read_inval = bad_r;
    S.overflow = S.min_depth = S.n_confirmed = S.cand_lo = S.cand_hi = S.pad = 0;
    A.st[j] = S;
  }
}

}  // namespace

// Block 0 clears the batch's counters, the next blocks take four regions
// each (job_begin).  With plan set (windows taken in their own order, so no
// cost order is needed) the blocks after them plan the windows and write
// their heads: the whole preparation of a plain launch is this kernel.
__global__ void __launch_bounds__(256) k_begin(EngineArgs A, const uint32_t* const* keep_prefix, uint32_t* counters,
                                               int n_counters, WinDev* wins, int plan) {
  const int32_t jb = (A.n_jobs + 3) / 4;
  int32_t b = (int32_t)blockIdx.x;
  if (b == 0) {
    if ((int)threadIdx.x < n_counters) counters[threadIdx.x] = 0;
    if (!plan) for (int k = threadIdx.x; k < (PL_BIN_COPIES + 1) * PL_COST_BINS; k += 256) A.bins[k] = 0;
    return;
  }
  b -= 1;
  if (b < jb) {
    const int32_t j = b * 4 + (int32_t)(threadIdx.x >> 6);
    if (j < A.n_jobs) job_begin(A, keep_prefix, j);
    return;
  }
  if (plan) plan_windows(A, b - jb, wins, true);
}

// The windows' read ranges and cost bins (persistent form), 64 windows a
// block.  Most windows of an even batch fall in a few bins, so what bounded
// this kernel was atomics on a few addresses of one cache line: a block
// counts in LDS, and its bins go to one of PL_BIN_COPIES copies, lines
// apart.  38,062 windows: 265 us with an atomic a window and the whole set
// searched for each window's last read, 41 us so.
__global__ void __launch_bounds__(1024) k_plan(EngineArgs A, WinDev* wins) {
  __shared__ uint32_t cnt[PL_COST_BINS];
  if (threadIdx.x < PL_COST_BINS) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int bin = plan_windows(A, blockIdx.x, wins, false);
  if (bin >= 0 && (threadIdx.x & 15) == 0) atomicAdd(&cnt[bin], 1u);
  __syncthreads();
  if (threadIdx.x < PL_COST_BINS && cnt[threadIdx.x])
    atomicAdd(&A.bins[(blockIdx.x % PL_BIN_COPIES) * PL_COST_BINS + threadIdx.x], cnt[threadIdx.x]);
}

// The window heads in cost order, most work first: a window's queue slot is
// its bin's first slot, plus the slots its bin has handed out (one atomic per
// bin and block), plus its rank in its block.  The order inside a bin is of
// no consequence.  (A radix sort of exact keys took ten launches.)
__global__ void __launch_bounds__(256) k_heads(EngineArgs A) {
  static_assert(PL_COST_BINS == 256, "one bin per thread");
  __shared__ uint32_t start[PL_COST_BINS], cnt[PL_COST_BINS];
  __shared__ uint32_t ws[4];
  const int tid = threadIdx.x;
  uint32_t v = 0;
#pragma unroll
  for (int k = 0; k < PL_BIN_COPIES; k++) v += A.bins[k * PL_COST_BINS + tid];
  const uint32_t inc = wave_scan_dpp(v);
  if ((tid & 63) == 63) ws[tid >> 6] = inc;
  cnt[tid] = 0;
  __syncthreads();
  uint32_t s = inc - v;
  for (int w = 0; w < (tid >> 6); w++) s += ws[w];
  start[tid] = s;
  const int32_t w = (int32_t)blockIdx.x * 256 + tid;
  uint32_t bin = 0, rank = 0;
  if (w < A.n_wins) { bin = A.cost[w]; rank = atomicAdd(&cnt[bin], 1u); }
  __syncthreads();
  if (cnt[tid]) start[tid] += atomicAdd(&A.bins[PL_BIN_COPIES * PL_COST_BINS + tid], cnt[tid]);
  __syncthreads();
  if (w < A.n_wins) put_head((WinHead*)A.heads, (int32_t)(start[bin] + rank), w, A.wins[w], A.jobs[A.wins[w].job], A.wins[w].m0);
}

// identity permutation + its length, for a sort whose count is in device memory
__global__ void k_iota(uint32_t* v, int32_t n, uint32_t* n_out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = (uint32_t)i;
  if (blockIdx.x == 0 && threadIdx.x == 0) *n_out = (uint32_t)n;
}

// ------------------------------------------------------------------ window
namespace {

// What both forms of the window's counters share: the fragment differences,
// the evidence records, errors.
struct SinkBase {
  int32_t *pc, *is;
  IndelRec* lrec;        // the window's record buffer in LDS
  uint32_t lrec_cap;
  uint32_t* lrec_n;
  JobStat* st;
  int64_t bcount, aligned_n;
  __device__ void frag(int p, int d, int32_t size) { atomicAdd(&pc[p], d); atomicAdd(&is[p], size); }
  __device__ void aligned(int n) { aligned_n += n; }
  __device__ void count_base() { bcount++; }
  __device__ void edge(int64_t r) { atomicMin((unsigned long long*)&st->err_read_edge, (unsigned long long)r); }
};

// 64-bit counters for any depth: 76 bytes a position.
struct WideLds : SinkBase {
  static constexpr bool narrow = false;
  int W;
  unsigned long long *bs, *mqq, *ins_, *del_;
  uint32_t *bad_, *clp_;
  int32_t* bd;           // badPair differences of bad runs (clips, invalid reads' M bases)
  IndelRec* spill;
  uint2* spill_at;
  uint32_t* spill_n;
  uint32_t spill_cap;
  int32_t wi;
  int32_t* overflow;
  __device__ uint32_t* init(unsigned long long* lds, int w) {   // returns the depth histogram's place
    W = w;
    bs = lds; mqq = bs + 4 * W; ins_ = mqq + W; del_ = ins_ + W;
    bad_ = (uint32_t*)(del_ + W); clp_ = bad_ + W;
    pc = (int32_t*)(clp_ + W); is = pc + W; bd = is + W;
    return (uint32_t*)(bd + W);
  }
  __device__ void base(int p, int b, int32_t q, int32_t mq1) {
    atomicAdd(&bs[b * W + p], (unsigned long long)pack_base(q, mq1));
    atomicAdd(&mqq[p], (unsigned long long)pack_mq_q(mq1, q));
  }
  __device__ void slide(int p, int b, int32_t q, int32_t mq1) { base(p, b, q, mq1); }
  __device__ void bad(int p, int n) { atomicAdd(&bad_[p], (uint32_t)n); }
  __device__ void bad_run(int p, int n, int nW) { atomicAdd(&bd[p], 1); if (p + n < nW) atomicAdd(&bd[p + n], -1); }
  __device__ void clip(int p) { atomicAdd(&clp_[p], 1u); }
  // records collect in LDS and reach HBM together at the window's end; a
  // window with more than fit spills the rest (k_spill_place)
  __device__ void emit(const IndelRec& e) {
    const uint32_t j = atomicAdd(lrec_n, 1u);
    if (j < lrec_cap) { lrec[j] = e; return; }
    const uint32_t i = atomicAdd(spill_n, 1u);
    if (i < spill_cap) { spill[i] = e; spill_at[i] = make_uint2((uint32_t)wi, j); }
    else *overflow = 1;
  }
  __device__ void ins(int p, int32_t q, int32_t mq1, const IndelRec& e) {
    atomicAdd(&ins_[p], (unsigned long long)((1ull << 32) + (uint64_t)mq1));
    atomicAdd(&mqq[p], (unsigned long long)((uint64_t)(int64_t)q << 32));
    emit(e);
  }
  __device__ void del(int p, int32_t q, int32_t mq1, const IndelRec& e) {
    atomicAdd(&del_[p], (unsigned long long)((1ull << 32) + (uint64_t)mq1));
    atomicAdd(&mqq[p], (unsigned long long)pack_mq_q(mq1, q));
    emit(e);
  }
  __device__ int32_t bad_diff(int i) const { return bd[i]; }
  __device__ void finish(int p, uint8_t refb, const KConf& cf, int32_t pcv, int32_t isv, int32_t bdv, PosOut& o) const {
    const uint64_t b4[4] = {bs[p], bs[W + p], bs[2 * W + p], bs[3 * W + p]};
    finalize_position(b4, mqq[p], ins_[p], del_[p], bad_[p] + (uint32_t)bdv, clp_[p], pcv, isv, refb, cf, o);
  }
};

// 32-bit counters (NarrowCol), 60 bytes a position: a base of an m0 read is
// one 32-bit LDS add where the 64-bit form takes two 64-bit ones.  A window
// of more than PL_NARROW_MAX reads, slid bases and indels, of more records
// than the LDS buffer holds, or of a set with reads of many clips is left to
// the wide form (k_window): its quals and counts could leave their 20 and 12
// bits.  512 positions, narrow for wide: 24 Mb at 60x 2.05 -> 1.80 ms, 2 Mb
// at 100x 0.45 -> 0.30 ms (at 60x the window's own phases, not the bases,
// take two thirds of the time).
struct NarrowLds : SinkBase {
  static constexpr bool narrow = true;
  int W;
  int32_t m0;
  uint32_t* cell;        // [4][W]
  int32_t *qc, *mc, *qs; // [4][W], [W], [W]
  uint32_t *in_, *de_;
  uint32_t* cb;          // clips << 16, plus the badPair difference (signed)
  uint32_t* extra;       // slid bases and indels of the window
  __device__ uint32_t* init(unsigned long long* lds, int w) {
    W = w;
    cell = (uint32_t*)lds;
    qc = (int32_t*)(cell + 4 * W); mc = qc + 4 * W; qs = mc + W;
    in_ = (uint32_t*)(qs + W); de_ = in_ + W; cb = de_ + W;
    pc = (int32_t*)(cb + W); is = pc + W;
    return (uint32_t*)(is + W);
  }
  __device__ void base(int p, int b, int32_t q, int32_t mq1) {
    atomicAdd(&cell[b * W + p], (1u << PL_NARROW_SHIFT) + (uint32_t)q);
    if (mq1 != m0) { atomicAdd(&qc[b * W + p], (mq1 - m0) * q); atomicAdd(&mc[p], mq1 - m0); }
  }
  __device__ void slide(int p, int b, int32_t q, int32_t mq1) { atomicAdd(extra, 1u); base(p, b, q, mq1); }
  __device__ void bad(int p, int n) { atomicAdd(&cb[p], (uint32_t)n); if (p + 1 < W) atomicAdd(&cb[p + 1], 0u - (uint32_t)n); }
  __device__ void bad_run(int p, int n, int nW) { atomicAdd(&cb[p], 1u); if (p + n < nW) atomicAdd(&cb[p + n], ~0u); }
  __device__ void clip(int p) { atomicAdd(&cb[p], 1u << 16); }
  __device__ void emit(const IndelRec& e) {
    const uint32_t j = atomicAdd(lrec_n, 1u);
    if (j < lrec_cap) lrec[j] = e;
  }
  __device__ void ins(int p, int32_t q, int32_t mq1, const IndelRec& e) {
    atomicAdd(extra, 1u);
    atomicAdd(&in_[p], (1u << PL_NARROW_SHIFT) + (uint32_t)mq1);
    atomicAdd(&qs[p], q);
    emit(e);
  }
  __device__ void del(int p, int32_t q, int32_t mq1, const IndelRec& e) {
    atomicAdd(extra, 1u);
    atomicAdd(&de_[p], (1u << PL_NARROW_SHIFT) + (uint32_t)mq1);
    atomicAdd(&qs[p], q);
    emit(e);
  }
  __device__ int32_t bad_diff(int i) const { return (int32_t)(int16_t)(cb[i] & 0xffffu); }
  __device__ void finish(int p, uint8_t refb, const KConf& cf, int32_t pcv, int32_t isv, int32_t bdv, PosOut& o) const {
    NarrowCol N;
#pragma unroll
    for (int b = 0; b < 4; b++) { N.cell[b] = cell[b * W + p]; N.qcorr[b] = qc[b * W + p]; }
    N.mqcorr = mc[p]; N.qsum = qs[p];
    N.ins = in_[p]; N.del = de_[p];
    const uint32_t x = cb[p];
    N.clips = (x - (uint32_t)(int32_t)(int16_t)(x & 0xffffu)) >> 16; N.bad = (uint32_t)bdv;
    N.pc = pcv; N.is = isv; N.m0 = m0;
    finalize_narrow(N, refb, cf, o);
  }
};

// global-address-space views: loads through them compile to global_load_*
// (vector memory counter only) instead of flat loads that also hold the LDS
// counter the atomics wait on
typedef const int8_t __attribute__((address_space(1))) gi8;
typedef const uint8_t __attribute__((address_space(1))) gu8;
typedef const uint32_t __attribute__((address_space(1))) gu32;

struct __attribute__((aligned(16))) RunL {  // one run of a chunk of reads, one 16-byte LDS read
  int32_t off;     // first chunk of the run in the chunk stream
  uint32_t pi;     // window position | EF_* flags | mq1 << 16
  int32_t q0;      // sequence offset of the run's first base, from the reads' 4-aligned base
  int32_t pad;     // run length in bases
};

__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

}  // namespace

// The segments of a long read (n from sg) that can touch a window: the first
// whose reference span ends at or after L0 in *first, and how many follow
// with their locus below x (both ascend).  An aligned group of 16 lanes a
// read, all 64 lanes of the wave active; both searches probe together.
__device__ __forceinline__ int32_t long_seg_range(const Seg* sg, uint32_t n, int32_t L0, int64_t x, int lane,
                                                  uint32_t* first) {
  static_assert(PL_LONG_READS == 4, "16 lanes a read");
  const int gl = lane & 15, g0 = lane & 48;
  uint32_t lo[2] = {0, 0}, hi[2] = {n, n};
  while (__ballot(hi[0] - lo[0] > 16u || hi[1] - lo[1] > 16u)) {
    bool less[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t m = hi[k] - lo[k];
      less[k] = false;
      if (m > 16u) {
        const Seg& g = sg[lo[k] + (uint32_t)((uint64_t)(gl + 1) * m / 17)];
        less[k] = k == 0 ? seg_end(g) < L0 : (int64_t)seg_key(g) < x;
      }
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint64_t m = hi[k] - lo[k];
      const int c = __popcll((__ballot(less[k]) >> g0) & 0xffffull);
      const uint32_t a = lo[k];
      if (m > 16u) {
        if (c > 0) lo[k] = a + (uint32_t)(c * m / 17) + 1;
        if (c < 16) hi[k] = a + (uint32_t)((c + 1) * m / 17);
      }
    }
  }
  uint32_t at[2];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    bool less = false;
    if (lo[k] + gl < hi[k]) {
      const Seg& g = sg[lo[k] + gl];
      less = k == 0 ? seg_end(g) < L0 : (int64_t)seg_key(g) < x;
    }
    at[k] = lo[k] + (uint32_t)__popcll((__ballot(less) >> g0) & 0xffffull);
  }
  *first = at[0];
  return at[1] > at[0] ? (int32_t)(at[1] - at[0]) : 0;
}

// One workgroup owns a window of W positions; every counter of those
// positions lives in LDS until the window is done.  Each wave takes chunks of
// up to 64 reads, one read per lane: headers are loaded in parallel, each
// read is classified, and the trusted in-window bases of its runs (the M ops
// of 2-bit reads) are piled as one stream of PL_CHUNK-base pieces, one piece
// per lane.  Clips and indels are applied one segment per lane; other reads
// go through walk_read, one wave per read.
//
// What bounds it: latency.  At 60x a window is ~9 batches of pieces a wave
// (a third of the time) and a dozen dependent phases (head, read facts,
// segments, sums, columns, statistics) at 3 waves a SIMD; on 60 Mb at 60x
// VALU issue is half used, LDS a third, HBM 35% of 8 TB/s, and waves wait 65%
// of their cycles.  Measured on 24 Mb, 512 positions: the
// segment of the evidence records and the reference asked for before the
// sums, sums scanned in registers, simple runs in their table before the
// segments are applied (161 VGPRs for 168 and 2 spilled): 1.87 -> 1.80 ms.  Tried and
// slower: 4 waves a SIMD (16 spills, 1.99), loads two batches ahead (13
// spills, 2.09), 512 threads a window (3.86).
static_assert(PL_CHUNK % 2 == 1 && PL_CHUNK <= 31, "an odd chunk of at most 31 bases (two 16-base words)");

// LONG: the batch's read sets hold long reads (their segments and the
// nanopore base rule cost the other batches' kernel seven spilled registers).
// NARROW: the window's counters are 32-bit words (NarrowLds); a window they
// do not hold is added to A.wide_heads, and a wide launch of mode 2 piles those.
// mode: 0 a window per workgroup, 1 windows from the queue, 2 the windows of
// A.wide_heads from their queue.
template <int BLOCK, bool LONG, bool NARROW>
__global__ void __launch_bounds__(BLOCK, NARROW ? PL_NARROW_WAVES_EU : PL_WIN_WAVES_EU) k_window(EngineArgs A, int mode) {
  static_assert(!(LONG && NARROW), "long reads have an event every few bases");
  constexpr int NW = BLOCK / 64;
  using Counters = typename std::conditional<NARROW, NarrowLds, WideLds>::type;
  extern __shared__ __align__(16) unsigned long long lds[];
  const int W = A.W;
  __shared__ uint32_t s_extra, s_ncx;
  __shared__ uint16_t s_cx[NARROW ? PL_WIN_WALKS : 1];   // reads to walk, from win.plo
  const bool persistent = mode != 0;
  auto head_of = [&](int32_t q) { return A.heads[mode == 2 ? A.wide_heads[q] : q]; };
  int32_t* queue = mode == 2 ? A.wqueue : A.queue;
  const int32_t n_heads = mode == 2 ? (int32_t)*A.wide_wins : A.n_wins;
  __shared__ RunL s_run[NW * (2 * 64 + 1)];
  __shared__ int32_t ws_a[NW], ws_b[NW], ws_c[NW];
  __shared__ unsigned long long red[2][NW];
  __shared__ int32_t s_ovf;
  // (the bit tables of a long-read window take the room of 24 records)
  constexpr uint32_t RECS = LONG ? PL_WIN_RECS - 24 : PL_WIN_RECS;
  __shared__ IndelRec s_rec[RECS];
  __shared__ uint32_t s_nrec, s_recbase;
  // a bit per position: nanopore_exclude, and homo_run4 at its region index
  __shared__ uint64_t s_nx[LONG ? PL_MAX_WINDOW / 64 + 1 : 1], s_hx[LONG ? PL_MAX_WINDOW / 64 : 1];
  // the current window's head and the next one's, fetched while the
  // current window is piled (persistent form), with their queue slots
  __shared__ WinHead s_head[2];
  __shared__ int32_t s_slot[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lds_words = ((NARROW ? PL_NARROW_LDS_PER_POS : PL_WIN_LDS_PER_POS) * W) / 8 + 256 / 2;
  const KConf& cf = A.cf;

  if (tid == 0) {
    const int32_t q = persistent ? atomicAdd(queue, 1) : (int32_t)blockIdx.x;
    s_slot[0] = q;
    if (q < n_heads) s_head[0] = head_of(q);
  }
  __syncthreads();
  for (int iter = 0;; iter++) {
    const int cur = iter & 1;
    if (__builtin_amdgcn_readfirstlane(s_slot[cur]) >= n_heads) break;
    if (!persistent && iter > 0) break;
    // the next window's slot: taken now, its head loaded after the read loop
    int32_t next_slot = 0;
    if (persistent && tid == 0) next_slot = atomicAdd(queue, 1);
    // the head through LDS, made wave-uniform so every field is a scalar
    WinHead win;
    {
      const int32_t* hw = (const int32_t*)&s_head[cur];
      int32_t* dw = (int32_t*)&win;
#pragma unroll
      for (int k = 0; k < (int)(sizeof(WinHead) / 4); k++) dw[k] = __builtin_amdgcn_readfirstlane(hw[k]);
    }
    const int32_t wi = win.wi;
    JobDev J;
    J.rs = win.rs; J.start = win.start; J.stop = win.stop; J.qs = win.qs; J.qe = win.qe;
    J.size = win.stop - win.start + 1; J.win0 = 0; J.nwin = 0; J.out = win.out; J.rlo = 0; J.rhi = 0;
    const RSDev& R = A.rs[win.rs];
    const int32_t L0 = J.start + win.p0, L1 = J.start + win.p1, nW = win.p1 - win.p0;
    auto next_window = [&]() {                 // by thread 0
      s_slot[cur ^ 1] = persistent ? next_slot : n_heads;
      if (persistent && next_slot < n_heads) s_head[cur ^ 1] = head_of(next_slot);
    };
    auto to_wide = [&]() { A.wide_heads[atomicAdd(A.wide_wins, 1u)] = s_slot[cur]; };
    const int64_t reads_in = win.hi - win.plo + R.n_outlier;
    if (NARROW && reads_in > PL_NARROW_MAX) {
      if (tid == 0) { to_wide(); next_window(); }
      __syncthreads();
      continue;
    }
    // hot streams of this read set, held in scalar registers for the window
    const int8_t* __restrict__ gq = R.quals;
    const uint8_t* __restrict__ gb = R.bases2;
    const int64_t* __restrict__ gso = R.seq_off;
    const RMeta* __restrict__ gm = R.meta;
    // Each wave takes its own chunks of up to 64 reads (wave-strided over the
    // window's read range): staging, the run scan and the base loop are
    // wave-local, so the read loop has no workgroup barrier.  Where it takes
    // at most a quarter more chunks they are cut to the same size, as many
    // for each wave: 512-position windows of 530 reads 0.318 -> 0.306 ms a
    // 2 Mb batch, but windows of 290 reads, 8 chunks of 37 for 5 of 64,
    // 1.80 -> 1.94 ms a 24 Mb batch (staging is per chunk).  In a set of long
    // reads a chunk is PL_LONG_READS reads: a window has about a hundred.
    RunL* wrun = s_run + wave * (2 * 64 + 1);
    int CR = PL_LONG_READS;
    if (!(LONG && R.all_long)) {
      const int32_t n = (int32_t)(win.hi - win.plo);
      const int32_t ch = (n + 63) >> 6, even = (ch + NW - 1) / NW * NW;
      CR = ch <= NW || 4 * even <= 5 * ch ? (n > even ? (n + even - 1) / even : 1) : 64;
    }
    const bool stager = lane < CR;
    int64_t t0 = win.plo + CR * wave;
    {
      uint4* l4 = (uint4*)lds;   // 16-byte stores: lds is 16-byte aligned
      for (int k = tid; k < lds_words / 2; k += BLOCK) l4[k] = make_uint4(0u, 0u, 0u, 0u);
      if ((lds_words & 1) && tid == 0) lds[lds_words - 1] = 0ull;
    }
    if (tid == 0) { s_ovf = 0; s_nrec = 0; s_extra = 0; s_ncx = 0; }
    const bool nano = LONG && R.nano != 0;
    if constexpr (LONG) {
      for (int q0 = 64 * wave; q0 < W; q0 += BLOCK) {
        const bool in = q0 + lane < nW;
        const uint64_t xm = __ballot(in && nano && nanopore_exclude(R, J, (int64_t)win.p0 + q0 + lane));
        const uint64_t hm = __ballot(in && homo_run4(R, (int64_t)win.p0 + q0 + lane));
        if (lane == 0) { s_nx[q0 >> 6] = xm; s_hx[q0 >> 6] = hm; }
      }
      if (tid == 0) s_nx[W >> 6] = 0;
    }
    auto lr_drop = [&](uint32_t lr, int32_t dl) {
      const int d = dl - L0;
      return ((s_hx[d >> 6] | (lr == PL_LR_NANOPORE ? s_nx[d >> 6] : 0ull)) >> (d & 63) & 1ull) != 0;
    };
    __syncthreads();

    Counters sk;
    uint32_t* hist = sk.init(lds, W);          // PL_HIST entries
    sk.lrec = s_rec; sk.lrec_cap = RECS; sk.lrec_n = &s_nrec;
    sk.st = &A.st[win.job]; sk.bcount = 0; sk.aligned_n = 0;
    int32_t* const pcA = sk.pc;
    int32_t* const isA = sk.is;
    if constexpr (NARROW) {
      sk.m0 = win.m0;
      sk.extra = &s_extra;
    } else {
      sk.spill = A.spill; sk.spill_at = A.spill_at; sk.spill_n = A.spill_n; sk.spill_cap = A.spill_cap; sk.wi = wi;
      sk.overflow = A.overflow;
    }

    for (; t0 < win.hi; t0 += CR * NW) {
      RMeta m = RMeta(); int64_t seq0 = 0, seqE = 0;
      m.info = 0;
      if (stager && t0 + lane < win.hi) { m = gm[t0 + lane]; seq0 = gso[t0 + lane]; seqE = gso[t0 + lane + 1]; }
      const int64_t qbase = gso[t0];
      // ---- stage: one read per lane.  A simple read gives at most one run;
      // a read with clips or indels is applied below one segment per lane;
      // the rest (non-ACGT bases, too many segments) are walked.
      const int64_t r = t0 + lane;
      const int32_t qsh = (int32_t)(qbase & 3);
      Run ru0;
      ru0.n = 0;
      int nrun = 0;
      bool cplx = false, segr = false, lng = false;
      uint32_t rinfo = 0, rop0 = 0;   // facts of a segmented read, for the lanes that apply its segments
      int64_t rseq0 = 0;
      if (stager && r < win.hi) {
        if (!(m.info & RI_OUTLIER) && read_in_query(m, J)) {
          frag_event(m, J, L0, L1, sk);
          if (m.fp_hi >= L0 && m.fp_lo < L1) {
            if (seq0 - qbase >= PL_TILE_SPAN) cplx = true;
            else if (m.info & RI_SIMPLE) nrun = simple_run(m, seq0, cf, L0, L1, &ru0, &sk.aligned_n, &sk.bcount);
            else if (!(m.info & RI_EXOTIC) && ((m.info & RI_SEG_MASK) >> RI_SEG_SHIFT) < RI_SEG_MAX) {
              lng = LONG && (m.info & RI_LR_MASK) != 0;
              segr = !lng;
              rinfo = m.info; rop0 = m.op0; rseq0 = seq0;
            } else {
              cplx = true;
            }
          }
        }
      }
      const int32_t rlen = segr || lng ? (int32_t)(seqE - rseq0) : 0;
      // a run that only adds badPair over a range (M bases of an invalid
      // read) goes to the difference array, not to the base loop
      if (nrun > 0 && (ru0.fl & EF_BAD)) {
        if (ru0.n > 0) sk.bad_run(ru0.p0, ru0.n, nW);
        nrun = 0;
      }
      // ---- run table: simple runs (wave scan), then the segments' runs.  Runs
      // are cut in chunks of PL_CHUNK bases; .off is the run's first chunk in
      // the chunk stream, .n its length in bases.
      const uint64_t v = nrun > 0 ? (1ull << 32) + (uint64_t)((ru0.n + PL_CHUNK - 1) / PL_CHUNK) : 0ull;
      const uint64_t inc = wave_scan_dpp(v);
      const uint64_t tot = lane63(inc);
      if (nrun > 0) {
        const uint64_t ex = inc - v;
        wrun[(int32_t)(ex >> 32)] =
            RunL{(int32_t)(uint32_t)ex, (uint32_t)ru0.p0 | ru0.fl, (int32_t)(ru0.q - qbase) + qsh, ru0.n};
      }
      const int32_t Es = (int32_t)(tot >> 32);
      const int32_t Cs = (int32_t)(uint32_t)tot;
      // ---- reads with clips or indels, one lane per segment: each round
      // loads and applies the segments of as many pending reads as fit the
      // 64 lanes (usually all of the chunk's in one round).  Base-loop runs
      // are staged at wrun[64 ...] and appended after the simple runs; a
      // round whose runs would not fit, or a read of more than 64 segments,
      // joins the walked reads instead.
      int32_t ncr = 0;
      for (uint64_t pend = __ballot(segr); pend;) {
        const bool inp = (pend >> lane) & 1ull;
        const int nsg = inp ? (int)((rinfo & RI_SEG_MASK) >> RI_SEG_SHIFT) : 0;
        const int sinc = wave_scan_dpp(nsg);
        const uint64_t take = __ballot(inp && sinc <= 64);
        if (!take) {                         // over 64 segments: walked with the other complex reads
          if (lane == __ffsll((unsigned long long)pend) - 1) cplx = true;
          pend &= pend - 1;
          continue;
        }
        pend &= ~take;
        int own = -1, sidx = 0;
        for (uint64_t sm = take; sm; sm &= sm - 1) {
          const int o = __ffsll((unsigned long long)sm) - 1;
          const int no = __builtin_amdgcn_readlane(nsg, o);
          const int bo = __builtin_amdgcn_readlane(sinc, o) - no;
          if (lane >= bo && lane < bo + no) { own = o; sidx = lane - bo; }
        }
        const int src = own < 0 ? lane : own;
        const uint32_t info = (uint32_t)__shfl((int)rinfo, src, 64);
        const uint32_t op0 = (uint32_t)__shfl((int)rop0, src, 64);
        const int64_t s0 = ((int64_t)__shfl((int)(rseq0 >> 32), src, 64) << 32) |
                           (uint32_t)__shfl((int)(uint32_t)rseq0, src, 64);
        const int32_t Lc = __shfl(rlen, src, 64);
        const bool has = own >= 0;
        Seg g;
        if (has) g = R.segs[op0 + sidx];
        if (ncr + __popcll(__ballot(has && seg_has_run(cf, info, Lc, L0, L1, g))) > 64) {
          if ((take >> lane) & 1ull) cplx = true;   // runs would not fit: walked instead
          continue;
        }
        Run ru;
        int got = has ? seg_apply(R, J, cf, t0 + own, info, s0, Lc, L0, L1, g, ru, &sk.aligned_n, &sk.bcount, sk, lr_drop) : 0;
        if (got && (ru.fl & EF_BAD)) {
          sk.bad_run(ru.p0, ru.n, nW);
          got = 0;
        }
        const uint64_t gmask = __ballot(got != 0);
        if (got) wrun[64 + ncr + __popcll(gmask & lanemask_lt())] =
            RunL{ru.n, (uint32_t)ru.p0 | ru.fl, (int32_t)(ru.q - qbase) + qsh, 0};
        ncr += __popcll(gmask);
      }
      int32_t Cc = 0;
      if (ncr > 0) {
        // every lane reads its staged run before any lane writes (one wave,
        // LDS operations in order)
        RunL cr = RunL{0, 0u, 0, 0};
        if (lane < ncr) cr = wrun[64 + lane];
        const int32_t cn = lane < ncr ? (cr.off + PL_CHUNK - 1) / PL_CHUNK : 0;
        const int32_t ci = wave_scan_dpp(cn);
        Cc = lane63(ci);
        if (lane < ncr) wrun[Es + lane] = RunL{Cs + ci - cn, cr.pi, cr.q0, cr.off};
      }
      int32_t E = Es + ncr;
      int32_t CT = Cs + Cc;
      // The chunk's long reads follow, PL_LONG_READS at a time and 64 of
      // their segments a round: the runs of each round are a run table of
      // their own for the base loop below.  16 lanes hold one read's facts.
      uint64_t pendl = __ballot(lng);
      int lsrc = 0;
      uint32_t linfo = 0, lfirst = 0;
      int32_t lat = 0, ltot = 0, lp1 = 0, lp2 = 0, lp3 = 0;
      for (;;) {
      if (lane == 0) wrun[E] = RunL{CT, 0u, 0, 0};
      // LDS operations of one wave complete in order: the table written
      // above is what the loop below reads
      __builtin_amdgcn_wave_barrier();
      // ---- the bases of all runs: one chunk of PL_CHUNK consecutive bases of
      // one run per lane.  A chunk's quals come in as PL_CHUNK/4 + 2 dwords
      // and its 2-bit bases as PL_CHUNK/16 + 2, realigned with funnel shifts
      // (the loads of the next batch of chunks are in flight while the
      // current batch does its atomics); each base then costs its word and a
      // 2-bit extract and one LDS atomic (two in the wide form) whose step
      // offset is the instruction's immediate.  Lanes of one run are PL_CHUNK
      // (odd) positions apart, so their atomics spread over all LDS banks.
      if (CT > 0) {
        const int32_t mq = cf.min_qual;
        const uint32_t WB = (NARROW ? 4u : 8u) * (uint32_t)W;   // bytes of one base's counters
        const int64_t qb4 = qbase & ~(int64_t)3, qb16 = qbase & ~(int64_t)15;
        const gu32* tq32 = (const gu32*)(gq + qb4);
        const gu32* tb32 = (const gu32*)(gb + (qb16 >> 2));
        const uint32_t qd = (uint32_t)(qb4 - qb16);
        // Run of chunk cb + lane = the last run whose first chunk is <= it,
        // from the run of chunk cb - 1 (or of chunk 0) on: the first chunks
        // of the runs that start in the batch, as a bit mask.
        auto run_of = [&](int32_t cb, int cur) -> int {
          const int ib = cur + 1 + lane;
          const int32_t bnd = ib <= E ? wrun[ib].off : INT32_MAX;
          const int nb = __popcll(__ballot(bnd < CT && bnd < cb + 64));
          uint64_t starts = 0;
          for (int i = 0; i < nb; i++) starts |= 1ull << (__builtin_amdgcn_readlane(bnd, i) - cb);
          const uint64_t before = starts >> 1;              // starts at or before a lane's chunk: before it, shifted by one
          return cur + (int)(starts & 1ull) +
                 (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(before >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)before, 0u));
        };
        // sequence offset of chunk C of run ru (0 for a lane past the end)
        auto chunk_q = [&](const RunL& ru, int32_t C) -> uint32_t {
          return C < CT ? (uint32_t)(ru.q0 + PL_CHUNK * (C - ru.off)) : 0u;
        };
        // The loads of a batch are issued before the previous batch's
        // atomics, so they are in flight while those run.
        uint32_t qw[PL_CHUNK / 4 + 2], bw[PL_CHUNK / 16 + 2];
        auto load = [&](uint32_t q) {
#pragma unroll
          for (int k = 0; k < PL_CHUNK / 4 + 2; k++) qw[k] = tq32[(q >> 2) + k];
          const uint32_t qq = q + qd;
#pragma unroll
          for (int k = 0; k < PL_CHUNK / 16 + 2; k++) bw[k] = tb32[(qq >> 4) + k];
        };
        int rr = run_of(0, 0);
        RunL ru = wrun[lane < CT ? rr : 0];
        load(chunk_q(ru, lane));
        for (int32_t cb = 0; cb < CT; cb += 64) {
          const int32_t C = cb + lane;
          const bool act = C < CT;
          const int32_t d = PL_CHUNK * (C - ru.off);
          int32_t cnt = ru.pad - d;
          cnt = act ? (cnt < PL_CHUNK ? cnt : PL_CHUNK) : 0;
          const int32_t p = (int32_t)(ru.pi & 0xffffu) + (act ? d : 0);
          const uint32_t q = act ? (uint32_t)(ru.q0 + d) : 0u;
          const int32_t mq1 = (int32_t)((ru.pi >> 16) & 0x1ffu);
          const uint32_t qq = q + qd;
          uint32_t w[PL_CHUNK / 4 + 1];
#pragma unroll
          for (int k = 0; k < PL_CHUNK / 4 + 1; k++) w[k] = __builtin_amdgcn_alignbyte(qw[k + 1], qw[k], q & 3u);
          uint32_t x[PL_CHUNK / 16 + 1];
#pragma unroll
          for (int k = 0; k < PL_CHUNK / 16 + 1; k++) x[k] = __builtin_amdgcn_alignbit(bw[k + 1], bw[k], 2u * (qq & 15u));
          if (nano) {
            // nanopore bases inside CC_GG pile with quality 0: four mask bits to four bytes at a time
            const uint32_t* nx = (const uint32_t*)s_nx + (p >> 5);
            const uint32_t xb = (ru.pi & EF_NANO) && act ? __builtin_amdgcn_alignbit(nx[1], nx[0], (uint32_t)p & 31u) : 0u;
#pragma unroll
            for (int k = 0; k < PL_CHUNK / 4 + 1; k++)
              w[k] &= ~((((xb >> (4 * k)) & 15u) * 0x00204081u & 0x01010101u) * 255u);
          }
          // the next batch: its runs, and its loads
          RunL run_n = ru;
          uint32_t qn = 0u;
          if (cb + 64 < CT) {
            const int cur = lane63(rr);
            rr = run_of(cb + 64, cur);
            run_n = wrun[C + 64 < CT ? rr : cur];
            qn = chunk_q(run_n, C + 64);
          }
          load(qn);
          // The base's counter array is b*W entries on: a 24-bit multiply-add
          // (b < 4, 8*W < 2^24), the step an offset of the instruction.
          if constexpr (NARROW) {
            // Each base's word, its count bit and its qual, is one byte
            // permute of the quals and a mask with 0x10 in the valid bases'
            // bytes (bit 4 of byte 2 of the word: PL_NARROW_SHIFT); a lane's
            // bases past its chunk, or below minQual, add 0, so the 13 adds
            // need no execution mask: 3 VALU instructions a base where the
            // masked form took 7.  (An add of 0 past the window's positions
            // stays inside the counters.)
            static_assert(PL_NARROW_SHIFT == 20, "bit 4 of byte 2");
            uint32_t mm[PL_CHUNK / 4 + 1];
            uint32_t hi = 0;
#pragma unroll
            for (int k = 0; k < PL_CHUNK / 4 + 1; k++) {
              const int32_t nb = cnt - 4 * k;                  // valid bytes of word k
              const uint32_t vm = (uint32_t)((1ull << (8 * (nb < 0 ? 0 : nb > 4 ? 4 : nb))) - 1ull);
              w[k] &= vm;
              mm[k] = vm & 0x10101010u;
              hi |= w[k];
            }
            if (mq > 0 || __ballot((hi & 0x80808080u) != 0u)) {
              // quals below minQual (and negative ones): a byte of (qual | 128) -
              // minQual keeps its top bit where qual >= minQual
              const uint32_t mr = (uint32_t)(mq > 128 ? 128 : mq) * 0x01010101u;
#pragma unroll
              for (int k = 0; k < PL_CHUNK / 4 + 1; k++) {
                const uint32_t ok = mq > 127 ? 0u : (((w[k] | 0x80808080u) - mr) & ~w[k] & 0x80808080u) >> 7;
                w[k] &= ok * 255u;
                mm[k] &= ok * 255u;
              }
            }
            char* const cellp = (char*)(sk.cell + p);
            if (act) {
#pragma unroll
              for (int t = 0; t < PL_CHUNK; t++) {
                const uint32_t v = __builtin_amdgcn_perm(mm[t >> 2], w[t >> 2],
                                                         0x0c000c00u | (uint32_t)((4 + (t & 3)) << 16) | (uint32_t)(t & 3));
                const uint32_t b = (x[t >> 4] >> (2 * (t & 15))) & 3u;
                atomicAdd((uint32_t*)(cellp + __umul24(b, WB)) + t, v);
              }
            }
            const int32_t dm = mq1 - sk.m0;
            if (act && dm != 0) {                              // a read of another adjMq: its bases' differences
              char* const qcp = (char*)(sk.qc + p);
              int32_t* const mcp = sk.mc + p;
#pragma unroll
              for (int t = 0; t < PL_CHUNK; t++) {
                const uint32_t b = (x[t >> 4] >> (2 * (t & 15))) & 3u;
                if (t < cnt) {
                  atomicAdd((int32_t*)(qcp + __umul24(b, WB)) + t, dm * (int32_t)((w[t >> 2] >> (8 * (t & 3))) & 255u));
                  atomicAdd(mcp + t, (mm[t >> 2] >> (8 * (t & 3)) & 255u) ? dm : 0);
                }
              }
            }
          } else {
            // With minQual >= 0 every qual that passes is non-negative, so
            // qual*mq1 >= 0 and the count part is the constant
            // 1 << PL_BASE_SHIFT (pack_base without its sign extension).
            unsigned long long* bsp = sk.bs + p;
            unsigned long long* mqp = sk.mqq + p;
            auto pile = [&](auto nonneg) {
#pragma unroll
              for (int t = 0; t < PL_CHUNK; t++) {
                const int32_t qual = (int32_t)(int8_t)(w[t >> 2] >> (8 * (t & 3)));
                const uint32_t b = (x[t >> 4] >> (2 * (t & 15))) & 3u;
                if (t < cnt && qual >= mq) {
                  unsigned long long* cell = (unsigned long long*)((char*)bsp + __umul24(b, WB)) + t;
                  const unsigned long long v = decltype(nonneg)::value
                                                   ? ((1ull << PL_BASE_SHIFT) | (uint32_t)(qual * mq1))
                                                   : (unsigned long long)pack_base(qual, mq1);
                  atomicAdd(cell, v);
                  atomicAdd(mqp + t, (unsigned long long)pack_mq_q(mq1, qual));
                }
              }
            };
            if (mq >= 0) pile(std::integral_constant<bool, true>{});
            else pile(std::integral_constant<bool, false>{});
          }
          ru = run_n;
        }
      }
      if constexpr (!LONG) break;
      // ---- the next round of a long read's segments
      E = CT = 0;
      bool more = true;
      while (more && E == 0) {
        if (lat >= ltot) {
          if (!pendl) { more = false; break; }
          int own = -1;
#pragma unroll
          for (int j = 0; j < PL_LONG_READS; j++) {
            const int l = pendl ? __ffsll((unsigned long long)pendl) - 1 : -1;
            if ((lane >> 4) == j) own = l;
            pendl &= pendl - 1;
          }
          lsrc = own < 0 ? 0 : own;
          linfo = (uint32_t)__shfl((int)rinfo, lsrc, 64);
          const uint32_t o = (uint32_t)__shfl((int)rop0, lsrc, 64);
          uint32_t lo = 0, n = 0;
          int32_t reach = 0;
          if (own >= 0) { const Seg h = R.segs[o]; n = (uint32_t)h.len; reach = h.fin; }
          lfirst = o + 1;
          const int32_t cnt = long_seg_range(R.segs + lfirst, n, L0, (int64_t)L1 + reach, lane, &lo);
          lfirst += lo;
          const int32_t c0 = __builtin_amdgcn_readlane(cnt, 0), c1 = __builtin_amdgcn_readlane(cnt, 16),
                        c2 = __builtin_amdgcn_readlane(cnt, 32), c3 = __builtin_amdgcn_readlane(cnt, 48);
          lat = 0;
          lp1 = c0; lp2 = lp1 + c1; lp3 = lp2 + c2; ltot = lp3 + c3;
          continue;
        }
        const int32_t t = lat + lane;
        const bool has = t < ltot;
        const int j = (t >= lp1) + (t >= lp2) + (t >= lp3);
        const int from = 16 * j;
        const int src = __shfl(lsrc, from, 64);
        const uint32_t info = (uint32_t)__shfl((int)linfo, from, 64);
        const uint32_t at = (uint32_t)__shfl((int)lfirst, from, 64) + (uint32_t)(t - (j == 0 ? 0 : j == 1 ? lp1 : j == 2 ? lp2 : lp3));
        const int64_t s0 = ((int64_t)__shfl((int)(rseq0 >> 32), src, 64) << 32) |
                           (uint32_t)__shfl((int)(uint32_t)rseq0, src, 64);
        const int32_t Lc = __shfl(rlen, src, 64);
        lat += 64;
        Seg g;
        if (has) g = R.segs[at];
        Run ru;
        ru.n = 0;
        int got = has ? seg_apply(R, J, cf, t0 + src, info, s0, Lc, L0, L1, g, ru, &sk.aligned_n, &sk.bcount, sk, lr_drop) : 0;
        if (got && (ru.fl & EF_BAD)) {
          sk.bad_run(ru.p0, ru.n, nW);
          got = 0;
        }
        const uint64_t lv = got ? (1ull << 32) + (uint64_t)((ru.n + PL_CHUNK - 1) / PL_CHUNK) : 0ull;
        const uint64_t li = wave_scan_dpp(lv), lt = lane63(li);
        if (got) wrun[(int32_t)((li - lv) >> 32)] =
            RunL{(int32_t)(uint32_t)(li - lv), (uint32_t)ru.p0 | ru.fl, (int32_t)(ru.q - qbase) + qsh, ru.n};
        E = (int32_t)(lt >> 32);
        CT = (int32_t)(uint32_t)lt;
      }
      if (!more) break;
      }
      // ---- everything else about the chunk's complex reads: the wide form
      // walks them here, the narrow one after the read loop, where the
      // loop's registers are free
      if constexpr (NARROW) {
        if (cplx) {
          const uint32_t k = atomicAdd(&s_ncx, 1u);
          if (k < PL_WIN_WALKS) s_cx[k] = (uint16_t)(r - win.plo);
        }
      } else {
        for (uint64_t cm = __ballot(cplx); cm; cm &= cm - 1) {
          const int l = __ffsll((unsigned long long)cm) - 1;
          walk_read(R, J, cf, t0 + l, L0, L1, lane, 64, sk, false);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    bool many_clips = false;
    // reads that reach the window only through their fragments: 8 bytes
    // each, +1/+size at position 0 summed per wave
    {
      // read the descriptors again here rather than hold them through the read loop
      asm volatile("" ::: "memory");
      const FragTail* __restrict__ ft = R.ftail;
      many_clips = NARROW && R.scal[7] != 0;
      const int64_t flo = win.lo, fhi = win.plo;
      uint32_t c0 = 0, s0 = 0;
      for (int64_t r = flo + tid; r < fhi; r += BLOCK) {
        const FragTail t = ft[r];
        if (frag_tail_event(t, L0, L1, sk)) { c0++; s0 += (uint32_t)t.size; }
      }
      c0 = wave_total_dpp(c0);
      s0 = wave_total_dpp(s0);
      if (lane == 0 && c0) sk.frag(0, (int32_t)c0, (int32_t)s0);
    }
    if constexpr (!NARROW) {
      for (int64_t k = wave; k < R.n_outlier; k += NW)
        walk_read(R, J, cf, uniform64(R.outliers[k]), L0, L1, lane, 64, sk, true);
    }
    if (tid == 0) next_window();
    __syncthreads();
    if constexpr (NARROW) {
      const int32_t ncx = s_ncx <= PL_WIN_WALKS ? (int32_t)s_ncx : 0;
      const int32_t nwk = ncx + (int32_t)R.n_outlier;
      if (nwk > 0) {
        for (int32_t k = wave; k < nwk; k += NW)
          walk_read(R, J, cf, uniform64(k < ncx ? win.plo + s_cx[k] : R.outliers[k - ncx]), L0, L1, lane, 64, sk, k >= ncx);
        __syncthreads();
      }
    }
    if (NARROW && (s_nrec > RECS || many_clips || s_ncx > PL_WIN_WALKS || reads_in + s_extra > PL_NARROW_MAX)) {
      // beyond the narrow counters: nothing of the window has left the
      // workgroup, the wide form piles it again
      if (tid == 0) to_wide();
      __syncthreads();
      continue;
    }

    // Each wave finishes one span of the window's 64-position tiles.  The
    // physCov, insertSize and badPair differences are summed a span (Int adds
    // wrap like Java's: 32-bit adds do the same), and scanned in registers
    // tile by tile.  What has a memory latency of its own, the segment of the
    // window's evidence records and the first tile's reference bases, is
    // asked for before the sums.
    const int span = 64 * (((W >> 6) + NW - 1) / NW), q_lo = span * wave, q_hi = q_lo + span < W ? q_lo + span : W;
    const uint32_t nt = s_nrec;
    uint32_t recb = 0;
    if (tid == 0 && nt) recb = atomicAdd(A.rec_n, nt);
    const uint8_t* __restrict__ gref = R.ref + (L0 - 1);
    uint8_t refN = q_lo + lane < nW ? gref[q_lo + lane] : (uint8_t)0;
    {
      int32_t spc = 0, sis = 0, sbd = 0;
      for (int p = q_lo + lane; p < q_hi; p += 64) {
        spc = j_add(spc, pcA[p]); sis = j_add(sis, isA[p]); sbd = j_add(sbd, sk.bad_diff(p));
      }
      spc = wave_total_dpp(spc); sis = wave_total_dpp(sis); sbd = wave_total_dpp(sbd);
      if (lane == 0) { ws_a[wave] = spc; ws_b[wave] = sis; ws_c[wave] = sbd; }
    }
    if (tid == 0) s_recbase = recb;
    __syncthreads();
    int32_t cpc = 0, cis = 0, cbd = 0;
    for (int w2 = 0; w2 < wave; w2++) {
      cpc = j_add(cpc, ws_a[w2]); cis = j_add(cis, ws_b[w2]); cbd = j_add(cbd, ws_c[w2]);
    }
    // the window's evidence records, in one segment of the batch's:
    // coalesced 32-byte stores (room for the spilled ones at its end)
    {
      const uint32_t base = s_recbase, nl = nt < RECS ? nt : RECS;
      if (tid == 0) {
        A.win_rec[2 * wi] = base;
        A.win_rec[2 * wi + 1] = nt;
        if (nt && base + nt > A.rec_cap) *A.overflow = 1;
      }
      for (uint32_t t = tid; t < nl; t += BLOCK) {
        const uint32_t k = base + t;
        if (k < A.rec_cap) A.rec[k] = s_rec[t];
      }
    }
    const int64_t G = A.G;
    uint32_t wmask = 0;   // bit i: position q_lo + 64*i + lane is wide
    for (int q0 = q_lo, it = 0; q0 < q_hi; q0 += 64, it++) {
      const int p = q0 + lane;
      const bool act = p < nW;
      const uint8_t refb = refN;
      if (q0 + 64 < q_hi) refN = p + 64 < nW ? gref[p + 64] : (uint8_t)0;
      const int32_t ipc = j_add(cpc, wave_scan_dpp(pcA[p])), iis = j_add(cis, wave_scan_dpp(isA[p])),
                    ibd = j_add(cbd, wave_scan_dpp(sk.bad_diff(p)));
      cpc = lane63(ipc); cis = lane63(iis); cbd = lane63(ibd);
      bool is_cand = false, defer = false;
      if (act) {
        PosOut o;
        sk.finish(p, refb, cf, ipc, iis, ibd, o);
        const int64_t g = J.out + win.p0 + p;
#pragma unroll
        for (int f = 0; f < PL_NFIELDS; f++) A.pile[(int64_t)f * G + g] = o.f[f];
        if (o.wide) { o.call.flags |= PL_CF_WIDE; wmask |= 1u << it; }
        A.calls[g] = o.call;
        if (o.overflow) s_ovf = 1;
        const int d = call_disp(o.call);
        defer = o.defer;
        is_cand = !o.defer && (d == PL_D_SNP || d == PL_D_AMB);
        if (!o.defer && d == PL_D_CONFIRMED) {
          const int64_t dep = (int64_t)(uint32_t)o.f[0] + (uint32_t)o.f[1] + (uint32_t)o.f[2] + (uint32_t)o.f[3] +
                              o.f[PL_F_DELETIONS];
          atomicAdd(&hist[dep > 255 ? 255 : (dep < 0 ? 0 : dep)], 1u);
        }
      }
      // the candidates as a bit per position, in order without a sort; the
      // deferred columns as a list, those of 64 positions together in order
      // (indel_columns finds its way back by that)
      const uint64_t cm = __ballot(is_cand);
      if (lane == 0) A.cmask[(int64_t)wi * (W >> 6) + (q0 >> 6)] = cm;
      const uint32_t kd = wave_append(A.defer_n, defer);
      if (defer) {
        if (kd < A.defer_cap) A.defer[kd] = (uint32_t)(J.out + win.p0 + p);
        else *A.overflow = 1;
      }
    }
    // wide columns (a qualSum beyond int32): the window's entries, in one
    // segment of the batch's list, with their exact sums from the LDS words
    if (!NARROW && __syncthreads_or(wmask != 0)) {
      const uint32_t mine = (uint32_t)__popc(wmask);
      const uint32_t inc = wave_scan_dpp(mine);
      if (lane == 63) ws_a[wave] = (int32_t)inc;
      __syncthreads();
      uint32_t pre = inc - mine, tot = 0;
      for (int w2 = 0; w2 < NW; w2++) { if (w2 < wave) pre += (uint32_t)ws_a[w2]; tot += (uint32_t)ws_a[w2]; }
      if (tid == 0) {
        s_recbase = atomicAdd(A.wide_n, tot);
        A.win_wide[2 * wi] = (int32_t)s_recbase;
        A.win_wide[2 * wi + 1] = (int32_t)tot;
      }
      __syncthreads();
      for (uint32_t m = wmask; m; m &= m - 1) {
        const int p = q_lo + 64 * (__ffs(m) - 1) + lane;
        const uint32_t k = s_recbase + pre++;
        if (k < A.wide_cap) {
          WideCol wc;
          wc.gpos = (uint32_t)(J.out + win.p0 + p);
          wc.pad = 0;
          if constexpr (!NARROW) for (int b = 0; b < 4; b++) { uint32_t n; unpack_base(sk.bs[b * W + p], &wc.qs[b], &n); }
          A.wide[k] = wc;
        } else {
          *A.overflow = 1;
        }
      }
    } else if (tid == 0) {
      A.win_wide[2 * wi] = 0;
      A.win_wide[2 * wi + 1] = 0;
    }
    // region baseCount and the aligned-base unit
    unsigned long long bc = wave_total_dpp((unsigned long long)sk.bcount);
    unsigned long long al = wave_total_dpp((unsigned long long)sk.aligned_n);
    if (lane == 0) { red[0][wave] = bc; red[1][wave] = al; }
    __syncthreads();
    JobStat& S = A.st[win.job];
    if (tid == 0) {
      unsigned long long t0s = 0, t1s = 0;
      for (int w2 = 0; w2 < NW; w2++) { t0s += red[0][w2]; t1s += red[1][w2]; }
      if (t0s) atomicAdd((unsigned long long*)&S.base_count, t0s);
      if (t1s) atomicAdd((unsigned long long*)&S.aligned, t1s);
      if (s_ovf) atomicOr(&S.overflow, 1);
    }
    for (int d = tid; d < PL_HIST; d += BLOCK)
      if (hist[d]) atomicAdd(&A.hist[(int64_t)win.job * PL_HIST + d], hist[d]);
    __syncthreads();
  }
}

template __global__ void k_window<256, false, true>(EngineArgs, int);
template __global__ void k_window<512, false, true>(EngineArgs, int);
template __global__ void k_window<1024, false, true>(EngineArgs, int);
template __global__ void k_window<256, false, false>(EngineArgs, int);
template __global__ void k_window<512, false, false>(EngineArgs, int);
template __global__ void k_window<1024, false, false>(EngineArgs, int);
template __global__ void k_window<256, true, false>(EngineArgs, int);
template __global__ void k_window<512, true, false>(EngineArgs, int);
template __global__ void k_window<1024, true, false>(EngineArgs, int);

// ------------------------------------------------------------------ records
// Spilled records into their windows' segments, each at the place it took
// among the window's records when it was found.
__global__ void __launch_bounds__(256) k_spill_place(EngineArgs A) {
  const uint32_t n = *A.spill_n < A.spill_cap ? *A.spill_n : A.spill_cap;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint2 at = A.spill_at[i];
    const uint32_t k = A.win_rec[2 * at.x] + at.y;
    if (k < A.rec_cap) A.rec[k] = A.spill[i];
  }
}

// ------------------------------------------------------------------ radix sort
// One stable 8-bit pass of an LSD sort of (hi:lo, v) records held as three
// arrays: digits per tile (k_rs_hist), the scan of digit-major counts, and
// the scatter.  A digit comes from lo for shift < 32, else from hi.
__device__ __forceinline__ uint32_t rs_digit(const uint32_t* lo, const uint32_t* hi, uint32_t i, int shift) {
  return (shift < 32 ? lo[i] >> shift : hi[i] >> (shift - 32)) & 255u;
}
// Few tiles (FUSED): counts are kept tile by tile, and every block of the
// scatter adds up the tiles before it itself, one coalesced load a tile, in
// place of three scan kernels of 15 us together.  75 tiles: scatter 13 -> 16
// us, so a pass 34 -> 22 us.  A sort that tiles of 1,024 records cut in no
// more tiles than RS_FUSED_TILES takes those: shorter blocks.  K-mer graphs
// of 130,000 / 200,000 / 520,000 / 700,000 / 2,000,000 occurrences with the
// line at 64 tiles: 202 / 210 / 276 / 279 / 361 us, at 128: 187 / 211 / 240 /
// 279 / 360, at 256: 184 / 197 / 238 / 244 / 361, at 512: 189 / 201 / 294 /
// 250 / 403 (the loads are as long as the scans were).
template <int ITEMS, bool FUSED>
__global__ void __launch_bounds__(256) k_rs_hist(const uint32_t* lo, const uint32_t* hi, uint32_t n, int shift,
                                                 uint32_t* hist, int32_t nblocks) {
  __shared__ uint32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t base = blockIdx.x * (256 * ITEMS);
#pragma unroll
  for (int i = 0; i < ITEMS; i++) {
    const uint32_t idx = base + i * 256 + threadIdx.x;
    if (idx < n) atomicAdd(&h[rs_digit(lo, hi, idx, shift)], 1u);
  }
  __syncthreads();
  hist[FUSED ? (int64_t)blockIdx.x * 256 + threadIdx.x : (int64_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// A tile's records are ranked wave by wave (each wave a quarter of the tile,
// 64 records a round, no workgroup barrier between rounds), put in digit
// order in LDS and stored from there, so that consecutive lanes store
// consecutive records of a digit.  12.4 M records of 12 bytes: 100 us a
// pass, 3.0 TB/s read and written (its stores come in runs of ~16 records).  off: the scanned counts, or the tiles' own (FUSED).
template <int ITEMS, bool FUSED>
__global__ void __launch_bounds__(256) k_rs_scatter(const uint32_t* lo, const uint32_t* hi, const uint32_t* v,
                                                    uint32_t* lo2, uint32_t* hi2, uint32_t* v2, uint32_t n, int shift,
                                                    const uint32_t* off, int32_t nblocks) {
  constexpr uint32_t TILE = 256 * ITEMS;
  __shared__ uint32_t cnt[4][256];
  __shared__ uint32_t dst[256];                              // a digit's place in the output, less its place in the tile
  __shared__ uint32_t ws[4], wd[4];
  __shared__ uint32_t slo[TILE], shi[TILE], sv[TILE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int w = 0; w < 4; w++) cnt[w][tid] = 0;
  __syncthreads();
  const uint32_t base = blockIdx.x * TILE, wbase = base + (uint32_t)wave * (TILE / 4);
  const uint32_t have = n - base < TILE ? n - base : TILE;
  uint32_t kl[ITEMS], kh[ITEMS], kv[ITEMS], at[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    const uint32_t i = wbase + 64 * r + lane;
    const bool in = i < n;
    kl[r] = in ? lo[i] : 0u;
    kh[r] = in ? hi[i] : 0u;
    kv[r] = in ? v[i] : 0u;
  }
#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    const bool in = wbase + 64 * r + lane < n;
    const uint32_t d = (shift < 32 ? kl[r] >> shift : kh[r] >> (shift - 32)) & 255u;
    uint64_t m = __ballot(in);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = ((d >> b) & 1u) != 0;
      const uint64_t bb = __ballot(in && bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t rank = (uint32_t)__popcll(m & lanemask_lt());
    // one wave's LDS operations complete in order: every lane reads the
    // count before its digit's first lane raises it
    at[r] = cnt[wave][d] + rank;
    __builtin_amdgcn_wave_barrier();
    if (in && rank == 0) cnt[wave][d] += (uint32_t)__popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    uint32_t c[4], t = 0;
    for (int w = 0; w < 4; w++) { c[w] = cnt[w][tid]; t += c[w]; }
    const uint32_t inc = wave_scan_dpp(t);
    uint32_t before = 0, all = 0, incd = 0;
    if constexpr (FUSED) {
      const int32_t me = (int32_t)blockIdx.x;
#pragma unroll 8
      for (int32_t k = 0; k < nblocks; k++) {
        const uint32_t x = off[256 * k + tid];
        all += x;
        before += k < me ? x : 0u;
      }
      incd = wave_scan_dpp(all);
      if (lane == 63) wd[wave] = incd;
    } else {
      before = off[(int64_t)tid * nblocks + blockIdx.x];
    }
    if (lane == 63) ws[wave] = inc;
    __syncthreads();
    uint32_t s = inc - t;
    for (int w = 0; w < wave; w++) s += ws[w];
    if constexpr (FUSED) {
      before += incd - all;
      for (int w = 0; w < wave; w++) before += wd[w];
    }
    dst[tid] = before - s;
    for (int w = 0; w < 4; w++) { cnt[w][tid] = s; s += c[w]; }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    if (wbase + 64 * r + lane < n) {
      const uint32_t d = (shift < 32 ? kl[r] >> shift : kh[r] >> (shift - 32)) & 255u;
      const uint32_t p = cnt[wave][d] + at[r];
      slo[p] = kl[r];
      shi[p] = kh[r];
      sv[p] = kv[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    const uint32_t p = 256 * r + tid;
    if (p < have) {
      const uint32_t a = slo[p], b = shi[p];
      const uint32_t o = dst[(shift < 32 ? a >> shift : b >> (shift - 32)) & 255u] + p;
      lo2[o] = a;
      hi2[o] = b;
      v2[o] = sv[p];
    }
  }
}

template __global__ void k_rs_hist<4, true>(const uint32_t*, const uint32_t*, uint32_t, int, uint32_t*, int32_t);
template __global__ void k_rs_hist<16, true>(const uint32_t*, const uint32_t*, uint32_t, int, uint32_t*, int32_t);
template __global__ void k_rs_hist<16, false>(const uint32_t*, const uint32_t*, uint32_t, int, uint32_t*, int32_t);

// ------------------------------------------------------------------ indel pass
namespace {
__device__ __forceinline__ int32_t job_of(const JobDev* jobs, int32_t n_jobs, int64_t g) {
  int32_t lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    int32_t m = (lo + hi + 1) >> 1;
    if (jobs[m].out <= g) lo = m; else hi = m - 1;
  }
  return lo;
}
}  // namespace

namespace {

// The strict majority over a column's records, by the whole wave.  The
// window's records are not sorted: a window holds a handful, and the wave
// tests 64 keys at a time, which costs less than sorting every record of
// the batch did (four radix passes, 20 launches).  Each lane runs a
// Boyer-Moore vote over the matching records of its strided share,
// comparing (length, hash) classes; the 64 partial votes are merged pairwise
// (a merge keeps a majority class if there is one), and the winning class's
// string is counted exactly.  A class with a strict majority whose
// representative string falls short (a hash collision) is resolved by the
// serial scan.  Same result as col_majority.
__device__ Majority wave_majority(const RSDev& R, const ColRecs& C, int lane) {
  Majority m;
  m.n = m.win = 0;
  m.rec = -1;
  int32_t vl = -1, vc = 0, n = 0;
  uint32_t vh = 0;
  int64_t vr = -1;
  for (int64_t i = C.a + lane; i < C.b; i += 64) {
    const IndelRec& e = C.recs[i];
    if (e.key != C.key) continue;
    n++;
    if (vc == 0) { vl = e.len; vh = e.hash; vr = i; vc = 1; }
    else if (e.len == vl && e.hash == vh) vc++;
    else vc--;
  }
  m.n = wave_sum(n);
  if (m.n == 0) return m;
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t ol = __shfl_xor(vl, d, 64), oc = __shfl_xor(vc, d, 64);
    const uint32_t oh = (uint32_t)__shfl_xor((int)vh, d, 64);
    const int64_t orr = __shfl_xor((long long)vr, d, 64);
    if (ol == vl && oh == vh) vc += oc;
    else if (vc >= oc) vc -= oc;
    else { vl = ol; vh = oh; vr = orr; vc = oc - vc; }
  }
  const int64_t cr = __shfl((long long)vr, 0, 64);
  if (cr < 0) return m;
  const IndelRec c = C.recs[cr];
  int32_t cls = 0, same = 0;
  for (int64_t i = C.a + lane; i < C.b; i += 64) {
    const IndelRec& e = C.recs[i];
    if (e.key == C.key && e.len == c.len && e.hash == c.hash) {
      cls++;
      if (rec_same(R, e, c)) same++;
    }
  }
  cls = wave_sum(cls);
  same = wave_sum(same);
  if (2 * same > m.n) { m.win = same; m.rec = cr; return m; }
  if (2 * cls > m.n) return col_majority(R, C);                    // collision inside the majority class
  m.win = same;                                                     // no strict majority
  return m;
}

// the region (job) holding batch position g: the last job whose first
// position is <= g, by the whole wave: 64 probes a round
__device__ int32_t wave_job_of(const JobDev* jobs, int32_t n_jobs, int64_t g, int lane) {
  int32_t lo = 0, hi = n_jobs;                          // first job with out > g lies in [lo, hi]
  while (hi - lo > 64) {
    const int64_t m = hi - lo;
    const int32_t probe = lo + (int32_t)(((int64_t)(lane + 1) * m) / 65);
    const int k = __popcll(__ballot(jobs[probe].out <= g));
    const int32_t plo = lo + (int32_t)(((int64_t)k * m) / 65);
    const int32_t phi = lo + (int32_t)(((int64_t)(k + 1) * m) / 65);
    if (k > 0) lo = plo + 1;
    if (k < 64) hi = phi;
  }
  const int32_t i = lo + lane;
  return lo + __popcll(__ballot(i < hi && jobs[i].out <= g)) - 1;
}

}  // namespace

namespace {

// Place in the defer list of column g, or -1 when the window kernel did not
// defer it: a bit per position and the place of each 64 positions' first take
// 0.2 bytes a position where an index of its own would take four.
__device__ __forceinline__ int64_t defer_place(const EngineArgs& A, const JobDev& J, int64_t g) {
  const int32_t w = J.win0 + (int32_t)((g - J.out) / A.W), p = (int32_t)((g - J.out) % A.W);
  const int64_t word = (int64_t)w * (A.W >> 6) + (p >> 6);
  const uint64_t m = A.dmask[word], bit = 1ull << (p & 63);
  if (!(m & bit)) return -1;
  const uint32_t k = A.dbase[word] + (uint32_t)__popcll(m & (bit - 1ull));
  return k < A.defer_cap ? (int64_t)k : -1;
}

// The winning record of a column the deletion pass changed: in the deferred
// column's place, or else a mark on the record.
__device__ __forceinline__ void put_record(const EngineArgs& A, const JobDev& J, int64_t g, int64_t rec) {
  const int64_t k = defer_place(A, J, g);
  if (k >= 0) A.drec[k] = (int32_t)rec;
  else if (rec >= 0) A.rec[rec].flags |= PL_REC_WINS;
}

// The winning record of column g, called with an insertion or a deletion (key
// kind 0 or 1); -1: none.
__device__ __forceinline__ int64_t col_record(const EngineArgs& A, const JobDev& J, int64_t g, uint32_t kind) {
  const int64_t k = defer_place(A, J, g);
  if (k >= 0) return A.drec[k];
  const int32_t w = J.win0 + (int32_t)((g - J.out) / A.W);
  const ColRecs C = col_recs(A.rec, A.rec_cap, A.win_rec, w, *A.spill_n, A.spill_cap, ((uint32_t)g << 1) | kind);
  for (int64_t i = C.a; i < C.b; i++)
    if (C.recs[i].key == C.key && (C.recs[i].flags & PL_REC_WINS)) return i;
  return -1;
}

}  // namespace

// One wave per listed column: the full BaseCall with the column's evidence
// records (hetIndelCall), lane 0 writing the results.
// mode 0: deferred columns (writes call, marks candidates, counts confirmed)
// mode 1: columns changed by the deletion pass (keeps disposition bits)
// Both leave the column's winning record where col_record finds it.
__device__ void indel_columns(const EngineArgs& A, const uint32_t* list, uint32_t n, int mode, uint32_t first,
                              uint32_t nw) {
  const int lane = threadIdx.x & 63;
  for (uint32_t i = first; i < n; i += nw) {
    const uint32_t g = list[i];
    const int32_t j = wave_job_of(A.jobs, A.n_jobs, g, lane);
    const JobDev& J = A.jobs[j];
    const RSDev& R = A.rs[J.rs];
    const int32_t w = J.win0 + (int32_t)((g - J.out) / A.W);
    Col c = load_col(A.pile, A.G, g);
    const uint16_t wflag = A.calls[g].flags & PL_CF_WIDE;
    if (wflag) wide_patch(c, A.wide, A.wide_cap, A.win_wide, J, A.W, g);
    const uint8_t refb = R.ref[J.start + (int64_t)(g - J.out) - 1];
    const BaseFacts bf = base_facts(c);
    int32_t pct = 0;
    const int need = indel_kind_needed(c, A.cf, &pct);
    int indel = 0;
    bool homo = true;
    int64_t wrec = -1;
    if (need) {
      const ColRecs C = col_recs(A.rec, A.rec_cap, A.win_rec, w, *A.spill_n, A.spill_cap, (g << 1) | (uint32_t)(need - 1));
      const Majority mj = wave_majority(R, C, lane);
      if (mj.rec >= 0) {
        const IndelRec& e = A.rec[mj.rec];
        const int d = het_indel_decide(mj.n, mj.win, e.len, (e.flags & 2u) != 0, pct, A.cf);
        if (d) { indel = need; homo = d == 2; wrec = mj.rec; }
      }
    }
    if (lane != 0) continue;
    pl_call cl = make_call(bf, indel, homo, refb, A.cf);
    cl.flags |= wflag;
    if (mode == 0) {
      A.drec[i] = (int32_t)wrec;
      const int32_t p = (int32_t)((g - J.out) % A.W);
      const int64_t word = (int64_t)w * (A.W >> 6) + (p >> 6);
      atomicOr((unsigned long long*)&A.dmask[word], 1ull << (p & 63));
      if (i == 0 || list[i - 1] >= g || list[i - 1] < g - (uint32_t)(p & 63)) A.dbase[word] = i;   // its word's first
      A.calls[g] = cl;
      const int d = call_disp(cl);
      const int64_t dep = c.depth();
      if (d == PL_D_CONFIRMED) atomicAdd(&A.hist[(int64_t)j * PL_HIST + (dep > 255 ? 255 : (dep < 0 ? 0 : dep))], 1u);
      else if (d != PL_D_NONE) atomicOr((unsigned long long*)&A.cmask[word], 1ull << (p & 63));
    } else {
      put_record(A, J, g, wrec);
      pl_call& o = A.calls[g];
      o.base = cl.base; o.alt = cl.alt; o.q = cl.q;
      o.flags = (uint16_t)((cl.flags & ~PL_CF_DISP_MASK) | (o.flags & PL_CF_DISP_MASK) | PL_CF_DELETED);
    }
  }
}

__global__ void __launch_bounds__(256) k_indel_pass(EngineArgs A) {
  const uint32_t n = *A.defer_n < A.defer_cap ? *A.defer_n : A.defer_cap;
  indel_columns(A, A.defer, n, 0, (blockIdx.x * blockDim.x + threadIdx.x) >> 6, (gridDim.x * blockDim.x) >> 6);
}

// ------------------------------------------------------------------ candidates
// The change candidates in position order, from the windows' candidate
// masks: windows follow each other in position order, so a candidate's place
// is the number of mask bits before its own.  A block takes PL_CAND_WORDS
// mask words; k_cand_sums gives each block's bits (launched when there is
// more than one block), k_cand_list adds those of the blocks before it.  The
// masks are an eighth of a byte per position, so both passes cost their
// launch; sorting a candidate list took 17 launches.
#define PL_CAND_WORDS 2048
#define PL_CAND_PER (PL_CAND_WORDS / 256)
__global__ void __launch_bounds__(256) k_cand_sums(EngineArgs A, int64_t n_words, uint32_t* sums) {
  const int64_t x0 = (int64_t)blockIdx.x * PL_CAND_WORDS + threadIdx.x;
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < PL_CAND_PER; k++) {
    const int64_t x = x0 + 256 * k;
    if (x < n_words) n += (uint32_t)__popcll(A.cmask[x]);
  }
  n = wave_sum(n);
  __shared__ uint32_t ws[4];
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ void __launch_bounds__(256) k_cand_list(EngineArgs A, int64_t n_words, const uint32_t* sums) {
  __shared__ uint32_t ws[4], wp[4];
  const int tid = threadIdx.x;
  const int32_t MW = A.W >> 6;
  uint32_t pre = 0;
  for (int64_t b = tid; b < (int64_t)blockIdx.x; b += 256) pre += sums[b];
  pre = wave_sum(pre);
  if ((tid & 63) == 0) wp[tid >> 6] = pre;
  const int64_t x0 = (int64_t)blockIdx.x * PL_CAND_WORDS + (int64_t)tid * PL_CAND_PER;
  uint64_t m[PL_CAND_PER];
  uint32_t n = 0;
#pragma unroll
  for (int k = 0; k < PL_CAND_PER; k++) {
    m[k] = x0 + k < n_words ? A.cmask[x0 + k] : 0ull;
    n += (uint32_t)__popcll(m[k]);
  }
  const uint32_t inc = wave_scan_dpp(n);
  if ((tid & 63) == 63) ws[tid >> 6] = inc;
  __syncthreads();
  uint32_t at = wp[0] + wp[1] + wp[2] + wp[3] + inc - n;
  for (int w = 0; w < (tid >> 6); w++) at += ws[w];
#pragma unroll
  for (int k = 0; k < PL_CAND_PER; k++) {
    const int64_t x = x0 + k;
    if (x >= n_words) break;
    const int32_t wi = (int32_t)(x / MW), word = (int32_t)(x - (int64_t)wi * MW);
    const bool edge = word == 0 || word == MW - 1;
    if (!m[k] && !edge) continue;
    const WinDev win = A.wins[wi];
    const JobDev& J = A.jobs[win.job];
    if (word == 0 && win.p0 == 0) A.st[win.job].cand_lo = (int32_t)at;
    const uint64_t dm = m[k] ? A.dmask[x] : 0ull;              // an insertion or deletion was deferred
    const uint32_t db = dm ? A.dbase[x] : 0u;
    for (uint64_t b = m[k]; b; b &= b - 1) {
      const int64_t g = J.out + win.p0 + 64 * word + (__ffsll((unsigned long long)b) - 1);
      if (at < A.cand_cap) {
        const pl_call cl = A.calls[g];
        int64_t dep = 0;
        for (int f = 0; f < 4; f++) dep += (int64_t)(uint32_t)A.pile[(int64_t)(PL_F_COUNT_A + f) * A.G + g];
        dep += A.pile[(int64_t)PL_F_DELETIONS * A.G + g];
        Cand c;
        c.gpos = (uint32_t)g;
        c.depth = (int32_t)dep;
        c.kind = call_disp(cl);
        c.len = 0;
        c.rec = -1;
        if (c.kind == PL_D_INS || c.kind == PL_D_DEL) {
          c.rec = A.drec[db + (uint32_t)__popcll(dm & ((b & (0ull - b)) - 1ull))];
          c.len = A.rec[c.rec].len;
        }
        c.base = cl.base;
        c.alt = cl.alt;
        c.pad = 0;
        A.cand[at] = c;
      } else {
        *A.overflow = 1;
      }
      at++;
    }
    if (word == MW - 1 && win.p1 == J.size) A.st[win.job].cand_hi = (int32_t)at;
    if (x == n_words - 1) *A.cand_n = at;
  }
}

// ------------------------------------------------------------------ Pass 1
// GenomeRegion.postProcess Pass 1 (GenomeRegion.scala:221-272) for one
// region per wave.  Only deletion calls carry state along the scan (a
// called deletion suppresses the candidates under it), so: the region's
// deletion candidates are scanned in order to find the active ones (few);
// every candidate is then cleared at once if too shallow or under an active
// deletion; each active deletion's positions are then mutated by the lanes.
// Same result as finalize_job, which a region with more than PL_FIN_DELS
// active deletions runs serially.
__global__ void __launch_bounds__(64) k_finalize(EngineArgs A) {
  __shared__ int64_t s_dg[PL_FIN_DELS];
  __shared__ int32_t s_dl[PL_FIN_DELS];
  const int32_t j = blockIdx.x;
  if (j >= A.n_jobs) return;
  const int lane = threadIdx.x;
  const JobDev& J = A.jobs[j];
  JobStat& st = A.st[j];
  const uint32_t* hist = A.hist + (int64_t)j * PL_HIST;
  Cand* cand = A.cand;
  const int64_t a = st.cand_lo;
  const int64_t b = st.cand_hi < (int64_t)A.cand_cap ? st.cand_hi : (int64_t)A.cand_cap;
  const int32_t md = min_depth_of(A.cf, st.base_count, J.size);
  const bool none = st.read_count == 0;
  // active deletions, in order
  int nd = 0;
  int64_t delEnd = -1;
  bool serial = false;
  for (int64_t c0 = a; c0 < b && !serial; c0 += 64) {
    const int64_t k = c0 + lane;
    const bool isd = k < b && !none && cand[k].kind == PL_D_DEL && cand[k].depth >= md;
    for (uint64_t m = __ballot(isd); m; m &= m - 1) {
      const int l = __ffsll((unsigned long long)m) - 1;
      const int64_t g = (int64_t)cand[c0 + l].gpos;
      const int32_t len = cand[c0 + l].len;
      if (g <= delEnd) continue;
      if (nd == PL_FIN_DELS) { serial = true; break; }
      if (lane == 0) { s_dg[nd] = g; s_dl[nd] = len; }
      nd++;
      delEnd = g + len - 1;
    }
  }
  __syncthreads();
  if (serial) {
    if (lane == 0)
      finalize_job(A.cf, J, st, hist, A.pile, A.G, A.calls, cand, a, b, A.mutated, A.mutated_n, A.mutated_cap,
                   A.overflow);
    return;
  }
  // every candidate at once: shallow, or under an active deletion (not its own)
  for (int64_t c0 = a; c0 < b; c0 += 64) {
    const int64_t k = c0 + lane;
    if (k >= b) continue;
    const int64_t g = (int64_t)cand[k].gpos;
    int lo = 0, hi = nd;                                  // active deletions starting before g
    while (lo < hi) { const int mid = (lo + hi) >> 1; if (s_dg[mid] < g) lo = mid + 1; else hi = mid; }
    const bool shadowed = lo > 0 && g <= s_dg[lo - 1] + s_dl[lo - 1] - 1;
    if (none || shadowed || cand[k].depth < md) cand[k].kind = 0;
  }
  // the active deletions: deleted positions take the deletion count (Pass 1
  // mutation, GenomeRegion.scala:262-264), confirmed positions under them leave the count
  int64_t dropped = 0;
  for (int i = 0; i < nd; i++) {
    const int64_t g = s_dg[i];
    const int32_t len = s_dl[i];
    const int32_t dcount = A.pile[(int64_t)PL_F_DELETIONS * A.G + g];
    for (int32_t q = 1 + lane; q < len; q += 64) {
      const int64_t gj = g + q;
      int64_t dep = 0;
      for (int bb = 0; bb < 4; bb++) dep += (int64_t)(uint32_t)A.pile[(int64_t)(PL_F_COUNT_A + bb) * A.G + gj];
      dep += A.pile[(int64_t)PL_F_DELETIONS * A.G + gj];
      if (call_disp(A.calls[gj]) == PL_D_CONFIRMED && dep >= md) dropped++;
      A.pile[(int64_t)PL_F_DELETIONS * A.G + gj] = j_add(A.pile[(int64_t)PL_F_DELETIONS * A.G + gj], dcount);
      A.calls[gj].flags |= PL_CF_DELETED;
      const uint32_t slot = atomicAdd(A.mutated_n, 1u);
      if (slot < A.mutated_cap) A.mutated[slot] = (uint32_t)gj;
      else *A.overflow = 1;
    }
  }
  dropped = wave_sum(dropped);
  int64_t nconf = 0;     // minDepth above the histogram: counted by k_after
  if (md <= PL_CONF_HIST_MAX) for (int d = md + lane; d < PL_HIST; d += 64) nconf += hist[d];
  nconf = wave_sum(nconf);
  if (lane == 0) {
    st.min_depth = md;
    if (md > PL_CONF_HIST_MAX && st.read_count != 0) atomicOr(A.deep, 1u);
    if (nconf > 0) nconf = nconf - dropped > 0 ? nconf - dropped : 0;   // the serial scan stops decrementing at 0
    st.n_confirmed = (int32_t)nconf;
  }
}

// After the deletion pass: the first PL_AFTER_BLOCKS blocks call the columns
// it changed again and spell the insertions, the rest give the exact confirmed count of the regions
// whose minDepth lies above the depth histogram (a --mindepth of 256 or more,
// or a region averaging more than about 2,555x), whose every position is
// tested.  The two write different things of a position and the count looks
// at no deleted one, so one launch does both; it is short when no region
// needs the count and no deletion was called.
#define PL_AFTER_BLOCKS 256
__global__ void __launch_bounds__(256) k_after(EngineArgs A) {
  __shared__ uint32_t s_n;
  if (blockIdx.x < PL_AFTER_BLOCKS) {
    const uint32_t n = *A.mutated_n < A.mutated_cap ? *A.mutated_n : A.mutated_cap;
    indel_columns(A, A.mutated, n, 1, (blockIdx.x * blockDim.x + threadIdx.x) >> 6, (PL_AFTER_BLOCKS * blockDim.x) >> 6);
    // the strings of the insertions that became changes
    const uint32_t nc = *A.cand_n < A.cand_cap ? *A.cand_n : A.cand_cap;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < nc; k += PL_AFTER_BLOCKS * blockDim.x) {
      Cand& c = A.cand[k];
      if (c.kind != PL_D_INS || c.len > PL_CAND_INS) continue;
      const RSDev& R = A.rs[A.jobs[job_of(A.jobs, A.n_jobs, c.gpos)].rs];
      const IndelRec& e = A.rec[c.rec];
      for (int32_t q = 0; q < c.len; q++) c.ins[q] = rec_char(R, e, q);
    }
    return;
  }
  if (*(volatile uint32_t*)A.deep == 0) return;   // no region needs the exact count
  for (int32_t w = (int32_t)blockIdx.x - PL_AFTER_BLOCKS; w < A.n_wins; w += (int32_t)gridDim.x - PL_AFTER_BLOCKS) {
    const WinDev win = A.wins[w];
    JobStat& S = A.st[win.job];
    const int32_t md = S.min_depth;
    if (md <= PL_CONF_HIST_MAX || S.read_count == 0) continue;
    const JobDev& J = A.jobs[win.job];
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    uint32_t n = 0;
    for (int p = win.p0 + threadIdx.x; p < win.p1; p += blockDim.x) {
      const int64_t g = J.out + p;
      int64_t dep = 0;
      for (int b = 0; b < 4; b++) dep += (uint32_t)A.pile[(int64_t)(PL_F_COUNT_A + b) * A.G + g];
      dep += A.pile[(int64_t)PL_F_DELETIONS * A.G + g];
      n += confirmed_final(A.calls[g], dep, md, S.read_count) ? 1u : 0u;
    }
    n = wave_sum(n);
    if ((threadIdx.x & 63) == 0 && n) atomicAdd(&s_n, n);
    __syncthreads();
    if (threadIdx.x == 0 && s_n) atomicAdd(&S.n_confirmed, (int32_t)s_n);
    __syncthreads();
  }
}

// ------------------------------------------------------------------ export
// final dispositions of one window's positions (GenomeRegion.scala:255)
__global__ void k_final_flags(EngineArgs A) {
  const WinDev win = A.wins[blockIdx.x];
  const JobDev& J = A.jobs[win.job];
  const JobStat& S = A.st[win.job];
  for (int p = win.p0 + threadIdx.x; p < win.p1; p += blockDim.x) {
    const int64_t g = J.out + p;
    int64_t dep = 0;
    for (int b = 0; b < 4; b++) dep += (uint32_t)A.pile[(int64_t)(PL_F_COUNT_A + b) * A.G + g];
    dep += A.pile[(int64_t)PL_F_DELETIONS * A.G + g];
    uint16_t f = A.calls[g].flags;
    const int cand = (f & PL_CF_DISP_MASK) >> PL_CF_DISP_SHIFT;
    int disp = cand;
    if (S.read_count == 0 || (f & PL_CF_DELETED) || dep < S.min_depth) disp = PL_D_NONE;
    A.calls[g].flags = (uint16_t)((f & ~PL_CF_DISP_MASK) | (disp << PL_CF_DISP_SHIFT));
  }
}

// the insertion strings too long for their candidate, into a byte pool
__global__ void k_ins_strings(EngineArgs A, const Cand* sorted, const int64_t* idx, const int64_t* off, int32_t n, uint8_t* pool) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Cand& c = sorted[idx[i]];
  const IndelRec& e = A.rec[c.rec];
  const int32_t j = job_of(A.jobs, A.n_jobs, c.gpos);
  const RSDev& R = A.rs[A.jobs[j].rs];
  for (int32_t q = 0; q < e.len; q++) pool[off[i] + q] = rec_char(R, e, q);
}

#include "pl_vcf_kernels.hip"
#include "pl_track_kernels.hip"
