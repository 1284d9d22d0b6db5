// Bucket accumulation kernels, the constant-work fold and reduction (templated on the coordinate
// field), shared by kernels_msm.hip (G1) and kernels_msm_g2*.hip (G2), and the layout of an
// accumulation's scratch. The variable-work merges and reduction are in kernels_msm_tail.hip.
// See kernels_msm.hip for the pipeline.
#pragma once
#include <algorithm>
#include <string>

#include "bn254.cuh"
#include "internal.h"

namespace g16 {

inline size_t accum_align_up(size_t x) { return (x + 255) & ~(size_t)255; }

inline uint32_t accum_seg(const MsmPlan& p, size_t point_bytes) {
  return p.seg[point_bytes == 128 ? 0 : 1];
}

template <int = 0>
__global__ void k_clear_cnt(uint32_t* cnt) {
  if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
}
// Segments past its first beyond which a bucket goes to the heavy path's parallel sums, per
// point that merges it (k_tail_merge): a chain of dependent additions runs on few waves. At 32
// the dense buckets of the standalone G2 MSM's narrow top window kept its merge running with
// most SIMDs idle.
static constexpr uint32_t MERGE_SPAN = 8;

__device__ __forceinline__ Fr ld_fr(const uint4* p) {
  uint4 a = p[0], b = p[1];
  return {{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}
__device__ __forceinline__ void st_fr(uint4* p, const Fr& x) {
  p[0] = make_uint4(x.v[0], x.v[1], x.v[2], x.v[3]);
  p[1] = make_uint4(x.v[4], x.v[5], x.v[6], x.v[7]);
}
__device__ __forceinline__ Fq ld_fq(const uint4* p) {
  uint4 a = p[0], b = p[1];
  return {{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}
__device__ __forceinline__ void st_fq(uint4* p, const Fq& x) {
  p[0] = make_uint4(x.v[0], x.v[1], x.v[2], x.v[3]);
  p[1] = make_uint4(x.v[4], x.v[5], x.v[6], x.v[7]);
}

// Field element loads in units of 32 bytes (2 x uint4).
template <class C>
__device__ __forceinline__ void ld_f(Fp<C>& x, const uint4* p) {
  uint4 a = p[0], b = p[1];
  x = {{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}
template <bool INL, class B>
__device__ __forceinline__ void ld_f(Fq2T<INL, B>& x, const uint4* p) {
  ld_f(x.c0, p);
  ld_f(x.c1, p + 2);
}
template <class C>
__device__ __forceinline__ void st_f(uint4* p, const Fp<C>& x) {
  p[0] = make_uint4(x.v[0], x.v[1], x.v[2], x.v[3]);
  p[1] = make_uint4(x.v[4], x.v[5], x.v[6], x.v[7]);
}
template <bool INL, class B>
__device__ __forceinline__ void st_f(uint4* p, const Fq2T<INL, B>& x) {
  st_f(p, x.c0);
  st_f(p + 2, x.c1);
}

template <class F> struct Words { static constexpr int N = sizeof(F) / 16; };  // uint4s per F

template <class F>
__device__ __forceinline__ Aff<F> ld_aff(const uint4* base, uint32_t i) {
  constexpr int W = Words<F>::N;
  const uint4* p = base + (size_t)i * 2 * W;
  Aff<F> a;
  ld_f(a.x, p);
  ld_f(a.y, p + W);
  return a;
}

template <class F>
__device__ __forceinline__ void st_aff(uint4* base, size_t i, const Aff<F>& a) {
  constexpr int W = Words<F>::N;
  uint4* p = base + i * 2 * W;
  st_f(p, a.x);
  st_f(p + W, a.y);
}

template <class F>
__device__ __forceinline__ Xyzz<F> ld_xyzz(const uint4* base, size_t i) {
  constexpr int W = Words<F>::N;
  const uint4* p = base + i * 4 * W;
  Xyzz<F> r;
  ld_f(r.X, p);
  ld_f(r.Y, p + W);
  ld_f(r.ZZ, p + 2 * W);
  ld_f(r.ZZZ, p + 3 * W);
  return r;
}

template <class F>
__device__ __forceinline__ void st_xyzz(uint4* base, size_t i, const Xyzz<F>& r) {
  constexpr int W = Words<F>::N;
  uint4* p = base + i * 4 * W;
  st_f(p, r.X);
  st_f(p + W, r.Y);
  st_f(p + 2 * W, r.ZZ);
  st_f(p + 3 * W, r.ZZZ);
}

// How the constant-work kernels see a point: (X : Y : Z) with the complete formulas (POps in
// words; COps below runs them on limbs), stored in an XYZZ-sized slot as (X, Y, Z, 0).
template <class F>
struct POps {
  using P = Proj<F>;
  static __device__ __forceinline__ P inf() { return proj_inf<F>(); }
  static __device__ __forceinline__ P add(const P& a, const P& b) { return proj_add(a, b); }
  static __device__ __forceinline__ P load(const uint4* base, size_t i) {
    const Xyzz<F> x = ld_xyzz<F>(base, i);
    return {x.X, x.Y, x.ZZ};
  }
  static __device__ __forceinline__ void store(uint4* base, size_t i, const P& p) {
    st_xyzz(base, i, Xyzz<F>{p.X, p.Y, p.Z, f_zero<F>()});
  }
  static __device__ __forceinline__ P sel(bool c, const P& a, const P& b) { return proj_sel(c, a, b); }
  static __device__ __forceinline__ P add_aff(const P& p, const Aff<F>& a) { return proj_add_aff(p, a); }
};

// The constant-work kernels' arithmetic: the complete formulas on 29-bit limbs (P1L for G1, P2L
// for G2; POps for any other field), loaded from and stored to the same (X, Y, Z, 0) slots
// (words below 2q).
template <class F>
struct COps : POps<F> {};
template <>
struct COps<Fm2i> {
  using P = P2L;
  static __device__ __forceinline__ P inf() { return p2l_inf(); }
  static __device__ __forceinline__ P add(const P& a, const P& b) { return p2l_add(a, b); }
  static __device__ __forceinline__ P load(const uint4* base, size_t i) {
    return p2l_from(POps<Fm2i>::load(base, i));
  }
  static __device__ __forceinline__ void store(uint4* base, size_t i, const P& p) {
    POps<Fm2i>::store(base, i, p2l_out(p));
  }
  static __device__ __forceinline__ P sel(bool c, const P& a, const P& b) { return p2l_sel(c, a, b); }
  static __device__ __forceinline__ P add_aff(const P& p, const Aff<Fm2i>& a) {
    F2L x, y;
    f2l_of(a.x, x);
    f2l_of(a.y, y);
    return p2l_add_aff(p, x, y);
  }
};
template <>
struct COps<Fm> {
  using P = P1L;
  static __device__ __forceinline__ P inf() { return p1l_inf(); }
  static __device__ __forceinline__ P add(const P& a, const P& b) { return p1l_add(a, b); }
  static __device__ __forceinline__ P load(const uint4* base, size_t i) {
    return p1l_from(POps<Fm>::load(base, i));
  }
  static __device__ __forceinline__ void store(uint4* base, size_t i, const P& p) {
    POps<Fm>::store(base, i, p1l_out(p));
  }
  static __device__ __forceinline__ P sel(bool c, const P& a, const P& b) { return p1l_sel(c, a, b); }
  static __device__ __forceinline__ P add_aff(const P& p, const Aff<Fm>& a) {
    uint32_t x[9], y[9];
    limbs29_of(a.x.v, x);
    limbs29_of(a.y.v, y);
    return p1l_add_aff(p, x, y);
  }
};

// Window tables for merged MSMs (msm_window_tables): entry w n + i = 2^(c w) P_i, affine, from
// the previous window's point by c doublings and one inversion; infinity stays (0, 0).
template <class F>
__global__ void __launch_bounds__(128) k_window_tables(uint4* table, size_t n, int c, int W) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Aff<F> P = ld_aff<F>(table, (uint32_t)i);
  for (int w = 1; w < W; ++w) {
    if (!aff_is_inf(P)) {
      Xyzz<F> X = xyzz_dbl_aff(P);
      for (int k = 1; k < c; ++k) X = xyzz_dbl(X);
      P = xyzz_to_aff(X);
    }
    st_aff(table, (size_t)w * n + i, P);
  }
}

// ---------------------------------------------------------------------------------------
// bucket accumulation
// ---------------------------------------------------------------------------------------
// The bucket loop's running sum. Generic: an XYZZ point. G1 (Fm) and G2 (Fm2i): the limb
// forms G1L and G2L, whose mixed additions never leave 29-bit limbs (bn254.cuh); the value and
// every output are the same.
template <class F>
struct Acc {
  using T = Xyzz<F>;
  static __device__ __forceinline__ T inf() { return xyzz_inf<F>(); }
  static __device__ __forceinline__ T madd(const T& p, const Aff<F>& a, bool negate,
                                           const uint4*, uint32_t) {
    return xyzz_add_aff(p, negate ? aff_neg(a) : a);
  }
  static __device__ __forceinline__ Xyzz<F> out(const T& p) { return p; }
};

template <>
struct Acc<Fm> {
  using T = G1L;
  static __device__ __forceinline__ T inf() { return g1l_inf(); }
  static __device__ __forceinline__ T madd(const T& p, const Aff<Fm>& a, bool negate,
                                           const uint4*, uint32_t) {
    return g1l_madd(p, a, negate);
  }
  static __device__ __forceinline__ Xyzz<Fm> out(const T& p) { return g1l_pack(p); }
};

template <>
struct Acc<Fm2i> {
  using T = G2L;
  static __device__ __forceinline__ T inf() { return g2l_inf(); }
  // The doubling case reloads the base (entry i of `bases`) instead of keeping it live.
  static __device__ __forceinline__ T madd(const T& p, const Aff<Fm2i>& a, bool negate,
                                           const uint4* bases, uint32_t i) {
    if (aff_is_inf(a)) return p;
    if (f2l_zero(p.ZZ)) return g2l_from_aff(a, negate);
    G2L r;
    const int k = g2l_madd_core(p, a, negate, r);
    if (k == 1) {
      const Aff<Fm2i> b = ld_aff<Fm2i>(bases, i);
      return g2l_from(xyzz_dbl_aff(negate ? aff_neg(b) : b));
    }
    if (k == 2) return g2l_inf();
    return r;
  }
  static __device__ __forceinline__ Xyzz<Fm2i> out(const T& p) { return g2l_pack(p); }
};

// Segment t of the sorted entries: its runs added into XYZZ accumulators, a run whole inside
// the segment stored as its bucket, the end pieces to pfirst / plast.
template <class F>
__device__ __forceinline__ void accumulate_segment(size_t t, const uint2* __restrict__ ent,
                                                   const uint32_t* total, size_t nseg,
                                                   uint32_t seg,
                                                   const uint4* __restrict__ bases,
                                                   uint4* buckets, uint4* pfirst, uint4* plast) {
  if (t >= nseg) return;
  uint32_t T = total[0];
  size_t b = t * seg;
  if (b >= T) return;
  size_t e = b + seg < T ? b + seg : T;
  uint32_t cur = ent[b].x;
  bool starts = (b == 0) || ent[b - 1].x != cur;
  size_t rs = b;
  using A = Acc<F>;
  typename A::T acc = A::inf();
  // The next entry's point is loaded before this one is added, so the load latency of a
  // random base hides behind a mixed addition.
  uint32_t v = ent[b].y;
  Aff<F> a = ld_aff<F>(bases, v >> 1);  // merged: v >> 1 = w n + i, a window-table entry
  for (size_t k = b; k < e; ++k) {
    uint32_t key = ent[k].x;
    if (key != cur) {
      // Run [rs, k) of bucket `cur` ends inside the segment.
      if (starts) st_xyzz(buckets, cur, A::out(acc));
      else st_xyzz(pfirst, t, A::out(acc));  // rs == b: the run began in an earlier segment
      acc = A::inf();
      cur = key;
      starts = true;
      rs = k;
    }
    uint32_t v_next = 0;
    Aff<F> a_next;
    if (k + 1 < e) {
      v_next = ent[k + 1].y;
      a_next = ld_aff<F>(bases, v_next >> 1);
    }
    acc = A::madd(acc, a, v & 1, bases, v >> 1);
    v = v_next;
    a = a_next;
  }
  bool ends = (e == T) || ent[e].x != cur;
  const Xyzz<F> sum = A::out(acc);
  if (starts && ends) {
    st_xyzz(buckets, cur, sum);
  } else {
    if (rs == b) st_xyzz(pfirst, t, sum);
    st_xyzz(plast, t, sum);
  }
}

// The accumulations one launch works on: MSMs over the same or other sorted entries, each with
// its bases and its scratch.
static constexpr int QUEUE_JOBS = TAIL_JOBS;

struct AccQueueJob {
  const uint2* ent;
  const uint32_t* total;
  const uint4* bases;
  uint4 *buckets, *pfirst, *plast;
  uint32_t* cnt;  // heavy buckets and tasks, cleared here for the merges that follow
  uint64_t nseg;
  uint32_t seg;
};

struct AccQueue {
  AccQueueJob job[QUEUE_JOBS];
  uint32_t start[QUEUE_JOBS + 1];
  int n;
};

// The jobs' accumulation with each segment's sum spread over lanes (kernels_msm_tail.hip).
void accumulate_quad_jobs(int group, const AccQueue& q, uint64_t nseg, hipStream_t s);

// One launch over jobs of the same segment count (blockIdx.y picks the job).
template <class F>
__global__ void __launch_bounds__(128) k_accumulate(const AccQueue q) {
  const AccQueueJob& j = q.job[blockIdx.y];
  if (blockIdx.x == 0 && threadIdx.x < 4) j.cnt[threadIdx.x] = 0;
  accumulate_segment<F>((size_t)blockIdx.x * blockDim.x + threadIdx.x, j.ent, j.total, j.nseg,
                        j.seg, j.bases, j.buckets, j.pfirst, j.plast);
}

// ---------------------------------------------------------------------------------------
// Constant work (opt in; crates/cuda/src/msm.rs:143-164): every (scalar, window) has an entry
// (a zero digit's is flagged discard), and from the accumulation to the reduction no decision
// is a branch on the data: points are (X : Y : Z) added by the complete formulas (bn254.cuh),
// loops run a count the plan fixes, and what the data decide is picked by selects after the
// work is done. What the data still decide is where stores land (a bucket's address), as
// with the counting sort before it. Not constant time.
//
// Accumulation: thread t runs exactly `seg` iterations over segment t (a short last segment
// repeats its last entry, added and dropped). Every iteration stores the running sum once:
// to its bucket when a run that began inside the segment ends, to slot 2t (head) when the
// segment's first run ends, else to slot 2t + 1 (tail), which the end overwrites with the
// last run. Slot rows hold the bucket key, or FOLD_NONE.
// ---------------------------------------------------------------------------------------
static constexpr uint32_t FOLD_NONE = 0xFFFFFFFFu;
// Slots a fold thread walks. A group emits at most two slots (its first and last run), so a
// level shrinks the slot count only for FOLD_LEN > 2; 8 measured best (G1 MSM 2^20 3.08 ms,
// G2 2^18 4.30 ms, against 3.13 / 4.38 at 4 and 3.19 / 4.59 at 16).
static constexpr uint32_t FOLD_LEN = 8;
static_assert(FOLD_LEN > 2, "each fold level must shrink the slot count");

// One launch serves up to TAIL_JOBS MSMs over one plan's entries (blockIdx.y).
struct ConstJob {
  const uint4* bases;
  uint4 *buckets, *fold[2];
  uint32_t* rows[2];
};
struct ConstJobs {
  ConstJob job[TAIL_JOBS];
};

template <class F>
__global__ void __launch_bounds__(128) k_accumulate_const(const uint2* __restrict__ ent,
                                                          const uint32_t* total, size_t nseg,
                                                          uint32_t seg, const ConstJobs jobs) {
  using O = COps<F>;
  const uint4* __restrict__ bases = jobs.job[blockIdx.y].bases;
  uint4 *buckets = jobs.job[blockIdx.y].buckets, *slots = jobs.job[blockIdx.y].fold[0];
  uint32_t* rows = jobs.job[blockIdx.y].rows[0];
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nseg) return;
  const size_t b = t * seg, T = total[0];  // the plan's entry count: b < T for t < nseg
  if (b >= T) {  // not reached on a full entry list; keeps every read inside it regardless
    rows[2 * t] = FOLD_NONE;
    rows[2 * t + 1] = FOLD_NONE;
    return;
  }
  const uint32_t len = (uint32_t)(b + seg < T ? seg : T - b);
  uint32_t cur = ent[b].x;
  bool first = true;
  const typename O::P inf = O::inf();
  typename O::P acc = inf;
  for (uint32_t i = 0; i < seg; ++i) {
    const bool live = i < len;
    const uint2 e = ent[b + (live ? i : len - 1)];
    const uint32_t key = live ? e.x : cur;
    const bool boundary = key != cur;
    const bool to_bucket = boundary && !first;
    const size_t slot = 2 * t + ((boundary && first) ? 0 : 1);
    O::store(to_bucket ? buckets : slots, to_bucket ? cur : slot, acc);
    rows[slot] = cur;
    first = first && !boundary;
    acc = O::sel(boundary, inf, acc);
    cur = key;
    Aff<F> a = ld_aff<F>(bases, e.y >> 2);
    const bool keep = !live || (e.y & 2u) || aff_is_inf(a);
    a.y = f_sel((e.y & 1u) != 0, neg(a.y), a.y);
    const typename O::P sum = O::add_aff(acc, a);
    acc = O::sel(keep, acc, sum);
  }
  const size_t slot = 2 * t + (first ? 0 : 1);
  O::store(slots, slot, acc);
  rows[slot] = cur;
  rows[2 * t + 1] = first ? FOLD_NONE : cur;
}

// One level of the fold: thread g walks slots [g FOLD_LEN, (g + 1) FOLD_LEN) of the level's m
// (exactly FOLD_LEN iterations; past m it repeats the last slot as empty), adding runs of equal
// rows. A run that ends inside the group, other than its first, is complete (all of a bucket's
// pieces are consecutive) and goes to its bucket; the group's first and last runs go to slots
// 2g and 2g + 1 of the next level (k_scan_const takes over at ScanSlots::FROM slots).
template <class F>
__global__ void __launch_bounds__(128) k_fold_const(const ConstJobs jobs, int from, uint32_t m) {
  using O = COps<F>;
  const ConstJob& job = jobs.job[blockIdx.y];
  const uint4* in = job.fold[from];
  const uint32_t* in_rows = job.rows[from];
  uint4 *out = job.fold[1 - from], *buckets = job.buckets;
  uint32_t* out_rows = job.rows[1 - from];
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t groups = (m + FOLD_LEN - 1) / FOLD_LEN;
  if (g >= groups) return;
  const uint32_t lo = g * FOLD_LEN, hi = lo + FOLD_LEN < m ? lo + FOLD_LEN : m;
  uint32_t cur = FOLD_NONE;
  bool first = true;
  const typename O::P inf = O::inf();
  typename O::P acc = inf;
  for (uint32_t i = lo; i < lo + FOLD_LEN; ++i) {
    const bool live = i < hi;
    const uint32_t j = live ? i : hi - 1;
    const uint32_t r = live ? in_rows[j] : FOLD_NONE;
    const bool empty = r == FOLD_NONE;
    const bool boundary = !empty && r != cur;
    const bool finished = boundary && cur != FOLD_NONE;
    const bool to_head = finished && first;
    const bool to_bucket = finished && !to_head;
    const size_t slot = 2 * (size_t)g + (to_head ? 0 : 1);
    O::store(to_bucket ? buckets : out, to_bucket ? cur : slot, acc);
    out_rows[slot] = cur;
    first = first && !finished;
    acc = O::sel(boundary, inf, acc);
    cur = boundary ? r : cur;
    const typename O::P q = O::sel(empty, inf, O::load(in, j));
    acc = O::add(acc, q);
  }
  const bool has_run = cur != FOLD_NONE;
  const size_t slot = 2 * (size_t)g + (first ? 0 : 1);
  O::store(out, slot, acc);
  out_rows[slot] = has_run ? cur : FOLD_NONE;
  out_rows[2 * (size_t)g + 1] = (has_run && !first) ? cur : FOLD_NONE;
}

// The fold's end: a workgroup per BLOCK slots, a slot per thread. The non-empty slots are packed
// to the front in order (their rows stay sorted, so each bucket's pieces are adjacent), then a
// segmented inclusive scan in LDS runs one addition per level for every thread: at distance d a
// thread adds the value d slots back where that slot has its row (the slots between belong to
// the same run) and keeps its own otherwise. The last slot of a run then holds the run's sum and
// stores it to its bucket; with several workgroups a workgroup's first and last runs go to
// slots 2b and 2b + 1 of the next level instead, as a fold group's do. A level of 512 slots to 2
// is 9 additions deep, where fold levels are 8 deep for a factor of 4, at 9 times their work; so
// folds run down to FROM slots (G1 131072, G2 32768: a level there is about as long on the device
// as it is deep). The level count depends on m only. Other lines, MI355X: G1 at 65536, MSM of 2^15
// 688 us for 658 and 2^18 1154 for 1127; at 262144, the 100k-constraint prove 3.61 ms for 3.35. G2
// at 16384, MSM of 2^15 1381 us for 1265 and 2^18 3727 for 3593; at 65536, 2^14 1111 for 1209, 2^16
// 1783 for 1888, and the 131k prove 4.27 ms for 4.39, with 300k and 450k within 0.4 %: the better
// line for G2 lies between.
// BLOCK: slots per scan, as many threads as the point form's registers allow in one workgroup.
template <class F>
struct ScanSlots {
  static constexpr bool G2 = sizeof(typename COps<F>::P) > 128;
  static constexpr uint32_t N = G2 ? 256 : 512;
  static constexpr uint32_t FROM = G2 ? 32768 : 131072;
};

template <class F, uint32_t BLOCK>
__global__ void __launch_bounds__(BLOCK) k_scan_const(const ConstJobs jobs, int from,
                                                      uint32_t count) {
  const ConstJob& job = jobs.job[blockIdx.y];
  const size_t at = (size_t)blockIdx.x * BLOCK;  // below count
  const uint4* in = job.fold[from] + at * Words<F>::N * 4;
  const uint32_t* in_rows = job.rows[from] + at;
  uint4* buckets = job.buckets;
  const uint32_t m = count - at < BLOCK ? (uint32_t)(count - at) : BLOCK;
  const bool last_level = gridDim.x == 1;
  using O = COps<F>;
  using P = typename O::P;
  __shared__ P sh[BLOCK];
  __shared__ uint32_t rows[BLOCK];
  __shared__ uint32_t wave_count[BLOCK / 64];
  const uint32_t i = threadIdx.x, lane = i & 63u, wave = i >> 6;
  const bool live = i < m;
  const uint32_t j = live ? i : m - 1;  // m >= 1
  uint32_t r = live ? in_rows[j] : FOLD_NONE;
  const bool has = r != FOLD_NONE;
  P v = O::sel(has, O::load(in, j), O::inf());
  // Pack: position = non-empty slots before this one.
  const uint64_t ball = __ballot(has);
  const uint32_t before = (uint32_t)__popcll(ball & ((1ull << lane) - 1ull));
  if (lane == 0) wave_count[wave] = (uint32_t)__popcll(ball);
  __syncthreads();
  uint32_t pos = before, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < BLOCK / 64; ++w) {
    pos += w < wave ? wave_count[w] : 0u;
    total += wave_count[w];
  }
  if (has) {
    sh[pos] = v;
    rows[pos] = r;
  }
  if (i >= total) {  // positions no slot packs into
    sh[i] = O::inf();
    rows[i] = FOLD_NONE;
  }
  __syncthreads();
  v = sh[i];
  r = rows[i];
  for (uint32_t d = 1; d < m; d <<= 1) {
    __syncthreads();  // every read of the previous level is done
    sh[i] = v;
    __syncthreads();
    const uint32_t k = i >= d ? i - d : i;
    const bool take = i >= d && rows[k] == r;
    const P sum = O::add(sh[k], v);
    v = O::sel(take, sum, v);
  }
  const bool end = r != FOLD_NONE && (i + 1 == BLOCK || rows[i + 1] != r);
  const bool head = !last_level && r == rows[0], tail = !last_level && !head && i + 1 == total;
  const size_t slot = 2 * (size_t)blockIdx.x + (tail ? 1 : 0);
  if (end) O::store(head || tail ? job.fold[1 - from] : buckets, head || tail ? slot : r, v);
  if (!last_level && i < 2) {  // the next level's rows: first run, last run if another
    const uint32_t first = total ? rows[0] : FOLD_NONE, last = total ? rows[total - 1] : FOLD_NONE;
    job.rows[1 - from][2 * (size_t)blockIdx.x + i] =
        i == 0 ? first : (last != first ? last : FOLD_NONE);
  }
}

// Every bucket starts as the identity (a bucket no entry names is never stored).
template <class F>
__global__ void k_fill_proj_inf(const ConstJobs jobs, size_t K) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < K) POps<F>::store(jobs.job[blockIdx.y].buckets, i, POps<F>::inf());
}

// Several MSMs' bucket accumulations as one persistent launch over a device-side work queue:
// the grid is sized to what the device holds at once, and each workgroup takes tiles of 128
// segments from a shared counter until every job's segments are done. Tile t belongs to job
// d with start[d] <= t < start[d + 1]; segments past a job's device-side entry count end at once.
static constexpr uint32_t QUEUE_TILE = 128;  // segments per tile = threads per workgroup

template <class F>
__global__ void __launch_bounds__(QUEUE_TILE) k_accumulate_queue(AccQueue q, uint32_t* counter) {
  __shared__ uint32_t tile;
  const uint32_t tiles = q.start[q.n];
  if (blockIdx.x == 0 && threadIdx.x < 4)
    for (int d = 0; d < q.n; ++d) q.job[d].cnt[threadIdx.x] = 0;
  for (;;) {
    if (threadIdx.x == 0) tile = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t t = tile;
    __syncthreads();  // every lane has read `tile` before lane 0 overwrites it
    if (t >= tiles) return;
    int d = 0;
    while (d + 1 < q.n && t >= q.start[d + 1]) ++d;
    const AccQueueJob& j = q.job[d];
    accumulate_segment<F>((size_t)(t - q.start[d]) * QUEUE_TILE + threadIdx.x, j.ent, j.total,
                          j.nseg, j.seg, j.bases, j.buckets, j.pfirst, j.plast);
  }
}

// Interior segments per heavy-bucket task (kernels_msm_tail.hip).
static constexpr uint32_t HEAVY_TASK = 256;

// ---------------------------------------------------------------------------------------
// window reduction: S_w = sum_j (j+1) B_{w,j}
// ---------------------------------------------------------------------------------------
// The buckets of a window fall in G groups of B = 2^lg. With T_g = sum_i B_{gB+i} and
// U_g = sum_i (i+1) B_{gB+i},
//   S_w = sum_g U_g + B sum_g g T_g = sum_g U_g + sum_k 2^(k+lg) Q_k,
//   Q_k = sum of T_g over the g whose bit k is set.
// Level 1 makes T and U; level 2 is a plain sum per (window, row) — row 0 sums U, row k+1 is
// Q_k. A row's items are cut into S slices (S a power of two that divides every row's count), one
// workgroup each; with S > 1 the slice sums go to a scratch array and each row's S of them are
// added after. Every chain is short; the doublings of the bit weights happen once, in the host's
// pass over all windows (kernels_msm_tail.hip).
// Buckets per group. A group's chain is 2 (B - 1) additions and the rows' trees cost more per
// point than chains do, so many sets of many buckets (a large standalone MSM) take 8: whole G1
// MSM 2^20 1637 -> 1606 us, whole G2 MSM 2^18 1547 -> 1524 (MI355X).
inline uint32_t reduce_group_size(const MsmPlan& p) {
  const uint32_t B = !p.merged && (size_t)p.windows * p.nb >= 65536 ? 8u : 4u;
  return p.nb < B ? p.nb : B;
}
inline int ilog2_u32(uint32_t x) {
  int l = 0;
  while ((2u << l) <= x) ++l;
  return l;
}

// Slices per row of G groups over `sets` bucket sets, a point taking `lanes` lanes (k_tail_rows:
// 256 / lanes points per workgroup). A slice costs its chain of additions and a tree of
// log2(points): with at least two items per point while the device has room (512 workgroups),
// eight beyond.
inline uint32_t tail_slices(uint32_t G, uint32_t sets, uint32_t lanes) {
  const uint32_t rows = 1 + (uint32_t)ilog2_u32(G), points = 256 / lanes;
  uint32_t S = 1;
  for (;;) {
    const uint64_t blocks = (uint64_t)2 * S * rows * sets;
    if (S >= 256 || 2 * S > G / 2 || 2 * S * (blocks <= 512 ? 2 : 8) * points > G) return S;
    S *= 2;
  }
}

// Scratch of one accumulation (one base vector over one sorted entry list): buckets, the
// segment end partials, heavy-bucket bookkeeping, task sums, reduction groups, counters.
struct AccumLayout {
  size_t buckets, pfirst, plast, heavy, tasks, task_sum, gT, gU, cnt;
  size_t fold0, frows0, fold1, frows1;  // constant work: the fold's two levels of slots
  size_t total;
};

// Slots the constant-work fold needs: 2 per segment, then 2 per group of FOLD_LEN.
inline size_t fold_slots0(size_t nseg) { return 2 * nseg; }
inline size_t fold_slots1(size_t nseg) { return 2 * ((2 * nseg + FOLD_LEN - 1) / FOLD_LEN) + 2; }

inline AccumLayout accum_layout(const MsmPlan& p, size_t pt) {
  size_t K = (size_t)msm_bucket_sets(p) * p.nb;
  const uint32_t seg = accum_seg(p, pt);
  size_t nseg = (p.max_entries + seg - 1) / seg;
  size_t max_heavy = nseg / MERGE_SPAN + 2;
  size_t max_tasks = nseg / HEAVY_TASK + max_heavy + 2;
  uint32_t B = reduce_group_size(p);
  size_t G = p.nb / B;
  AccumLayout L;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t r = off;
    off += accum_align_up(bytes);
    return r;
  };
  L.buckets = take(pt * K);
  L.pfirst = take(p.constant ? 0 : pt * (nseg + 1));  // constant work keeps slots instead
  L.plast = take(p.constant ? 0 : pt * (nseg + 1));
  L.heavy = take(12 * max_heavy);
  L.tasks = take(8 * max_tasks);
  L.task_sum = take(pt * max_tasks);
  L.gT = take(pt * G * msm_bucket_sets(p));
  L.gU = take(pt * G * msm_bucket_sets(p));
  L.cnt = take(16);
  L.fold0 = take(p.constant ? pt * fold_slots0(nseg) : 0);
  L.frows0 = take(p.constant ? 4 * fold_slots0(nseg) : 0);
  L.fold1 = take(p.constant ? pt * fold_slots1(nseg) : 0);
  L.frows1 = take(p.constant ? 4 * fold_slots1(nseg) : 0);
  L.total = off;
  return L;
}

inline size_t msm_accum_scratch_bytes_impl(const MsmPlan& p, int group) {
  return accum_layout(p, group == 1 ? 128 : 256).total;
}

// Pointers into one accumulation's scratch.
struct AccumPtrs {
  uint4 *buckets, *pfirst, *plast, *task_sum, *gT, *gU;
  // The reduction's slice sums: S per row, in the place of the segment partials (constant work:
  // the slots), no longer needed by then, so S is cut to what they hold.
  uint4* parts;
  uint32_t S;
  uint32_t *heavy, *tasks, *cnt;
  uint4 *fold0, *fold1;
  uint32_t *frows0, *frows1;
  uint32_t seg;  // entries per segment
  size_t nseg;
};

// Launches the constant-work fold of n jobs over field F. The G1 one is defined here; the G2 one
// (F = Fm2i, products expanded in place so the latency-bound fold does not spill) lives in
// kernels_msm_g2_tail.hip, so the slow G2 kernels compile in parallel translation units.
template <class F>
struct ConstTail {
  static void fold(const ConstJobs& jobs, size_t nseg, int n, hipStream_t s);
};

template <class F>
inline void tail_fold_const(const ConstJobs& jobs, size_t nseg, int n, hipStream_t s) {
  // Fold levels (2 nseg slots, then 2 per group of FOLD_LEN), then scan levels (2 per
  // workgroup), until one workgroup's scan holds the rest.
  constexpr uint32_t SCAN = ScanSlots<F>::N;
  size_t m = fold_slots0(nseg);
  if (m == 0) return;
  int from = 0;
  for (; m > ScanSlots<F>::FROM; from = 1 - from) {
    const size_t groups = (m + FOLD_LEN - 1) / FOLD_LEN;
    hipLaunchKernelGGL(k_fold_const<F>, dim3((unsigned)((groups + 127) / 128), n), dim3(128), 0, s,
                       jobs, from, (uint32_t)m);
    G16_LAUNCH_CHECK("msm fold (constant work)");
    m = 2 * groups;
  }
  for (;; from = 1 - from) {
    const size_t blocks = (m + SCAN - 1) / SCAN;
    hipLaunchKernelGGL((k_scan_const<F, SCAN>), dim3((unsigned)blocks, n), dim3(SCAN), 0, s, jobs,
                       from, (uint32_t)m);
    G16_LAUNCH_CHECK("msm fold scan (constant work)");
    if (blocks == 1) return;
    m = 2 * blocks;
  }
}

// F: the coordinate field in the MSM's Montgomery form R' = 2^261 (Fm, or Fm2i for G2); the
// bases must already be in that form (msm_bases_to_msm_form).
template <class F>
inline AccumPtrs accum_ptrs(const MsmPlan& p, void* scratch) {
  constexpr size_t PT = sizeof(Xyzz<F>);
  AccumLayout L = accum_layout(p, PT);
  char* q = static_cast<char*>(scratch);
  AccumPtrs a;
  a.buckets = reinterpret_cast<uint4*>(q + L.buckets);
  a.pfirst = reinterpret_cast<uint4*>(q + L.pfirst);
  a.plast = reinterpret_cast<uint4*>(q + L.plast);
  a.heavy = reinterpret_cast<uint32_t*>(q + L.heavy);
  a.tasks = reinterpret_cast<uint32_t*>(q + L.tasks);
  a.task_sum = reinterpret_cast<uint4*>(q + L.task_sum);
  a.gT = reinterpret_cast<uint4*>(q + L.gT);
  a.gU = reinterpret_cast<uint4*>(q + L.gU);
  a.cnt = reinterpret_cast<uint32_t*>(q + L.cnt);
  a.fold0 = reinterpret_cast<uint4*>(q + L.fold0);
  a.frows0 = reinterpret_cast<uint32_t*>(q + L.frows0);
  a.fold1 = reinterpret_cast<uint4*>(q + L.fold1);
  a.frows1 = reinterpret_cast<uint32_t*>(q + L.frows1);
  a.seg = accum_seg(p, PT);
  a.nseg = (p.max_entries + a.seg - 1) / a.seg;
  const uint32_t G = p.nb / reduce_group_size(p), sets = (uint32_t)msm_bucket_sets(p);
  const uint64_t rows = (uint64_t)(1 + ilog2_u32(G)) * sets;
  a.S = tail_slices(G, sets, PT == 128 ? 4 : 8);
  a.parts = p.constant ? a.fold0 : a.pfirst;
  while (a.S > 1 && a.S * rows > 2 * a.nseg) a.S /= 2;
  return a;
}

inline TailJob tail_job(const MsmPlan& p, const AccumPtrs& a, void* window_out) {
  TailJob j{};
  j.offset = p.offset;
  j.sets = (uint32_t)msm_bucket_sets(p);
  j.K = j.sets * p.nb;
  j.seg = a.seg;
  j.B = reduce_group_size(p);
  j.G = p.nb / j.B;
  j.rows = 1 + (uint32_t)ilog2_u32(j.G);
  j.S = a.S;
  j.avg_pieces = (uint32_t)(p.max_entries / ((size_t)a.seg * j.K));
  j.buckets = a.buckets;
  j.pfirst = a.pfirst;
  j.plast = a.plast;
  j.task_sum = a.task_sum;
  j.gT = a.gT;
  j.gU = a.gU;
  j.parts = a.parts;
  j.out = static_cast<uint4*>(window_out);
  j.heavy = a.heavy;
  j.tasks = a.tasks;
  j.cnt = a.cnt;
  return j;
}

// The bucket accumulations of up to QUEUE_JOBS variable-work MSMs of one group (each: plan,
// bases, scratch), then their merges and reductions into window_out, all jobs in each launch.
// With `counter` (a device word, cleared here by a kernel first) the accumulation is one
// persistent launch of `grid` workgroups that take tiles of segments from it; without, the jobs
// have the same entries and run side by side.
template <class F>
inline void accumulate_jobs_impl(int group, const MsmPlan* const* plans, const void* const* bases,
                                 void* const* scratch, void* const* window_out, int n,
                                 uint32_t* counter, int grid, hipStream_t s, hipEvent_t* ev) {
  if (n < 1 || n > QUEUE_JOBS) throw ArgError{"accumulation of " + std::to_string(n) + " jobs"};
  AccQueue q{};
  TailJobs t{};
  q.n = t.n = n;
  for (int d = 0; d < n; ++d) {
    if (plans[d]->constant) throw ArgError{"constant-work MSMs accumulate on their own"};
    const AccumPtrs a = accum_ptrs<F>(*plans[d], scratch[d]);
    q.job[d] = AccQueueJob{plans[d]->ent, plans[d]->total, static_cast<const uint4*>(bases[d]),
                           a.buckets, a.pfirst, a.plast, a.cnt, a.nseg, a.seg};
    const size_t tiles = (a.nseg + QUEUE_TILE - 1) / QUEUE_TILE;
    if (q.start[d] + tiles >= (1ull << 32)) throw ArgError{"accumulation queue too long"};
    q.start[d + 1] = q.start[d] + (uint32_t)tiles;
    t.job[d] = tail_job(*plans[d], a, window_out[d]);
  }
  if (ev) G16_CHECK(hipEventRecord(ev[0], s));
  if (counter) {
    hipLaunchKernelGGL(k_clear_cnt<0>, dim3(1), dim3(64), 0, s, counter);
    G16_LAUNCH_CHECK("msm queue counter");
    const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>((size_t)grid, q.start[n]));
    hipLaunchKernelGGL(k_accumulate_queue<F>, dim3(blocks), dim3(QUEUE_TILE), 0, s, q, counter);
  } else {
    uint64_t nseg = 1;  // at least one workgroup: it clears the counters
    for (int d = 0; d < n; ++d) nseg = std::max(nseg, q.job[d].nseg);
    // Segments' sums over 4 (G1) or 8 (G2) lanes each while those lanes take at most two waves
    // per SIMD: there they end sooner than one lane each (G1 MSM of 4099 points 351 -> 324 us,
    // G2 of 1021 points 511 -> 444); at sixteen the device is full and the extra work shows
    // (65k-constraint prove 1.38 -> 1.74 ms).
    const uint64_t lanes = nseg * n * (group == 1 ? 4 : 8);
    if (lanes <= 131072) accumulate_quad_jobs(group, q, nseg, s);
    else hipLaunchKernelGGL(k_accumulate<F>, dim3((unsigned)((nseg + 127) / 128), n), dim3(128), 0, s, q);
  }
  G16_LAUNCH_CHECK("msm accumulate");
  if (ev) G16_CHECK(hipEventRecord(ev[1], s));
  tail_merge_jobs(group, t, s);
  if (ev) G16_CHECK(hipEventRecord(ev[2], s));
  tail_reduce_jobs(group, false, t, s);
  if (ev) G16_CHECK(hipEventRecord(ev[3], s));
}

// Up to TAIL_JOBS constant-work MSMs over one plan's entries, every launch over all of them.
template <class F>
inline void accumulate_const_impl(int group, const MsmPlan& p, const void* const* bases,
                                  void* const* scratch, void* const* window_out, int n,
                                  hipStream_t s, hipEvent_t* ev) {
  if (n < 1 || n > TAIL_JOBS) throw ArgError{"accumulation of " + std::to_string(n) + " jobs"};
  ConstJobs jobs{};
  TailJobs t{};
  t.n = n;
  AccumPtrs a{};
  for (int d = 0; d < n; ++d) {
    a = accum_ptrs<F>(p, scratch[d]);
    jobs.job[d] = ConstJob{static_cast<const uint4*>(bases[d]), a.buckets, {a.fold0, a.fold1},
                           {a.frows0, a.frows1}};
    t.job[d] = tail_job(p, a, window_out[d]);
  }
  const unsigned grid = (unsigned)((a.nseg + 127) / 128);
  const size_t K = (size_t)msm_bucket_sets(p) * p.nb;
  if (ev) G16_CHECK(hipEventRecord(ev[0], s));
  hipLaunchKernelGGL(k_fill_proj_inf<F>, dim3((unsigned)((K + 255) / 256), n), dim3(256), 0, s,
                     jobs, K);
  G16_LAUNCH_CHECK("msm buckets (constant work)");
  if (a.nseg) {
    hipLaunchKernelGGL(k_accumulate_const<F>, dim3(grid, n), dim3(128), 0, s, p.ent, p.total,
                       a.nseg, a.seg, jobs);
    G16_LAUNCH_CHECK("msm accumulate (constant work)");
  }
  if (ev) G16_CHECK(hipEventRecord(ev[1], s));
  ConstTail<F>::fold(jobs, a.nseg, n, s);
  if (ev) G16_CHECK(hipEventRecord(ev[2], s));
  tail_reduce_jobs(group, true, t, s);
  if (ev) G16_CHECK(hipEventRecord(ev[3], s));
}

}  // namespace g16
