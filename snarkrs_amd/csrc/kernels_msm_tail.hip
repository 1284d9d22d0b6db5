// The variable-work MSM's tail on points spread over lanes (msm_quad.cuh): merges of buckets
// that span segments, heavy buckets, window reduction. One launch of each kernel serves up to
// TAIL_JOBS MSMs (blockIdx.y), so that MSMs over the same entries pay each chain of dependent
// additions once, not one after the other.
//
// What bounds these kernels is the length of their chains: a few hundred waves at most, each
// addition waiting for the last. MI355X, one lane per point -> points over lanes, us
// (reduction groups of 4; see reduce_group_size for the last two):
//                                merge       heavy buckets   groups      rows and slices
//   G1, 1000-constraint prove    34 -> 12    40 -> 31        47 -> 20    60 -> 24
//   G2, 1000-constraint prove    91 -> 16    126 -> 46       140 -> 27   156 -> 44
//   G1 MSM 2^20 (17 sets)        90 -> 91    126 -> 54       87 -> 80    187 -> 174
//   G2 MSM 2^18 (20 sets)        136 -> 77   267 -> 76       143 -> 68   252 -> 143
#include "msm_accum.cuh"
#include "msm_quad.cuh"

namespace g16 {

static constexpr int TAIL_BLOCK = 256;

// A heavy bucket (more than `span` segments after its first) is cut into tasks of HEAVY_TASK
// interior segments: heavy[h] = {bucket, first task, task count}, tasks[t] = {first, end
// segment}, cnt = {heavy buckets, tasks}.
__device__ __forceinline__ void register_heavy(const TailJob& j, uint32_t k, uint32_t sa,
                                               uint32_t sb) {
  const uint32_t interior = sb - sa - 1;
  const uint32_t ntask = (interior + HEAVY_TASK - 1) / HEAVY_TASK;
  const uint32_t slot = atomicAdd(&j.cnt[0], 1u);
  const uint32_t tb = atomicAdd(&j.cnt[1], ntask);
  j.heavy[3 * slot] = k;
  j.heavy[3 * slot + 1] = tb;
  j.heavy[3 * slot + 2] = ntask;
  for (uint32_t t = 0; t < ntask; ++t) {
    const uint32_t lo = sa + 1 + t * HEAVY_TASK;
    j.tasks[2 * (tb + t)] = lo;
    j.tasks[2 * (tb + t) + 1] = lo + HEAVY_TASK < sb ? lo + HEAVY_TASK : sb;
  }
}

// The bucket accumulation (accumulate_segment's work, a segment per point) for MSMs whose
// segments fill little of the device at one lane each: an addition is 2-4 us deep instead of 5
// (G1) or 13 (G2), with the slots of 16 products (G1) where a lane's mixed addition takes 10, and
// the moves.
template <bool G2>
__global__ void __launch_bounds__(TAIL_BLOCK) k_accumulate_quad(const AccQueue q) {
  using Q = Quad<G2>;
  const AccQueueJob& j = q.job[blockIdx.y];
  if (blockIdx.x == 0 && threadIdx.x < 4) j.cnt[threadIdx.x] = 0;
  const uint64_t t = (uint64_t)blockIdx.x * (TAIL_BLOCK / Q::LANES) + Q::slot();
  const uint64_t T = j.total[0], b = t * j.seg;
  const bool alive = t < j.nseg && b < T;
  const uint64_t e = !alive ? b : b + j.seg < T ? b + j.seg : T;
  const uint32_t len = (uint32_t)(e - b);
  uint32_t cur = alive ? j.ent[b].x : 0u;
  bool starts = alive && (b == 0 || j.ent[b - 1].x != cur);
  bool first = true;  // the run began at the segment's start
  // Lanes 0 and 1 of a quad read the base's x and y.
  const uint32_t at = (Q::coord() & 1u) * (Q::POINT_WORDS / 4) + Q::comp() * 2;
  const auto fetch = [&](uint32_t i, uint2& en, uint4& lo, uint4& hi) {
    en = j.ent[b + i];
    const uint4* p = j.bases + (size_t)(en.y >> 1) * (Q::POINT_WORDS / 2) + at;
    lo = p[0];
    hi = p[1];
  };
  Coord acc = Q::inf();
  uint2 en = make_uint2(0, 0);
  uint4 lo = make_uint4(0, 0, 0, 0), hi = lo;
  if (len) fetch(0, en, lo, hi);
#pragma unroll 1
  for (uint32_t i = 0; __any(i < len); ++i) {
    const bool live = i < len;
    if (live && en.x != cur) {
      if (starts) Q::store(j.buckets, cur, acc);
      else Q::store(j.pfirst, t, acc);
      acc = Q::inf();
      cur = en.x;
      starts = true;
      first = false;
    }
    const Coord p = Q::from_affine(lo, hi, (en.y & 1u) != 0, live);
    if (i + 1 < len) fetch(i + 1, en, lo, hi);
    acc = Q::add(acc, p);
  }
  if (!alive) return;
  const bool ends = e == T || j.ent[e].x != cur;
  if (starts && ends) {
    Q::store(j.buckets, cur, acc);
  } else {
    if (first) Q::store(j.pfirst, t, acc);
    Q::store(j.plast, t, acc);
  }
}

void accumulate_quad_jobs(int group, const AccQueue& q, uint64_t nseg, hipStream_t s) {
  const auto launch = [&](auto kernel, uint32_t points) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((nseg + points - 1) / points), q.n),
                       dim3(TAIL_BLOCK), 0, s, q);
  };
  if (group == 1) launch(k_accumulate_quad<false>, TAIL_BLOCK / Quad<false>::LANES);
  else launch(k_accumulate_quad<true>, TAIL_BLOCK / Quad<true>::LANES);
  G16_LAUNCH_CHECK("msm accumulate (points over lanes)");
}

// Buckets that span segments, L points each: point i of a bucket adds every L-th of its pieces
// (plast of its first segment, pfirst of the rest), then the L points add up. A bucket past
// MERGE_SPAN pieces per point goes to the heavy path. Empty buckets become infinity; a bucket
// inside one segment was stored whole by the accumulation.
template <bool G2, uint32_t L>
__global__ void __launch_bounds__(TAIL_BLOCK) k_tail_merge(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  constexpr uint32_t BUCKETS = TAIL_BLOCK / Q::LANES / L;
  if (blockIdx.x * BUCKETS >= j.K) return;
  const uint32_t k = blockIdx.x * BUCKETS + Q::slot() / L, sub = Q::slot() % L;
  uint32_t t = 1, sb = 0, sa = 0;  // an empty chain
  bool store = false;
  if (k < j.K) {
    const uint32_t s = j.offset[k], e = j.offset[k + 1];
    if (s == e) {
      store = true;  // of infinity
    } else {
      const uint32_t a = s / j.seg, b = (e - 1) / j.seg;
      if (b - a >= MERGE_SPAN * L) {
        if (sub == 0 && Q::leader()) register_heavy(j, k, a, b);
      } else if (a != b) {
        store = true;
        sa = a;
        sb = b;
        t = a + sub;
      }
    }
  }
  const auto piece = [&](uint32_t i) { return Q::load(i == sa ? j.plast : j.pfirst, i); };
  Coord acc = Q::inf(), b = Q::inf();
  if (t <= sb) acc = piece(t);
  t += L;
  uint32_t off = L / 2;
  bool chain = true;
#pragma unroll 1
  for (;;) {
    if (chain && __any(t <= sb)) {
      b = t <= sb ? piece(t) : Q::inf();
      t += L;
    } else {
      chain = false;
      if (off == 0) break;
      b = Q::from_below(acc, off, sub < off);
      off >>= 1;
    }
    acc = Q::add(acc, b);
  }
  if (store && sub == 0) Q::store(j.buckets, k, acc);
}

// Each task's interior segment partials summed by one block.
template <bool G2>
__global__ void __launch_bounds__(TAIL_BLOCK) k_tail_heavy_tasks(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  constexpr uint32_t POINTS = TAIL_BLOCK / Q::LANES;
  const uint32_t nt = j.cnt[1];
  for (uint32_t t = blockIdx.x; t < nt; t += gridDim.x) {
    uint32_t i = j.tasks[2 * t] + Q::slot();
    const uint32_t hi = j.tasks[2 * t + 1];
    Coord acc = i < hi ? Q::load(j.pfirst, i) : Q::inf();
    acc = Q::template block_sum<TAIL_BLOCK>(acc, [&](Coord& b) {
      i += POINTS;
      if (!__any(i < hi)) return false;
      b = i < hi ? Q::load(j.pfirst, i) : Q::inf();
      return true;
    });
    if (Q::slot() == 0) Q::store(j.task_sum, t, acc);
    __syncthreads();
  }
}

// A heavy bucket's task sums and its two end pieces (item nt: plast of the first segment,
// nt + 1: pfirst of the last).
template <bool G2>
__global__ void __launch_bounds__(TAIL_BLOCK) k_tail_heavy_finish(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  constexpr uint32_t POINTS = TAIL_BLOCK / Q::LANES;
  const uint32_t nh = j.cnt[0];
  for (uint32_t h = blockIdx.x; h < nh; h += gridDim.x) {
    const uint32_t k = j.heavy[3 * h], tb = j.heavy[3 * h + 1], nt = j.heavy[3 * h + 2];
    const uint32_t sa = j.offset[k] / j.seg, sb = (j.offset[k + 1] - 1) / j.seg;
    const auto item = [&](uint32_t i) {
      const uint4* src = i < nt ? j.task_sum : (i == nt ? j.plast : j.pfirst);
      return Q::load(src, i < nt ? (size_t)tb + i : (i == nt ? sa : sb));
    };
    uint32_t i = Q::slot();
    const uint32_t n = nt + 2;
    Coord acc = i < n ? item(i) : Q::inf();
    acc = Q::template block_sum<TAIL_BLOCK>(acc, [&](Coord& b) {
      i += POINTS;
      if (!__any(i < n)) return false;
      b = i < n ? item(i) : Q::inf();
      return true;
    });
    if (Q::slot() == 0) Q::store(j.buckets, k, acc);
    __syncthreads();
  }
}

// Level 1 of the window reduction (see msm_accum.cuh): group g's T = sum_i B_{gB+i} and
// U = sum_i (i+1) B_{gB+i}, one point per group, 2 (B - 1) additions.
template <bool G2, bool CW>
__global__ void __launch_bounds__(TAIL_BLOCK) k_tail_groups(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  const uint32_t t = blockIdx.x * (TAIL_BLOCK / Q::LANES) + Q::slot();
  const uint32_t n = j.sets * j.G;
  if (blockIdx.x * (TAIL_BLOCK / Q::LANES) >= n) return;
  const uint32_t g = t < n ? t : n - 1;  // past the last group: repeat it, store nothing
  const size_t base = (size_t)g * j.B;
  const auto bucket = [&](size_t i) {
    return CW ? Q::load_proj(j.buckets, i) : Q::load(j.buckets, i);
  };
  Coord run = bucket(base + j.B - 1), acc = run;
#pragma unroll 1
  for (int i = 2 * (int)j.B - 3; i >= 0; --i) {  // odd: run += B_{i/2}; even: acc += run
    const Coord next = bucket(base + (uint32_t)(i >> 1));
    const Coord r = Q::template add<CW>((i & 1) ? run : acc, (i & 1) ? next : run);
    if (i & 1) run = r;
    else acc = r;
  }
  if (t < n) {
    Q::store(j.gT, t, run);
    Q::store(j.gU, t, acc);
  }
}

// Level 2: block x = ((w rows + r) S + slice) sums its slice of row r of set w; S = 1 writes
// the host's row, else a slice sum for k_tail_slices.
template <bool G2, bool CW>
__global__ void __launch_bounds__(TAIL_BLOCK) k_tail_rows(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  if (blockIdx.x >= j.sets * j.rows * j.S) return;
  constexpr uint32_t POINTS = TAIL_BLOCK / Q::LANES;
  const uint32_t sl = blockIdx.x % j.S, wr = blockIdx.x / j.S;
  const uint32_t w = wr / j.rows, r = wr % j.rows;
  const size_t base = (size_t)w * j.G;
  const uint4* src = r == 0 ? j.gU : j.gT;
  const uint32_t k = r == 0 ? 0 : r - 1, low = (1u << k) - 1u, count = r == 0 ? j.G : j.G / 2;
  const uint32_t per = count / j.S, m1 = (sl + 1) * per;
  // row 0: every g; row k + 1: m with a 1 inserted at bit k
  const auto item = [&](uint32_t m) {
    return Q::load(src, base + (r == 0 ? m : ((m & ~low) << 1) | (1u << k) | (m & low)));
  };
  uint32_t m = sl * per + Q::slot();
  Coord acc = m < m1 ? item(m) : Q::inf();
  acc = Q::template block_sum<TAIL_BLOCK, CW>(acc, [&](Coord& b) {
    m += POINTS;
    if (!__any(m < m1)) return false;
    b = m < m1 ? item(m) : Q::inf();
    return true;
  });
  if (Q::slot() == 0) {
    if (j.S == 1) Q::store_out(j.out, blockIdx.x, acc);
    else Q::store(j.parts, blockIdx.x, acc);
    __threadfence_system();  // `out` may be pinned host memory the host reads next
  }
}

// Row x = w rows + r: out[x] = sum of parts[x S .. x S + S), one wave per row.
template <bool G2, bool CW>
__global__ void __launch_bounds__(64) k_tail_slices(const TailJobs jobs) {
  using Q = Quad<G2>;
  const TailJob& j = jobs.job[blockIdx.y];
  if (j.S == 1 || blockIdx.x >= j.sets * j.rows) return;
  uint32_t i = Q::slot();
  const size_t base = (size_t)blockIdx.x * j.S;
  Coord acc = i < j.S ? Q::load(j.parts, base + i) : Q::inf();
  acc = Q::template block_sum<64, CW>(acc, [&](Coord& b) {
    i += Q::WAVE_POINTS;
    if (!__any(i < j.S)) return false;
    b = i < j.S ? Q::load(j.parts, base + i) : Q::inf();
    return true;
  });
  if (Q::slot() == 0) {
    Q::store_out(j.out, blockIdx.x, acc);
    __threadfence_system();  // `out` may be pinned host memory the host reads next
  }
}

// The stage-11 products of key points and blinders: block x of proof y sums the entries of its
// point's table of 256 doublings (2^w P, XYZZ) at the scalar's set bits, as a chain of four (G2:
// eight) additions per point of the block and a tree: 57 us for the five products of 16 proofs,
// 59-67 us beside one proof's other kernels (MI355X). On the host they were five double-and-add
// chains on the calling thread, 600 us, longer than all the kernels of a 1000-constraint proof.
//   x: 0 r delta1, 1 s alpha1, 2 r beta1, 3 rs delta1, 4 s delta2
template <bool G2>
__device__ __forceinline__ void blind_product(const uint4* table, const uint32_t* scalar,
                                              uint4* out) {
  using Q = Quad<G2>;
  constexpr uint32_t POINTS = TAIL_BLOCK / Q::LANES;
  const auto term = [&](uint32_t w) {
    return w < 256 && ((scalar[w >> 5] >> (w & 31u)) & 1u) ? Q::load(table, w) : Q::inf();
  };
  uint32_t w = Q::slot();
  Coord acc = term(w);
  acc = Q::template block_sum<TAIL_BLOCK>(acc, [&](Coord& b) {
    w += POINTS;
    if (w - Q::slot() >= 256) return false;
    b = term(w);
    return true;
  });
  if (Q::slot() == 0) {
    Q::store_out(out, 0, acc);
    __threadfence_system();  // `out` is pinned host memory the host reads next
  }
}

__global__ void __launch_bounds__(TAIL_BLOCK) k_blind(const uint4* tables,
                                                      const uint32_t* scalars, uint4* out) {
  const uint32_t x = blockIdx.x, y = blockIdx.y;
  const uint32_t point[5] = {0, 1, 2, 0, 0}, which[5] = {0, 1, 0, 2, 1};
  __shared__ uint32_t k[8];  // the scalar, read from host memory once
  if (threadIdx.x < 8) k[threadIdx.x] = scalars[(y * 3 + which[x]) * 8 + threadIdx.x];
  __syncthreads();
  uint4* o = out + (size_t)(y * 5 + x) * 16;
  if (x < 4) blind_product<false>(tables + point[x] * 256 * 8, k, o);
  else blind_product<true>(tables + 3 * 256 * 8, k, o);
}

void launch_blind(const void* tables, const void* scalars, void* out, uint32_t proofs,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_blind, dim3(5, proofs), dim3(TAIL_BLOCK), 0, s,
                     static_cast<const uint4*>(tables), static_cast<const uint32_t*>(scalars),
                     static_cast<uint4*>(out));
  G16_LAUNCH_CHECK("blinding products");
}

template <class Fn>
static uint32_t most(const TailJobs& t, Fn f) {
  uint32_t m = 0;
  for (int i = 0; i < t.n; ++i) m = std::max<uint32_t>(m, f(t.job[i]));
  return m;
}

template <bool G2, uint32_t L>
static void launch_merge(const TailJobs& t, hipStream_t s) {
  constexpr uint32_t per = TAIL_BLOCK / Quad<G2>::LANES / L;
  const uint32_t K = most(t, [](const TailJob& j) { return j.K; });
  hipLaunchKernelGGL((k_tail_merge<G2, L>), dim3((K + per - 1) / per, t.n), dim3(TAIL_BLOCK), 0, s,
                     t);
  G16_LAUNCH_CHECK("msm merge");
}

template <bool G2>
static void merge_jobs(const TailJobs& t, hipStream_t s) {
  // Points per bucket from the average pieces per bucket. With both lines at half as many pieces
  // G2 MSMs of 2^16 and 2^18 take 865 and 1721 us for 773 and 1533 and a batch of sixteen
  // 60k-constraint proofs 12.2 ms for 11.0; at twice as many the 1.1M-constraint prove takes 15.0
  // ms for 11.7 and the 5000-constraint one 753 us for 707, though G1 MSMs of 2^16 and 2^18
  // gain (478 for 510 us, 708 for 775): one pair of lines is a compromise (MI355X).
  const uint32_t m = most(t, [](const TailJob& j) { return j.avg_pieces; });
  if (m < 3) launch_merge<G2, 1>(t, s);
  else if (m < 24) launch_merge<G2, 4>(t, s);
  else launch_merge<G2, 8>(t, s);
  hipLaunchKernelGGL(k_tail_heavy_tasks<G2>, dim3(512, t.n), dim3(TAIL_BLOCK), 0, s, t);
  G16_LAUNCH_CHECK("msm heavy tasks");
  hipLaunchKernelGGL(k_tail_heavy_finish<G2>, dim3(128, t.n), dim3(TAIL_BLOCK), 0, s, t);
  G16_LAUNCH_CHECK("msm heavy finish");
}

template <bool G2, bool CW>
static void reduce_jobs(const TailJobs& t, hipStream_t s) {
  constexpr uint32_t per = TAIL_BLOCK / Quad<G2>::LANES;
  const uint32_t groups = most(t, [](const TailJob& j) { return j.sets * j.G; });
  hipLaunchKernelGGL((k_tail_groups<G2, CW>), dim3((groups + per - 1) / per, t.n), dim3(TAIL_BLOCK), 0,
                     s, t);
  G16_LAUNCH_CHECK("msm reduce groups");
  const uint32_t rows = most(t, [](const TailJob& j) { return j.sets * j.rows * j.S; });
  hipLaunchKernelGGL((k_tail_rows<G2, CW>), dim3(rows, t.n), dim3(TAIL_BLOCK), 0, s, t);
  G16_LAUNCH_CHECK("msm reduce rows");
  if (most(t, [](const TailJob& j) { return j.S; }) > 1) {
    const uint32_t sr = most(t, [](const TailJob& j) { return j.sets * j.rows; });
    hipLaunchKernelGGL((k_tail_slices<G2, CW>), dim3(sr, t.n), dim3(64), 0, s, t);
    G16_LAUNCH_CHECK("msm reduce slices");
  }
}

void tail_merge_jobs(int group, const TailJobs& t, hipStream_t s) {
  if (group == 1) merge_jobs<false>(t, s);
  else merge_jobs<true>(t, s);
}

void tail_reduce_jobs(int group, bool constant, const TailJobs& t, hipStream_t s) {
  if (group == 1) constant ? reduce_jobs<false, true>(t, s) : reduce_jobs<false, false>(t, s);
  else constant ? reduce_jobs<true, true>(t, s) : reduce_jobs<true, false>(t, s);
}

}  // namespace g16
