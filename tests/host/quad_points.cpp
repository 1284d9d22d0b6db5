// The points spread over lanes (snarkrs_amd/csrc/msm_quad.cuh) on an emulated wave, for
// tests/test_limb_points.py: each lane is a fiber, and a lane move or vote ends a lane's turn, so
// that it finds every lane's operand when its next turn comes (a wave's lanes take part in every
// operation, as the kernels have it). The code that runs is the kernels' own. Checked against the word-form XYZZ formulas of bn254.cuh: additions (general,
// doublings, cancellations and infinity in one wave, with and without constant work), doublings,
// loads, stores and block sums, with every coordinate's bound after each step and operands at the
// top of theirs. Prints "ok <steps>", or the first mismatches and exits 1.
#include <hip/hip_runtime.h>
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <random>
#include <vector>

// ---- the emulated block --------------------------------------------------------------
namespace emu {
constexpr int MOST = 256;
enum State { READY, BARRIER, DONE };
struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack = std::vector<char>(256 << 10);
  State state = DONE;
  unsigned ops = 0;
};
static Fiber fiber[MOST];
static ucontext_t scheduler;
static int cur = 0, threads = 0;
static uint32_t value[2][MOST];
static int kind[2][MOST];
static std::function<void()> body;

static void enter() {
  body();
  fiber[cur].state = DONE;
}
static void turn_over() { swapcontext(&fiber[cur].ctx, &scheduler); }

// Every lane's x of the same operation; two buffers, since a lane may be one operation ahead.
static const uint32_t* exchange(int what, uint32_t x) {
  const int b = fiber[cur].ops++ & 1;
  value[b][cur] = x;
  kind[b][cur] = what;
  turn_over();
  return value[b];
}
static uint32_t from(int what, uint32_t x, int src) {
  const uint32_t* v = exchange(what, x);
  if (kind[(fiber[cur].ops - 1) & 1][src] != what) {
    std::printf("lane %d reads lane %d, which is at another operation\n", cur, src);
    std::fflush(stdout);
    std::_Exit(1);  // on a fiber's stack
  }
  return v[src];
}
static uint32_t dpp(uint32_t x, int ctrl) {
  if (ctrl != 0x128 && ctrl > 0xff) std::_Exit(2);
  // row_ror:8 swaps the halves of 16 lanes; otherwise two bits per lane of a quad
  const int src = ctrl == 0x128 ? cur ^ 8 : (cur & ~3) | ((ctrl >> (2 * (cur & 3))) & 3);
  return from(ctrl, x, src);
}
static uint32_t bpermute(int addr, uint32_t x) {
  return from(0x1000, x, (cur & ~63) | ((addr >> 2) & 63));
}
static bool any(bool p) {
  const uint32_t* v = exchange(0x1001, p);
  bool r = false;
  for (int l = cur & ~63, e = l + 64; l < e; ++l) r |= v[l] != 0;
  return r;
}
static void barrier() {
  fiber[cur].state = BARRIER;
  turn_over();
}
static void run(int n, std::function<void()> f) {
  body = std::move(f);
  threads = n;
  for (int i = 0; i < n; ++i) {
    getcontext(&fiber[i].ctx);
    fiber[i].ctx.uc_stack.ss_sp = fiber[i].stack.data();
    fiber[i].ctx.uc_stack.ss_size = fiber[i].stack.size();
    fiber[i].ctx.uc_link = &scheduler;
    makecontext(&fiber[i].ctx, enter, 0);
    fiber[i].state = READY;
    fiber[i].ops = 0;
  }
  for (;;) {
    bool ran = false;
    for (int w = 0; w < n; w += 64) {  // a wave runs until all its lanes end or wait
      bool ready = true;
      while (ready) {
        ready = false;
        for (int i = w; i < w + 64; ++i)
          if (fiber[i].state == READY) {
            cur = i;
            swapcontext(&scheduler, &fiber[i].ctx);
            ready = ran = true;
          }
      }
    }
    if (!ran) break;
    for (int i = 0; i < n; ++i)
      if (fiber[i].state == BARRIER) fiber[i].state = READY;
  }
}
struct Idx {
  unsigned x;
};
}  // namespace emu

#undef __device__
#define __device__
#undef __shared__
#define __shared__ static
#define threadIdx (emu::Idx{(unsigned)emu::cur})
#define __lane_id() (emu::cur & 63)
#define __any(p) emu::any(p)
#define __syncthreads() emu::barrier()
#define __builtin_amdgcn_mov_dpp(x, ctrl, rows, banks, bound) emu::dpp((uint32_t)(x), ctrl)
#define __builtin_amdgcn_ds_bpermute(addr, x) emu::bpermute(addr, (uint32_t)(x))
#include "../../snarkrs_amd/csrc/msm_quad.cuh"

using namespace g16;

static std::mt19937_64 rng(7);
static long bad = 0, steps = 0;
static void report(const char* what, int a, int b) {
  if (++bad <= 8) std::printf("%s: %d %d\n", what, a, b);
}

// ---- values --------------------------------------------------------------------------
// x against k q, limbs of any size: negative, zero or positive
static int against_kq(const uint32_t x[9], int k) {
  int64_t c = 0, d[10];
  for (int j = 0; j < 9; ++j) {
    const int64_t v = (int64_t)x[j] - (int64_t)Fq29::p29(j) * k + c;
    d[j] = v & 0x1fffffff;
    c = v >> 29;
  }
  if (c < 0) return -1;
  for (int j = 0; j < 9; ++j)
    if (d[j]) return 1;
  return c ? 1 : 0;
}
static bool below(const uint32_t x[9], int k, uint32_t limb) {
  for (int j = 0; j < 9; ++j)
    if (x[j] >= limb) return false;
  return against_kq(x, k) < 0;
}
static Fm word(const uint32_t x[9]) {  // below 2q, from any value below 16q
  uint32_t one[9], r[9];
  for (int j = 0; j < 9; ++j) one[j] = one29(j);
  mont29_limbs<Fq29>(x, one, r);
  Fm w;
  pack29(r, w.v);
  return w;
}
static bool equal(const Fm& a, const Fm& b) { return is_zero(sub(a, b)); }
static bool equal(const Fm2i& a, const Fm2i& b) { return equal(a.c0, b.c0) && equal(a.c1, b.c1); }
static Fm& comp(Fm& x, int) { return x; }
static Fm& comp(Fm2i& x, int c) { return c ? x.c1 : x.c0; }
static Fm rnd() {
  Fm a;
  do {
    for (int i = 0; i < 8; ++i) a.v[i] = (uint32_t)rng();
    a.v[7] &= 0x3fffffffu;
    uint32_t l[9];
    limbs29_of(a.v, l);
    if (against_kq(l, 1) < 0) return a;
  } while (true);
}

// One point as the lanes hold it: [coordinate][component][limb].
struct Lanes {
  uint32_t v[4][2][9] = {};
};
template <bool G2> using Field = std::conditional_t<G2, Fm2i, Fm>;

template <bool G2>
static Xyzz<Field<G2>> xyzz(const Lanes& p) {
  Xyzz<Field<G2>> r;
  for (int c = 0; c < (G2 ? 2 : 1); ++c) {
    comp(r.X, c) = word(p.v[0][c]);
    comp(r.Y, c) = word(p.v[1][c]);
    comp(r.ZZ, c) = word(p.v[2][c]);
    comp(r.ZZZ, c) = word(p.v[3][c]);
  }
  return r;
}
// The point's limbs plus multiples of q: `top` takes each coordinate to the top of its bound
// (X < 9q, Y < 5q, ZZ and ZZZ < 2q), with X's and Y's limbs as high as a carry leaves them.
template <bool G2>
static Lanes lanes(Xyzz<Field<G2>> p, bool top) {
  Lanes r;
  for (int c = 0; c < (G2 ? 2 : 1); ++c) {
    const Fm x[4] = {comp(p.X, c), comp(p.Y, c), comp(p.ZZ, c), comp(p.ZZZ, c)};
    const int k[4] = {9, 5, 2, 2};
    for (int i = 0; i < 4; ++i) {
      uint32_t* v = r.v[i][c];
      limbs29_of(x[i].v, v);
      const bool none = i >= 2 && is_zero(x[i]);  // infinity stays 0
      while (top && !none) {
        uint32_t n[9], cy = 0;
        for (int j = 0; j < 9; ++j) {
          n[j] = v[j] + Fq29::p29(j) + cy;
          cy = j < 8 ? n[j] >> 29 : 0;
          if (j < 8) n[j] &= 0x1fffffffu;
        }
        if (against_kq(n, k[i]) >= 0) break;
        for (int j = 0; j < 9; ++j) v[j] = n[j];
      }
      if (top && i < 2)
        for (int j = 8; j > 0; --j)
          if (v[j] && v[j - 1] < 8) v[j] -= 1, v[j - 1] += 1u << 29;
    }
  }
  return r;
}
template <bool G2>
static bool bounds(const Lanes& p) {
  for (int c = 0; c < (G2 ? 2 : 1); ++c)
    if (!below(p.v[0][c], 9, (1u << 29) + 8) || !below(p.v[1][c], 5, (1u << 29) + 8) ||
        !below(p.v[2][c], 2, 1u << 29) || !below(p.v[3][c], 2, 1u << 29))
      return false;
  return true;
}
template <class F>
static bool same(const Xyzz<F>& p, const Xyzz<F>& q) {
  const bool pi = is_zero(p.ZZ), qi = is_zero(q.ZZ);
  if (pi || qi) return pi == qi;
  return equal(mul(p.X, q.ZZ), mul(q.X, p.ZZ)) && equal(mul(p.Y, q.ZZZ), mul(q.Y, p.ZZZ));
}

template <bool G2>
static Coord get(const Lanes& p) {
  using Q = Quad<G2>;
  Coord r;
  for (int j = 0; j < 9; ++j) r.v[j] = p.v[Q::coord()][Q::comp()][j];
  return r;
}
template <bool G2>
static void set(Lanes& p, const Coord& r) {
  using Q = Quad<G2>;
  for (int j = 0; j < 9; ++j) p.v[Q::coord()][Q::comp()][j] = r.v[j];
}

// A point with random ZZ, ZZZ (ZZ^3 = ZZZ^2) on the curve y^2 = x^3 + b of a random (x, y); the
// formulas for a = 0 know no b.
template <class F>
static F rnd_f();
template <> Fm rnd_f<Fm>() { return rnd(); }
template <> Fm2i rnd_f<Fm2i>() { return Fm2i{rnd(), rnd()}; }
template <class F>
static Xyzz<F> scaled(const Xyzz<F>& p, const F& z = rnd_f<F>()) {
  const F z2 = mul(z, z), z3 = mul(z2, z);
  return Xyzz<F>{mul(p.X, z2), mul(p.Y, z3), mul(p.ZZ, z2), mul(p.ZZZ, z3)};
}
template <class F>
static Xyzz<F> rnd_point() {
  return scaled(Xyzz<F>{rnd_f<F>(), rnd_f<F>(), f_one<F>(), f_one<F>()});
}

// In G2 a component may be zero where the value is not: d with one component zero, and d whose
// square has one.
static Fm half_zero(Fm d, int) { return d; }
static Fm2i half_zero(Fm2i d, int how) {
  if (how == 0) d.c0 = f_zero<Fm>();
  if (how == 1) d.c1 = f_zero<Fm>();
  if (how == 2) d.c1 = d.c0;
  return d;
}

// ---- checks --------------------------------------------------------------------------
template <bool G2, bool CW>
static void additions(const char* name) {
  using Q = Quad<G2>;
  using F = Field<G2>;
  constexpr int N = Q::WAVE_POINTS;
  for (int it = 0; it < 24; ++it) {
    Lanes a[N], b[N], r[N];
    for (int i = 0; i < N; ++i) {
      Xyzz<F> p = rnd_point<F>(), q = rnd_point<F>();
      if (G2 && i >= N / 2) {  // x's or y's difference, ZZ or ZZZ
        const int how = (int)(rng() % 3);
        const F d = half_zero(rnd_f<F>(), how);
        p.ZZ = p.ZZZ = q.ZZ = q.ZZZ = f_one<F>();
        if (i & 1) q.X = add(p.X, d);
        else q.X = p.X, q.Y = add(p.Y, d);
        if (how < 2 && it % 4 == 0) p = scaled(p, half_zero(rnd_f<F>(), how));
      }
      // A third of the waves hold none of the rare cases, which skip the doubling.
      const int rare = it % 3 ? (int)(rng() % 6) : 5;
      if (rare == 0) q = scaled(p);                                // p + p, other coordinates
      if (rare == 1) q = scaled(p), q.Y = neg(q.Y);                // p - p
      if (rare == 2) q = xyzz_inf<F>();
      const bool p_inf = rare == 3 || (rare == 2 && rng() % 4 == 0);
      a[i] = lanes<G2>(p_inf ? xyzz_inf<F>() : p, it & 1);
      b[i] = lanes<G2>(q, it & 1);
      if (rare == 4) b[i] = a[i];                                  // p + p, the same limbs
    }
    emu::run(64, [&] {
      const uint32_t i = Q::slot();
      set<G2>(r[i], Q::template add<CW>(get<G2>(a[i]), get<G2>(b[i])));
    });
    for (int i = 0; i < N; ++i, ++steps) {
      if (!same(xyzz<G2>(r[i]), xyzz_add(xyzz<G2>(a[i]), xyzz<G2>(b[i])))) report(name, it, i);
      if (!bounds<G2>(r[i])) report("bounds (add)", it, i);
    }
  }
}

template <bool G2>
static void doublings() {
  using Q = Quad<G2>;
  using F = Field<G2>;
  constexpr int N = Q::WAVE_POINTS;
  for (int it = 0; it < 8; ++it) {
    Lanes a[N], r[N];
    for (auto& p : a) p = lanes<G2>(rnd_point<F>(), it & 1);
    emu::run(64, [&] { set<G2>(r[Q::slot()], Q::dbl(get<G2>(a[Q::slot()]))); });
    for (int i = 0; i < N; ++i, ++steps) {
      if (!same(xyzz<G2>(r[i]), xyzz_dbl(xyzz<G2>(a[i])))) report("double", it, i);
      if (!bounds<G2>(r[i])) report("bounds (double)", it, i);
    }
  }
}

// Stores and loads of every form.
template <bool G2>
static void memory() {
  using Q = Quad<G2>;
  using F = Field<G2>;
  constexpr int N = Q::WAVE_POINTS, W = Q::POINT_WORDS;
  for (int it = 0; it < 8; ++it) {
    Lanes a[N], kept[N], out[N], aff[N], proj[N];
    Xyzz<F> p[N];
    std::vector<uint4> mem(N * W), mem2(N * W), mem3(N * W), xy(N * W / 2);
    for (int i = 0; i < N; ++i) {
      p[i] = i == 1 ? xyzz_inf<F>() : rnd_point<F>();
      a[i] = lanes<G2>(p[i], it & 1);
      // the first two coordinates as an affine base (0, 0 the point at infinity), the first three
      // as a constant-work slot
      if (i == 1) p[i].X = p[i].Y = f_zero<F>();
      if (i > 2) p[i].X = half_zero(p[i].X, i & 1), p[i].Y = half_zero(p[i].Y, i & 1);
      std::memcpy(&xy[i * W / 2], &p[i], 8 * W);
      Xyzz<F> s = p[i];
      s.ZZZ = f_zero<F>();
      std::memcpy(&mem3[i * W], &s, 16 * W);
    }
    emu::run(64, [&] {
      const uint32_t i = Q::slot();
      Q::store(mem.data(), i, get<G2>(a[i]));
      Q::store_out(mem2.data(), i, get<G2>(a[i]));
      set<G2>(kept[i], Q::load(mem.data(), i));
      set<G2>(out[i], Q::load(mem2.data(), i));
      set<G2>(proj[i], Q::load_proj(mem3.data(), i));
      const uint32_t at = (Q::coord() & 1u) * (W / 4) + Q::comp() * 2;
      const uint4* base = xy.data() + i * (W / 2) + at;
      set<G2>(aff[i], Q::from_affine(base[0], base[1], i & 1, i != 2));
    });
    for (int i = 0; i < N; ++i, ++steps) {
      for (int k = 0; k < 4; ++k)
        for (int c = 0; c < (G2 ? 2 : 1); ++c) {
          if (!equal(word(kept[i].v[k][c]), word(a[i].v[k][c])) ||
              !below(kept[i].v[k][c], 5, 1u << 29))
            report("store", i, k);
          if (!equal(word(out[i].v[k][c]), word(a[i].v[k][c])) ||
              !below(out[i].v[k][c], 2, 1u << 29))
            report("store for the host", i, k);
        }
      Xyzz<F> want{p[i].X, (i & 1) ? neg(p[i].Y) : p[i].Y, f_one<F>(), f_one<F>()};
      if (i == 1 || i == 2) want = xyzz_inf<F>();
      if (!same(xyzz<G2>(aff[i]), want) || !bounds<G2>(aff[i])) report("affine base", it, i);
      const F z = p[i].ZZ, z2 = mul(z, z);
      const Xyzz<F> g = xyzz<G2>(proj[i]);
      if (!equal(g.X, mul(p[i].X, z)) || !equal(g.Y, mul(p[i].Y, z2)) || !equal(g.ZZ, z2) ||
          !equal(g.ZZZ, mul(z2, z)) || !bounds<G2>(proj[i]))
        report("constant-work slot", it, i);
    }
  }
}

// Sums of n multiples of one point over a block, every point of it with its own chain.
template <bool G2, int BLOCK, bool CW>
static void block_sums() {
  using Q = Quad<G2>;
  using F = Field<G2>;
  constexpr uint32_t POINTS = BLOCK / Q::LANES;
  std::vector<Xyzz<F>> multiple{xyzz_inf<F>(), rnd_point<F>()};
  for (int k = 2; k < 64; ++k) multiple.push_back(xyzz_add(multiple[k - 1], multiple[1]));
  for (uint32_t n : {0u, 1u, POINTS - 1, POINTS + 1, 3 * POINTS + 5}) {
    std::vector<Lanes> term(n);
    Xyzz<F> want = xyzz_inf<F>();
    for (uint32_t i = 0; i < n; ++i) {
      const Xyzz<F>& m = multiple[rng() % 64];
      term[i] = lanes<G2>(m, false);
      want = xyzz_add(want, m);
    }
    Lanes r;
    emu::run(BLOCK, [&] {
      uint32_t i = Q::slot();
      const auto item = [&] { return i < n ? get<G2>(term[i]) : Q::inf(); };
      const Coord acc = Q::template block_sum<BLOCK, CW>(item(), [&](Coord& b) {
        i += POINTS;
        if (!__any(i < n)) return false;
        b = item();
        return true;
      });
      if (Q::slot() == 0) set<G2>(r, acc);
    });
    ++steps;
    if (!same(xyzz<G2>(r), want)) report("block sum", BLOCK, (int)n);
    if (!bounds<G2>(r)) report("bounds (block sum)", BLOCK, (int)n);
  }
}

int main() {
  additions<false, false>("G1 add");
  additions<false, true>("G1 add, constant work");
  additions<true, false>("G2 add");
  additions<true, true>("G2 add, constant work");
  doublings<false>();
  doublings<true>();
  memory<false>();
  memory<true>();
  block_sums<false, 64, false>();
  block_sums<false, 256, true>();
  block_sums<true, 64, true>();
  block_sums<true, 256, false>();
  if (bad) {
    std::printf("%ld mismatches in %ld steps\n", bad, steps);
    return 1;
  }
  std::printf("ok %ld\n", steps);
  return 0;
}
