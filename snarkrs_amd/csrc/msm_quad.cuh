// XYZZ point additions spread over lanes, for the MSM's tails (merges, heavy buckets, window
// reduction) and everything else that is a short chain of dependent additions on few points.
//
// A general addition is 14 products one after the other on one lane, and with one wave on a
// SIMD each instruction waits for the one before: 6 us (G1) and 16-20 us (G2) per addition,
// nearly all of a tail's time. Here a G1 point lives in four neighbouring lanes, one
// coordinate each (X, Y, ZZ, ZZZ), and the same formula (add-2008-s) is four products deep:
//   1. U1 = X1 ZZ2 | S1 = Y1 ZZZ2 | U2 = X2 ZZ1 | S2 = Y2 ZZZ1     (own times xor-2 neighbour)
//   2. PP = P^2    | RR = R^2     | ZZ1 ZZ2     | ZZZ1 ZZZ2        (P = U2 - U1, R = S2 - S1)
//   3. PPP = P PP  | Q = U1 PP    | ZZ3         | -
//   4. S1 PPP      | R (Q - X3)   | -           | ZZZ3
// with the operands moved by quad-permute DPP. A G2 point takes eight lanes, the two components
// of each coordinate 8 lanes apart (row_ror:8), so an Fq2 product is two limb products and one
// reduction per lane instead of four and two. A wave holds 16 G1 points or 8 G2 points. The
// lanes' total work is about 1.3 times the one-lane form's, in a fifth of the depth; the code
// is a fraction of it too (a G2 addition: ~15 KB against 150 KB).
//
// Bounds as in bn254.cuh's limb points, with X < 9q and Y < 5q (Y3 is reduced as two products),
// ZZ, ZZZ < 2q; a stored coordinate is below 5q.
#pragma once
#include "bn254.cuh"
#include "internal.h"

// The moves below must stay moves: see the Makefile's NEEDED.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(G16_NO_DPP_COMBINE)
#error "compile with -mllvm -amdgpu-dpp-combine=0 -DG16_NO_DPP_COMBINE"
#endif

namespace g16 {

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, true);
}
constexpr int quad_ctrl(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }
constexpr int ROW_ROR8 = 0x128;

// One coordinate (G2: one component of one) of a point, in limbs.
struct Coord {
  uint32_t v[9];
};

__device__ __forceinline__ Coord coord_sel(bool c, const Coord& a, const Coord& b) {
  Coord r;
#pragma unroll
  for (int j = 0; j < 9; ++j) r.v[j] = c ? a.v[j] : b.v[j];
  return r;
}

template <bool G2>
struct Quad {
  static constexpr int LANES = G2 ? 8 : 4;           // lanes per point
  static constexpr int WAVE_POINTS = 64 / LANES;
  static constexpr int POINT_WORDS = G2 ? 16 : 8;    // uint4 per stored point

  // The point this thread works on, in its block, and its coordinate and component there.
  static __device__ __forceinline__ uint32_t slot() {
    return G2 ? ((threadIdx.x >> 4) << 1) | ((threadIdx.x >> 2) & 1u) : threadIdx.x >> 2;
  }
  static __device__ __forceinline__ uint32_t coord() { return threadIdx.x & 3u; }
  static __device__ __forceinline__ uint32_t comp() { return G2 ? (threadIdx.x >> 3) & 1u : 0u; }
  // Whether this is the point's first lane.
  static __device__ __forceinline__ bool leader() { return coord() == 0 && comp() == 0; }
  static __device__ __forceinline__ uint32_t word() {  // this lane's place in a stored point
    return G2 ? coord() * 4 + comp() * 2 : coord() * 2;
  }

  template <int A, int B, int C, int D>
  static __device__ __forceinline__ Coord perm(const Coord& x) {
    Coord r;
#pragma unroll
    for (int j = 0; j < 9; ++j) r.v[j] = dpp_mov<quad_ctrl(A, B, C, D)>(x.v[j]);
    return r;
  }
  static __device__ __forceinline__ Coord other_comp(const Coord& x) {
    Coord r;
#pragma unroll
    for (int j = 0; j < 9; ++j) r.v[j] = dpp_mov<ROW_ROR8>(x.v[j]);
    return r;
  }

  // x y, exact limbs below 2q. G2: c0 = x0 y0 - x1 y1, c1 = x1 y0 + x0 y1, as own times A plus
  // the other component times B.
  static __device__ __forceinline__ Coord mul(const Coord& x, const Coord& y) {
    Coord r;
    if constexpr (!G2) {
      mont29_limbs<Fq29>(x.v, y.v, r.v);
    } else {
      const Coord xo = other_comp(x), yo = other_comp(y);
      const bool c1 = comp() != 0;
      uint32_t A[9];
      int32_t B[9];
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        A[j] = c1 ? yo.v[j] : y.v[j];
        B[j] = c1 ? (int32_t)y.v[j] : -(int32_t)yo.v[j];
      }
      uint64_t t[17];
#pragma unroll
      for (int k = 0; k < 17; ++k) t[k] = 0;
      wide_mac(t, x.v, A);
#pragma unroll
      for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int j = 0; j < 9; ++j)
          t[i + j] += (uint64_t)((int64_t)(int32_t)xo.v[i] * (int64_t)B[j]);
      redc29<Fq29>(t, r.v);
    }
    return r;
  }
  static __device__ __forceinline__ Coord below2q(const Coord& x) {  // a product with one
    uint32_t one[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) one[j] = one29(j);
    Coord r;
    mont29_limbs<Fq29>(x.v, one, r.v);
    return r;
  }

  template <class K>
  static __device__ __forceinline__ Coord sub(const Coord& a, const Coord& b) {
    Coord r;
    sub29<K>(a.v, b.v, r.v);
    return r;
  }

  // Whether the (exact, below 2q) coordinate held by lane C of the quad is 0 mod q.
  template <int C>
  static __device__ __forceinline__ bool zero_at(const Coord& x) {
    uint32_t f = zero29(x.v) ? 1u : 0u;
    if constexpr (G2) f &= dpp_mov<ROW_ROR8>(f);
    return dpp_mov<quad_ctrl(C, C, C, C)>(f) != 0;
  }

  static __device__ __forceinline__ Coord inf() {
    Coord r;
#pragma unroll
    for (int j = 0; j < 9; ++j) r.v[j] = 0;
    return r;
  }

  // 2p (dbl-2008-s-1), p not infinity; its coordinates are taken below 2q first.
  static __device__ __forceinline__ Coord dbl(const Coord& p) {
    const uint32_t l = coord();
    const Coord a = below2q(p);
    Coord u;
#pragma unroll
    for (int j = 0; j < 9; ++j) u.v[j] = a.v[j] + a.v[j];
    norm29(u.v);                                    // lane 1: U = 2Y < 4q
    const Coord t1 = mul(coord_sel(l == 1, u, a), coord_sel(l == 1, u, a));  // X^2 | V = U^2
    const Coord V = perm<1, 1, 1, 1>(t1), X2 = perm<0, 0, 0, 0>(t1);
    Coord M;
#pragma unroll
    for (int j = 0; j < 9; ++j) M.v[j] = 3u * X2.v[j];
    norm29(M.v);                                    // M = 3 X^2 < 6q
    Coord x = coord_sel(l == 1, u, a);
    x = coord_sel(l == 3, M, x);
    const Coord t2 = mul(x, coord_sel(l == 3, M, V));  // S = X V | W = U V | ZZ3 | M^2
    const Coord S = perm<0, 0, 0, 0>(t2), W = perm<1, 1, 1, 1>(t2), MM = perm<3, 3, 3, 3>(t2);
    Coord X3;
#pragma unroll
    for (int j = 0; j < 9; ++j) X3.v[j] = MM.v[j] + Kq5::k(j) - S.v[j] - S.v[j];
    norm29(X3.v);                                   // X3 = M^2 + 5q - 2S < 7q
    const Coord T = sub<Kq10>(S, X3);               // S - X3 + 10q < 12q
    // lane 0: M T, lane 1: W Y, lane 3: W ZZZ
    const Coord t3 = mul(coord_sel(l == 0, M, W), coord_sel(l == 0, T, a));
    const Coord MT = perm<0, 0, 0, 0>(t3);
    const Coord Y3 = sub<Kq3>(MT, t3);              // lane 1: < 5q
    Coord r = coord_sel(l == 0, X3, Y3);
    r = coord_sel(l == 2, t2, r);
    return coord_sel(l == 3, t3, r);
  }

  // a + b. Every lane of the wave that reaches this takes part; the rare doubling or
  // cancellation of any of them is resolved by all of them together. Constant work (CW)
  // computes the doubling every time and picks the result by selects.
  template <bool CW = false>
  static __device__ __forceinline__ Coord add(const Coord& a, const Coord& b) {
    const uint32_t l = coord();
    const bool ia = zero_at<2>(a), ib = zero_at<2>(b);
    const Coord t1 = mul(a, perm<2, 3, 0, 1>(b));   // U1 | S1 | U2 | S2
    const Coord d = sub<Kq3>(perm<2, 3, 0, 1>(t1), t1);  // P | R, + 3q < 5q
    const Coord t2 = mul(coord_sel(l < 2, d, a), coord_sel(l < 2, d, b));  // PP | RR | ZZ12 | ZZZ12
    const bool same_x = zero_at<0>(t2) && !ia && !ib;
    Coord x = coord_sel(l == 1, perm<0, 0, 0, 0>(t1), t2);
    x = coord_sel(l == 0, d, x);
    const Coord t3 = mul(x, perm<0, 0, 0, 0>(t2));  // PPP | Q | ZZ3 | -
    const Coord ppp = perm<0, 0, 0, 0>(t3);
    Coord X3;  // lane 1: RR - PPP - 2Q + 7q < 9q
#pragma unroll
    for (int j = 0; j < 9; ++j)
      X3.v[j] = t2.v[j] + Kq7::k(j) - ppp.v[j] - t3.v[j] - t3.v[j];
    norm29(X3.v);
    const Coord T = sub<Kq10>(t3, X3);              // lane 1: Q - X3 + 10q < 12q
    x = coord_sel(l == 0, perm<1, 1, 1, 1>(t1), t2);
    x = coord_sel(l == 1, d, x);
    const Coord t4 = mul(x, coord_sel(l == 1, T, ppp));  // S1 PPP | R T | - | ZZZ3
    const Coord Y3 = sub<Kq3>(t4, perm<0, 0, 0, 0>(t4));  // lane 1: R T - S1 PPP + 3q < 5q
    Coord r = coord_sel(l == 0, perm<1, 1, 1, 1>(X3), Y3);
    r = coord_sel(l == 2, t3, r);
    r = coord_sel(l == 3, t4, r);
    if (CW || __any(same_x)) {
      const bool same_y = zero_at<1>(t2);
      const Coord d2 = dbl(a);
      r = coord_sel(same_x, coord_sel(same_y, d2, inf()), r);
    }
    r = coord_sel(ib, a, r);
    return coord_sel(ia, b, r);
  }

  static __device__ __forceinline__ Coord load(const uint4* base, size_t i) {
    const uint4* p = base + i * POINT_WORDS + word();
    const uint4 lo = p[0], hi = p[1];
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    Coord r;
    limbs29_of(w, r.v);
    return r;
  }
  // The affine point whose x lanes 0 hold and whose y lanes 1 hold as words (any values on the
  // other lanes), negated or not, with ZZ = ZZZ = 1; infinity for (0, 0) or where `live` is false.
  static __device__ __forceinline__ Coord from_affine(const uint4& lo, const uint4& hi, bool negate,
                                                      bool live) {
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    const uint32_t l = coord();
    Coord p;
    limbs29_of(w, p.v);
    const bool none = zero_at<0>(p) && zero_at<1>(p);
    const Coord m = sub<Kq3>(inf(), p);  // 3q - y < 3q
    p = coord_sel(l == 1 && negate, m, p);
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const uint32_t one = comp() == 0 ? one29(j) : 0u;
      p.v[j] = !live || none ? 0u : l >= 2 ? one : p.v[j];
    }
    return p;
  }
  // A constant-work slot (X, Y, Z, 0) of the point (X : Y : Z) as (X Z, Y Z^2, Z^2, Z^3).
  static __device__ __forceinline__ Coord load_proj(const uint4* base, size_t i) {
    const uint32_t l = coord();
    const Coord a = load(base, i), z = perm<2, 2, 2, 2>(a);
    const Coord t1 = mul(coord_sel(l == 3, z, a), z);  // X Z | Y Z | Z^2 | Z^2
    const Coord t2 = mul(t1, z);                       // - | Y Z^2 | - | Z^3
    return coord_sel((l & 1u) != 0, t2, t1);
  }
  static __device__ __forceinline__ void put(uint4* base, size_t i, const Coord& x) {
    uint32_t w[8];
    pack29(x.v, w);
    uint4* p = base + i * POINT_WORDS + word();
    p[0] = make_uint4(w[0], w[1], w[2], w[3]);
    p[1] = make_uint4(w[4], w[5], w[6], w[7]);
  }
  // Below 5q (X may be up to 9q), as the one-lane kernels store X.
  static __device__ __forceinline__ void store(uint4* base, size_t i, const Coord& x) {
    Coord v = x;
    below5q(v.v);
    put(base, i, v);
  }
  // Every coordinate below 2q, for the host.
  static __device__ __forceinline__ void store_out(uint4* base, size_t i, const Coord& x) {
    put(base, i, below2q(x));
  }

  // The point `off` (a power of two) places after this one in the wave, or infinity where
  // `take` is false. Points sit 4 lanes apart, two to a row of 16 in G2.
  static __device__ __forceinline__ Coord from_below(const Coord& x, uint32_t off, bool take) {
    const uint32_t step = G2 ? (off == 1 ? 4u : off * 8u) : off * 4u;
    const int src = (int)(((__lane_id() + step) & 63u) << 2);
    Coord r;
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const uint32_t y = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)x.v[j]);
      r.v[j] = take ? y : 0u;
    }
    return r;
  }

  // The sum over a block of BLOCK threads, left at slot 0, of each point's acc and the terms
  // that follow: next(b) sets b to the point's next term (infinity when it has none) and
  // returns whether any point of the wave had one. Chain, tree across the wave and tree across
  // the waves share one addition site. Every lane of the block must arrive; the caller puts a
  // barrier before the next use.
  template <int BLOCK, bool CW = false, class Next>
  static __device__ __forceinline__ Coord block_sum(Coord acc, Next next) {
    constexpr int WAVES = BLOCK / 64;
    __shared__ uint32_t sh[WAVES][9][LANES];
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t q = slot() & (WAVE_POINTS - 1);  // point in the wave
    const uint32_t lane_of_point = coord() + 4 * comp();
    uint32_t off = WAVE_POINTS / 2;
    bool chain = true, crossed = WAVES == 1;
#pragma unroll 1
    for (;;) {
      Coord b;
      if (chain) {
        chain = next(b);
        if (!chain) continue;
      } else {
        if (off == 0) {
          if (crossed) break;
          crossed = true;
          if (q == 0) {
#pragma unroll
            for (int j = 0; j < 9; ++j) sh[wave][j][lane_of_point] = acc.v[j];
          }
          __syncthreads();
          if (wave != 0) break;
#pragma unroll
          for (int j = 0; j < 9; ++j)
            acc.v[j] = q < (uint32_t)WAVES ? sh[q & (WAVES - 1)][j][lane_of_point] : 0u;
          off = WAVES / 2;
        }
        b = from_below(acc, off, q < off);
        off >>= 1;
      }
      acc = add<CW>(acc, b);
    }
    return acc;
  }
};

}  // namespace g16
