// The 29-bit-limb products and reductions of snarkrs_amd/csrc/bn254.cuh on limbs read from
// standard input, for tests/test_limb_reduce.py: a line "op limbs..." (nine limbs per operand)
// gives a line of result limbs.
//   q, r    mont29_limbs over Fq / Fr (two operands)
//   s       redc29 of a b + c d - e f - g h;  p  redc29 of a b + c d, which is never negative
//   u       redc29u of a b + c d + e f + g h
//   x       g1l_pack's X (one operand), as eight words
#include <cstdio>

#include "../../snarkrs_amd/csrc/bn254.cuh"

using namespace g16;

int main() {
  char op;
  while (std::scanf(" %c", &op) == 1) {
    const int n = op == 'q' || op == 'r' ? 2 : op == 'x' ? 1 : op == 'p' ? 4 : 8;
    uint32_t v[8][9], R[9] = {};
    for (int i = 0; i < n; ++i)
      for (int j = 0; j < 9; ++j)
        if (std::scanf("%u", &v[i][j]) != 1) return 1;
    uint64_t t[17] = {};
    int len = 9;
    if (op == 'q') {
      mont29_limbs<Fq29>(v[0], v[1], R);
    } else if (op == 'r') {
      mont29_limbs<Fr29>(v[0], v[1], R);
    } else if (op == 'x') {
      G1L p = g1l_inf();
      for (int j = 0; j < 9; ++j) p.X[j] = v[0][j];
      const Xyzz<Fm> w = g1l_pack(p);
      for (int j = 0; j < 8; ++j) R[j] = w.X.v[j];
      len = 8;
    } else {
      wide_mac(t, v[0], v[1]);
      wide_mac(t, v[2], v[3]);
      if (op == 's') {
        wide_msub(t, v[4], v[5]);
        wide_msub(t, v[6], v[7]);
        redc29<Fq29>(t, R);
      } else if (op == 'p') {
        redc29<Fq29, false>(t, R);
      } else {
        wide_mac(t, v[4], v[5]);
        wide_mac(t, v[6], v[7]);
        redc29u<Fq29>(t, R);
      }
    }
    for (int j = 0; j < len; ++j) std::printf("%u ", R[j]);
    std::printf("\n");
  }
  return 0;
}
