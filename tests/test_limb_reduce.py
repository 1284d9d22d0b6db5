"""The limb products' and reductions' results and bounds at their edges (bn254.cuh mont29_limbs,
redc29, redc29u, g1l_pack) against Python integers, on the host: every operand at the top of its
bound, limbs raised to 2^29 + 7, zero, multiples of the modulus, and random ones."""
import os
import random
import shutil
import subprocess

import pytest

from snarkrs_amd.wire import Q_MOD, R_MOD

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    exe = tmp_path_factory.mktemp("limb") / "limb_reduce"
    subprocess.run([HIPCC, "-O0", "-std=c++17", "--cuda-host-only", "-x", "hip",
                    os.path.join(HERE, "host", "limb_reduce.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)

    def call(lines):
        text = "\n".join(op + " " + " ".join(str(x) for v in vs for x in v) for op, vs in lines)
        r = subprocess.run([str(exe)], input=text + "\n", capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stderr
        out = [[int(x) for x in line.split()] for line in r.stdout.splitlines()]
        assert len(out) == len(lines)
        return out

    return call


def limbs(x):
    return [(x >> (29 * j)) & (2**29 - 1) for j in range(8)] + [x >> 232]


def value(v):
    return sum(x << (29 * j) for j, x in enumerate(v))


def raised(x):
    """The same value with every low limb as high as 2^29 + 7 allows."""
    v = limbs(x)
    for j in range(8, 0, -1):
        k = min(7, 2**29 + 7 - v[j - 1] >> 29, 1) if v[j] else 0
        if k and v[j - 1] < 8:
            v[j] -= 1
            v[j - 1] += 2**29
    return v


def operands(m, k, rng):
    """Values below k m: the largest, one whose low limbs are all ones, multiples of m, random."""
    top = k * m - 1
    ones = (top >> 232) - 1 << 232 | (1 << 232) - 1
    out = [top, ones, 0, 1, m, (k - 1) * m, m - 1] + [rng.randrange(k * m) for _ in range(12)]
    return [limbs(x) for x in out] + [raised(ones + 1), [2**29 + 7] * 8 + [(top >> 232) - 2]]


@pytest.mark.parametrize("op,m", [("q", Q_MOD), ("r", R_MOD)])
def test_product(run, op, m):
    rng = random.Random(5)
    a = operands(m, 12, rng) if op == "q" else operands(m, 5, rng)
    cases = [(x, y) for x in a for y in a]
    for (x, y), r in zip(cases, run([(op, c) for c in cases])):
        got = value(r)
        assert all(v < 2**29 for v in r)
        assert got < 2 * m and (got * 2**261 - value(x) * value(y)) % m == 0


@pytest.mark.parametrize("op,bounds", [("s", (8, 7, 8, 7, 8, 7, 2, 2)), ("p", (8, 8, 8, 8)),
                                       ("u", (7, 4, 4, 7, 6, 7, 7, 6))])
def test_sums(run, op, bounds):
    rng = random.Random(6)
    pools = [operands(Q_MOD, k, rng) for k in bounds]
    cases = [[p[0] for p in pools], [p[1] for p in pools], [p[-1] for p in pools]]
    cases += [[rng.choice(p) for p in pools] for _ in range(400)]
    # The sums' extremes of either sign.
    z = [0] * 9
    if op == "s":
        cases += [[p[i] for p in pools[:4]] + [z] * 4 for i in (0, 1, -1)]
        cases += [[z] * 4 + [p[i] for p in pools[4:]] for i in (0, 1, -1)]
    for c, r in zip(cases, run([(op, c) for c in cases])):
        v = [value(x) for x in c]
        want = v[0] * v[1] + v[2] * v[3]
        if op == "s":
            want -= v[4] * v[5] + v[6] * v[7]
        if op == "u":
            want += v[4] * v[5] + v[6] * v[7]
        got = value(r)
        assert all(x < 2**29 for x in r)
        assert got < 2 * Q_MOD and (got * 2**261 - want) % Q_MOD == 0


def column_bound(m, products, limb, top):
    """The largest any column of a sum of so many products gets in the reduction, where every
    dropped low word is 2^32 - 1 and every digit 2^29 - 1."""
    w = limbs(pow(2, -29, m) + (2 * m if m == Q_MOD else 0))
    op = [limb] * 8 + [top]
    t = [0] * 18
    for i in range(9):
        for j in range(9):
            t[i + j] += products * op[i] * op[j]
    most = max(t)
    for i in range(9):
        if i < 7:
            t[i + 1] += 8 * (t[i] >> 32)
            for j in range(9):
                t[i + 1 + j] += (2**32 - 1) * w[j]
        else:
            for j in range(9):
                t[i + j] += (2**29 - 1) * limbs(m)[j]
            t[i + 1] += t[i] >> 29
        most = max(most, max(t))
    return most


def test_column_bounds():
    limb, top = 2**29 + 7, 2**26
    assert column_bound(Q_MOD, 1, limb, top) < 22.0 * 2**58
    assert 2**63 < column_bound(R_MOD, 1, limb, top) < 37.2 * 2**58  # unsigned, below 2^64
    assert column_bound(Q_MOD, 2, limb, top) < 31.4 * 2**58          # redc29: signed
    assert column_bound(Q_MOD, 4, limb, top) < 51.3 * 2**58          # redc29u
    assert column_bound(R_MOD, 2, limb, top) > 2**63                 # not redc29's


@pytest.mark.parametrize("call", ["redc29", "redc29u"])
def test_lazy_reductions_refuse_large_limbs(tmp_path, call):
    header = os.path.join(HERE, "..", "snarkrs_amd", "csrc", "bn254.cuh")
    for field, fits in (("Fq29", True), ("Fr29", False)):
        src = tmp_path / "reduce.cpp"
        src.write_text(f'#include "{header}"\nusing namespace g16;\n'
                       f"void f(uint64_t* t, uint32_t* r) {{ {call}<{field}>(t, r); }}\n")
        r = subprocess.run([HIPCC, "-std=c++17", "--cuda-host-only", "-x", "hip", "-fsyntax-only",
                            str(src)], capture_output=True, text=True, timeout=300)
        assert (r.returncode == 0) == fits, r.stderr
        assert fits or "static assertion failed" in r.stderr


def test_pack(run):
    rng = random.Random(7)
    xs = operands(Q_MOD, 9, rng)
    xs += [limbs(k * Q_MOD + d) for k in range(9) for d in (0, 1)]
    xs += [limbs(k * Q_MOD - 1) for k in range(1, 10)]
    for x, r in zip(xs, run([("x", [x]) for x in xs])):
        got = sum(w << (32 * j) for j, w in enumerate(r))
        assert got < 5 * Q_MOD and (got - value(x)) % Q_MOD == 0
