"""Buckets around the merge's limits (one segment, a few, past the span that goes to the heavy
path, several heavy tasks), where every entry of a window falls in one bucket, over distinct,
equal and opposite bases: the tail's additions, doublings and cancellations on points spread over
lanes, against the closed form (sum k_i s) G."""
import pytest

from snarkrs_amd.wire import R_MOD, SplitMix64, fr_array

pytestmark = pytest.mark.gpu

SIZES = [1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 72, 73, 255, 256, 257, 287, 288, 289, 320, 321, 361,
         1999, 8192 + 33]


@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("kind", ["distinct", "equal", "opposite"])
def test_one_bucket_per_window(dev, group, kind):
    rng = SplitMix64(900 + group)
    for n in SIZES:
        k0 = rng.next_fr()
        if kind == "distinct":
            ks = [rng.next_fr() for _ in range(n)]
        elif kind == "equal":
            ks = [k0] * n
        else:
            ks = [k0 if i % 2 else R_MOD - k0 for i in range(n)]
        s = rng.next_fr() if n % 2 else 1 + n % 5
        bases = dev.fixed_base(group, fr_array(ks))
        got = dev.msm(group, bases, fr_array([s] * n))
        total = sum(ks) * s % R_MOD
        assert (got == dev.fixed_base(group, fr_array([total]))[0]).all(), (n, s)
