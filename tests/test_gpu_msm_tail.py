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


@pytest.mark.parametrize("group,n", [(1, 1021), (1, 4099), (2, 1021), (2, 5003)])
def test_least_scratch_runs_in_one_piece(dev, group, n):
    # A limit of exactly scratch_bytes holds the run (long segments); without one the same sum
    # comes from short segments.
    from snarkrs_amd.native import CeremonyMsm

    rng = SplitMix64(40 + n)
    ks = [rng.next_fr() for _ in range(n)]
    ss = [rng.next_fr() if i % 3 else i % 2 for i in range(n)]
    bases, scalars = dev.fixed_base(group, fr_array(ks)), fr_array(ss)
    want = dev.fixed_base(group, fr_array([sum(k * s for k, s in zip(ks, ss)) % R_MOD]))[0]
    lean = CeremonyMsm(dev, vram_limit=CeremonyMsm.scratch_bytes(group, n))
    for cer in (lean, CeremonyMsm(dev)):
        got = (cer.msm_g1 if group == 1 else cer.msm_g2)(bases, scalars)
        assert cer.last_runs() == 1
        assert (got == want).all()


@pytest.mark.parametrize("constant", [False, True])
@pytest.mark.parametrize("n", [1, 63, 762, 763, 1023, 1024, 1025, 4095, 4096, 4097, 6000])
def test_sort_of_small_msms(dev, n, constant):
    # The one-workgroup sort and the general one either side of their limit (762 points of 43
    # windows are its last) and of a round of threads, on boolean-heavy scalars (most entries in
    # one bucket).
    rng = SplitMix64(70 + n)
    ks = [rng.next_fr() for _ in range(n)]
    ss = [rng.next_fr() if i % 4 == 0 else i % 2 for i in range(n)]
    ss[0] = 0
    bases = dev.fixed_base(1, fr_array(ks))
    dev.set_constant_work(constant)
    try:
        got = dev.msm(1, bases, fr_array(ss))
    finally:
        dev.set_constant_work(False)
    total = sum(k * s for k, s in zip(ks, ss)) % R_MOD
    assert (got == dev.fixed_base(1, fr_array([total]))[0]).all()


@pytest.mark.parametrize("group,n", [(1, 33), (1, 1999), (1, 30011), (1, 65537), (2, 33),
                                     (2, 1999), (2, 20011)])
@pytest.mark.parametrize("same", [True, False])
def test_constant_work_runs(dev, group, n, same):
    # Runs that span several scan workgroups and fold groups (every scalar equal) or none, and the
    # branch-free reduction over mostly empty buckets.
    rng = SplitMix64(80 + n)
    ks = [rng.next_fr() for _ in range(257)]
    s0 = rng.next_fr()
    ss = [s0] * n if same else [rng.next_fr() for _ in range(n)]
    base = dev.fixed_base(group, fr_array(ks))
    bases = base[[i % 257 for i in range(n)]]
    dev.set_constant_work(True)
    try:
        got = dev.msm(group, bases, fr_array(ss))
    finally:
        dev.set_constant_work(False)
    total = sum(ks[i % 257] * s for i, s in enumerate(ss)) % R_MOD
    assert (got == dev.fixed_base(group, fr_array([total]))[0]).all()


@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("c", [2, 3, 4, 12, 13, 16])
@pytest.mark.parametrize("constant", [False, True])
def test_reduction_group_widths(dev, group, c, constant):
    # Windows either side of 2^16 buckets in all (groups of 4 and of 8), and windows of fewer
    # buckets than a group.
    from snarkrs_amd.devmem import DeviceArray

    n = 3001
    rng = SplitMix64(60 + c)
    ks = [rng.next_fr() for _ in range(n)]
    ss = [rng.next_fr() if i % 5 else i % 2 for i in range(n)]
    bases = DeviceArray(dev.fixed_base(group, fr_array(ks)))
    scalars = DeviceArray(fr_array(ss))
    dev.set_constant_work(constant)
    try:
        got = dev.msm_device(group, bases.addr, scalars.addr, n, c)
    finally:
        dev.set_constant_work(False)
    total = sum(k * s for k, s in zip(ks, ss)) % R_MOD
    assert (got == dev.fixed_base(group, fr_array([total]))[0]).all()


@pytest.mark.parametrize("group,n", [(1, 20480), (1, 20481), (2, 8192), (2, 8193)])
def test_segment_sums_over_lanes_and_not(dev, group, n):
    # Sixteen windows: the segments of the smaller n take 131072 lanes, the most that are spread,
    # and those of the next n one lane each.
    from snarkrs_amd.devmem import DeviceArray

    rng = SplitMix64(50 + n)
    ks = [rng.next_fr() for _ in range(257)]
    ss = [rng.next_fr() for _ in range(n)]
    base = dev.fixed_base(group, fr_array(ks))
    bases = DeviceArray(base[[i % 257 for i in range(n)]])
    got = dev.msm_device(group, bases.addr, DeviceArray(fr_array(ss)).addr, n, 16)
    total = sum(ks[i % 257] * s for i, s in enumerate(ss)) % R_MOD
    assert (got == dev.fixed_base(group, fr_array([total]))[0]).all()
