"""The framework's timed workloads: what a prover service has it do, over the range of sizes it
meets, through the package's public entry points.

Kinds of case:

* ``prove``  one Groth16 proof of a fresh witness against a resident key: witness in host memory
  (a command-line or service call) or already in HBM; uniform witnesses or 40 % boolean ones;
  variable-work MSMs or the opt-in constant-work ones;
* ``batch``  several proofs of one circuit in one call (a prover that keeps a queue);
* ``msm``    a standalone multi-scalar multiplication, G1 or G2 (ceremony and setup work), on
  resident inputs or on host slices, 30 % of the scalars in {0, 1};
* ``ntt``    polynomial transforms over Fr: a forward and an inverse transform of a resident
  vector (both directions, in place), or one forward transform of a host vector.

Every output is a whole point, proof or vector in the wire format (bytes), so results are exact.
"""
import math

import numpy as np
import torch

from snarkrs_amd import native, synth
from snarkrs_amd.devmem import DeviceArray

_devices = {}


def _device(constant=False):
    """One open GPU per setting, kept like a service keeps it."""
    if constant not in _devices:
        dev = native.Device(0)
        if constant:
            dev.set_constant_work(True)
        _devices[constant] = dev
    return _devices[constant]


def _prove(name, n, bits, device, constant=False):
    return {"name": name, "kind": "prove", "n": n, "bits": bits, "device": device,
            "constant": constant}


def listed():
    return [
        # The smallest circuits (a login or membership proof): latency of one call.
        _prove("prove_1000", 1000, 400, False),
        # A small application circuit, the lower end of the mixed batch and serving traffic.
        _prove("prove_22k", 22_027, 400, False),
        # The plain-prove size, a multiplication chain with a uniform witness already in HBM.
        _prove("prove_65536_resident", 1 << 16, 0, True),
        # The headline: 1.1 million constraints, 40 % boolean witness, from host memory.
        _prove("prove_1100k", 1_100_000, 400, False),
        # The same call with constant-work MSMs, for witnesses whose sparsity must not show.
        _prove("prove_131k_constant", 131_072, 400, False, True),
        # A queue of sixteen requests against one small circuit, proved in one call.
        {"name": "batch_16x26k", "kind": "batch", "n": 26_001, "bits": 400, "count": 16},
        # Standalone MSMs on resident inputs at the published benchmark sizes ...
        {"name": "msm_g1_2_20", "kind": "msm", "group": 1, "n": 1 << 20, "device": True},
        {"name": "msm_g2_2_18", "kind": "msm", "group": 2, "n": 1 << 18, "device": True},
        # ... and short odd ones on host slices, as a setup's per-contribution checks make them.
        {"name": "msm_g1_4099_host", "kind": "msm", "group": 1, "n": 4099, "device": False},
        {"name": "msm_g2_1021_host", "kind": "msm", "group": 2, "n": 1021, "device": False},
        # Transforms: both directions of the headline's domain in HBM, and a short host vector.
        {"name": "ntt_2_21_roundtrip", "kind": "ntt", "log_n": 21, "device": True},
        {"name": "ntt_2_13_host", "kind": "ntt", "log_n": 13, "device": False},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prove", "prove", "constant", "batch", "msm", "msm", "ntt"])
    if kind in ("prove", "constant"):
        constant = kind == "constant"
        return {"kind": "prove", "n": _log_uniform(rng, 900, 200_000 if constant else 1_000_000),
                "bits": rng.choice([0, 400, 400]), "device": rng.random() < 0.4,
                "constant": constant}
    if kind == "batch":
        return {"kind": "batch", "n": _log_uniform(rng, 4000, 60_000), "bits": 400,
                "count": rng.randint(3, 17)}
    if kind == "msm":
        group = rng.choice([1, 2])
        device = rng.random() < 0.6
        top = (1 << 20 if group == 1 else 1 << 18) if device else 1 << 15
        return {"kind": "msm", "group": group, "n": _log_uniform(rng, 500, top),
                "device": device}
    device = rng.random() < 0.6
    return {"kind": "ntt", "log_n": rng.randint(11, 21) if device else rng.randint(10, 16),
            "device": device}


def _workload(case, seed):
    n = case["n"]
    return synth.Workload(n_constraints=n, n_public=2, n_private_in=max(8, n // 11),
                          bool_permille=case["bits"], input_bool_permille=case["bits"],
                          seed=3 * seed + 21, setup_seed=3 * seed + 22,
                          witness_seed=3 * seed + 23)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prove", "batch"):
        dev = _device(case.get("constant", False))
        syn = synth.Synth(_workload(case, seed))
        key, wit = syn.key(dev)
        count = case.get("count", 1)
        wits = [wit] + [syn.witness(1000 * seed + 31 + i) for i in range(1, count)]
        syn.close()
        blind = synth.scalars(1000 * seed + 7, 2 * count, 0)
        circ = dev.prepare(key)
        if kind == "batch":
            return {"circ": circ,
                    "items": [(circ, w, blind[2 * i], blind[2 * i + 1])
                              for i, w in enumerate(wits)]}
        return {"circ": circ, "wit": DeviceArray(wit) if case["device"] else wit,
                "n_vars": len(wit), "r": blind[0], "s": blind[1]}
    dev = _device()
    if kind == "msm":
        n, group = case["n"], case["group"]
        bases = dev.fixed_base(group, synth.scalars(1000 * seed + 41, n, 0))
        scalars = synth.scalars(1000 * seed + 42, n, 300)
        if case["device"]:
            bases, scalars = DeviceArray(bases), DeviceArray(scalars)
        return {"bases": bases, "scalars": scalars}
    data = synth.scalars(1000 * seed + 51, 1 << case["log_n"], 0)
    if case["device"]:
        data = torch.from_numpy(data).cuda()
        torch.cuda.synchronize()  # the library transforms on a stream of its own
    return {"data": data}


def run(state):
    if "items" in state:
        return native.prove_batch(state["items"])
    if "circ" in state:
        circ, wit = state["circ"], state["wit"]
        if isinstance(wit, DeviceArray):
            return circ.prove_with_blinders_device(wit.addr, state["n_vars"], state["r"],
                                                   state["s"])
        return circ.prove_with_blinders(wit, state["r"], state["s"])
    dev = _device()
    if "scalars" in state:
        bases, scalars = state["bases"], state["scalars"]
        if isinstance(bases, DeviceArray):
            n = scalars.nbytes // 32
            return dev.msm_device(1 if bases.nbytes == 64 * n else 2, bases.addr, scalars.addr, n)
        return dev.msm(bases.shape[1] // 64, bases, scalars)
    data = state["data"]
    if isinstance(data, torch.Tensor):
        log_n = data.shape[0].bit_length() - 1
        dev.ntt_device(data.data_ptr(), log_n, 0)
        dev.ntt_device(data.data_ptr(), log_n, 1)
        return data
    return dev.ntt(data, 0)


# One Fq or Fr product is 64 32x32-bit multiply-adds for the product and 64 for its reduction;
# a multiply-add counts as two operations.
_PRODUCT = 2 * 128


def _msm_work(group, n):
    """A bucket method's additions at 16-bit windows, each the six products of an affine addition
    with a shared inversion (G2: three base products per product)."""
    return 16 * n * 6 * _PRODUCT * (1 if group == 1 else 3)


def _ntt_work(log_n):
    return (log_n << log_n >> 1) * _PRODUCT


def work(case):
    """What one pass cannot do without: each input read once, each output written once."""
    kind = case["kind"]
    if kind == "msm":
        n, g = case["n"], case["group"]
        return {"bytes": n * (32 + 64 * g) + 64 * g, "flops": _msm_work(g, n)}
    if kind == "ntt":
        transforms = 2 if case["device"] else 1
        return {"bytes": transforms * 64 << case["log_n"],
                "flops": transforms * _ntt_work(case["log_n"])}
    n = case["n"]
    n_vars = n + max(8, n // 11) + 3
    log_d = (n + 2).bit_length()
    domain = 1 << log_d
    count = case.get("count", 1)
    # Four G1 and one G2 base vector, two matrices of three terms a row, the coset's tables.
    key = n_vars * (3 * 64 + 128) + 64 * domain + 2 * 3 * n * 40 + 3 * 32 * domain
    proof = 32 * n_vars + 256
    flops = (3 * _msm_work(1, n_vars) + _msm_work(2, n_vars) + _msm_work(1, domain)
             + 6 * _ntt_work(log_d))
    return {"bytes": key + count * proof, "flops": count * flops}


def exact(case, seed):
    """Outputs are whole points and field elements: compared byte for byte."""
    return None
