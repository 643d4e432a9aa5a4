"""The library's rotation autotuner (cufhe_autotune_lvl1): it times every
valid jobs-per-workgroup choice for the loaded keys, plans created with
jobs_per_group 0 use its pick for their batch size, every choice computes
the same ciphertexts, and a key load clears the record."""
import numpy as np
import pytest

import conftest
import cufhe_amd as C
from conftest import load_lvl1_keys

pytestmark = pytest.mark.gpu


def test_autotune_picks_a_valid_kernel_and_plans_use_it(keys_lvl1):
    C.check(C.lib().cufhe_initialize(), "initialize")
    conftest._LOADED_LVL1["tag"] = None
    load_lvl1_keys(("fft", True), keys_lvl1["bk_kb"], keys_lvl1["ksk"],
                   backend=C.BACKEND_FFT, variant=C.BR_KEY_BUNDLE)
    n = 600
    best, times = C.autotune_lvl1(n)
    assert best in times and set(times) <= {1, 2, 4, 6, 8} and len(times) >= 4
    assert times[best] == min(times.values())
    rng = np.random.default_rng(31)
    ops = ["NAND", "XOR", "AND", "OR", "XNOR", "NOR"]
    names = [ops[i] for i in rng.integers(0, len(ops), n)]
    bits = rng.integers(0, 2, 2 * n).astype(np.uint8)
    pool = np.zeros((3 * n, C.TLWE1_WORDS), np.uint32)
    pool[: 2 * n] = C.encrypt_bits(1, 32, keys_lvl1["k1"], bits)
    gates = [(names[i], 2 * n + i, i, n + i, 0) for i in range(n)]
    outs = {}
    for c in (0, 1):
        d = C.DeviceBuffer.from_numpy(pool)
        plan = C.Plan(gates, d, jobs_per_group=c)
        if c == 0:
            assert plan.jobs_per_group == best
        plan.run()
        C.check(C.lib().cufhe_synchronize(), "sync")
        outs[c] = d.download(np.uint32, pool.shape)[2 * n:]
        plan.destroy()
    assert np.array_equal(outs[0], outs[1])
    want = [C.TRUTH[o](int(bits[i]), int(bits[n + i])) for i, o in enumerate(names)]
    assert list(C.decrypt_bits(1, keys_lvl1["k1"], outs[0])) == want
    # a key load clears the record: the built-in choice (8)
    conftest._LOADED_LVL1["tag"] = None
    load_lvl1_keys(("fft", True), keys_lvl1["bk_kb"], keys_lvl1["ksk"],
                   backend=C.BACKEND_FFT, variant=C.BR_KEY_BUNDLE)
    d = C.DeviceBuffer.from_numpy(pool)
    plan = C.Plan(gates, d, jobs_per_group=0)
    assert plan.jobs_per_group == 8
    plan.destroy()


@pytest.mark.parametrize("bundle", [True, False], ids=["bundle", "cmux"])
def test_same_launches_tie_and_small_plans_keep_the_mix(keys_lvl1, bundle):
    """At a whole number of rounds a fixed width is the default's launch: they get one
    time, the default is recorded, and smaller plans are not held to a fixed width."""
    C.check(C.lib().cufhe_initialize(), "initialize")
    conftest._LOADED_LVL1["tag"] = None
    load_lvl1_keys(("fft", bundle), keys_lvl1["bk_kb" if bundle else "bk"], keys_lvl1["ksk"],
                   backend=C.BACKEND_FFT, variant=C.BR_KEY_BUNDLE if bundle else C.BR_PLAIN)
    cus = 256
    d = C.DeviceBuffer(3 * C.TLWE1_WORDS * 4)
    for n, same in ((2 * cus, 2), (4 * cus, 4 if bundle else 2), (16 * cus, 4)):
        best, times = C.autotune_lvl1(n)
        assert times[8] == times[same] and times.get(6, times[8]) == times[8], (n, times)
        assert best == 8, (n, times)
        plan = C.Plan([("NAND", 2, 0, 1, 0)], d)
        assert plan.jobs_per_group == 8
        plan.destroy()


@pytest.mark.parametrize("bundle, counts", [
    (True, {(4096, 4): 1024, (4096, 8): 1024, (4096, 0): 1024, (4096, 2): 2048, (150, 8): 150, (1100, 6): 332}),
    (False, {(4096, 4): 2048, (4096, 1): 4096, (600, 8): 344}),
], ids=["bundle", "cmux"])
def test_rotation_workgroups_are_the_launched_ones(keys_lvl1, bundle, counts):
    C.check(C.lib().cufhe_initialize(), "initialize")
    conftest._LOADED_LVL1["tag"] = None
    load_lvl1_keys(("fft", bundle), keys_lvl1["bk_kb" if bundle else "bk"], keys_lvl1["ksk"],
                   backend=C.BACKEND_FFT, variant=C.BR_KEY_BUNDLE if bundle else C.BR_PLAIN)
    for (n, c), groups in counts.items():
        assert C.lib().cufhe_rotation_workgroups_lvl1(n, c) == groups, (n, c)
    assert C.lib().cufhe_rotation_workgroups_lvl1(10, 3) < 0
