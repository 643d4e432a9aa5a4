"""The lvl1 rotations at the edges of their workgroup widths: counts that fill
no workgroup, exactly one round, or one job more (FFT backend, key bundle and
CMUX keys); the lvl2 key-bundle rotation against the two-wave kernel."""
import numpy as np
import pytest

import cufhe_amd as C
import oracle as O
from conftest import load_lvl1_keys

pytestmark = pytest.mark.gpu

MOST = 1537


@pytest.fixture(scope="module", params=[True, False], ids=["bundle", "cmux"])
def rotations(request, keys_lvl1):
    """MOST random lvl0 samples, some with masks that round to 0, N and 2N - 1,
    and their rotations by the one-job workgroups."""
    kb = request.param
    C.check(C.lib().cufhe_initialize(), "initialize")
    bk = keys_lvl1["bk_kb" if kb else "bk"]
    load_lvl1_keys(("fft", kb), bk, keys_lvl1["ksk"], backend=C.BACKEND_FFT,
                   variant=C.BR_KEY_BUNDLE if kb else C.BR_PLAIN)
    rng = np.random.default_rng(61)
    tl0 = rng.integers(0, 2**32, (MOST, 637), dtype=np.uint64).astype(np.uint32)
    tl0[0] = 0
    tl0[1] = np.uint32(1 << 31)
    tl0[2] = np.uint32(0xFFFFFFFF)
    return kb, bk, tl0, _run(tl0, 1)


def _run(tl0, c):
    din = C.DeviceBuffer.from_numpy(tl0)
    dout = C.DeviceBuffer(tl0.shape[0] * C.TLWE1_WORDS * 4)
    C.check(C.lib().cufhe_bootstrap_lvl01(dout.ptr, din.ptr, C.MU1, tl0.shape[0], c, None), "bootstrap")
    return dout.download(np.uint32, (tl0.shape[0], C.TLWE1_WORDS))


def test_one_job_workgroups_equal_the_exact_oracle(rotations):
    # integers: the FP64 product is within a small fraction of a unit of them
    kb, bk, tl0, out = rotations
    for i in (0, 1, 2, 3, 1026, MOST - 1):
        acc = O.blind_rotate(1, O.EXACT, kb, tl0[i], bk, C.MU1)
        assert np.array_equal(out[i], O.sample_extract(1, acc)), i


@pytest.mark.parametrize("c", [0, 2, 4])
# 1281 to 1536: with the key bundle, two jobs per workgroup behind full rounds of four
@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 256, 257, 512, 513, 1024, 1027, 1281, 1300, 1536, MOST])
def test_widths_agree(rotations, c, n):
    _, _, tl0, out = rotations
    assert np.array_equal(_run(tl0[:n], c), out[:n])


# 25 workgroups are the fewest that read the key ahead; 259 leave three, and 300
# leave 44 of 256 CUs for a second round
@pytest.mark.parametrize("n", [24, 25, 259, 300])
def test_lvl2_bundle_equals_the_two_wave_kernel(keys_lvl2, n):
    """Every bit: both forms do the same operations in the same order."""
    C.check(C.lib().cufhe_initialize(), "initialize")
    C.initialize_lvl02(keys_lvl2["bk_kb"], keys_lvl2["ksk"])
    rng = np.random.default_rng(62)
    tl0 = rng.integers(0, 2**32, (n, 637), dtype=np.uint64).astype(np.uint32)
    tl0[0] = 0
    tl0[1] = np.uint32(1 << 31)
    tl0[2] = np.uint32(0xFFFFFFFF)
    din = C.DeviceBuffer.from_numpy(tl0)
    out = {}
    try:
        for c in (1, 2):
            C.check(C.lib().cufhe_set_lvl2_jobs_per_group(c), "jobs per group")
            dout = C.DeviceBuffer(n * C.TLWE2_WORDS * 8)
            C.check(C.lib().cufhe_bootstrap_lvl02(dout.ptr, din.ptr, C.MU2, n, None), "bootstrap")
            out[c] = dout.download(np.uint64, (n, C.TLWE2_WORDS))
    finally:
        C.check(C.lib().cufhe_set_lvl2_jobs_per_group(1), "jobs per group")
    assert np.array_equal(out[1], out[2])
