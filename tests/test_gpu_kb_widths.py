"""The key-bundle rotation at the edges of its workgroup widths: counts that fill
no workgroup, exactly one round, or one job more (FFT backend, lvl1)."""
import numpy as np
import pytest

import cufhe_amd as C
import oracle as O
from conftest import load_lvl1_keys

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rotations(keys_lvl1):
    """1027 random lvl0 samples, some with masks that round to 0, N and 2N - 1,
    and their rotations by the one-job workgroups."""
    C.check(C.lib().cufhe_initialize(), "initialize")
    load_lvl1_keys(("fft", True), keys_lvl1["bk_kb"], keys_lvl1["ksk"],
                   backend=C.BACKEND_FFT, variant=C.BR_KEY_BUNDLE)
    rng = np.random.default_rng(61)
    tl0 = rng.integers(0, 2**32, (1027, 637), dtype=np.uint64).astype(np.uint32)
    tl0[0] = 0
    tl0[1] = np.uint32(1 << 31)
    tl0[2] = np.uint32(0xFFFFFFFF)
    return tl0, _run(tl0, 1)


def _run(tl0, c):
    din = C.DeviceBuffer.from_numpy(tl0)
    dout = C.DeviceBuffer(tl0.shape[0] * C.TLWE1_WORDS * 4)
    C.check(C.lib().cufhe_bootstrap_lvl01(dout.ptr, din.ptr, C.MU1, tl0.shape[0], c, None), "bootstrap")
    return dout.download(np.uint32, (tl0.shape[0], C.TLWE1_WORDS))


def test_one_job_workgroups_equal_the_exact_oracle(rotations, keys_lvl1):
    # integers: the FP64 product is within a small fraction of a unit of them
    tl0, out = rotations
    for i in (0, 1, 2, 3, 1026):
        acc = O.blind_rotate(1, O.EXACT, True, tl0[i], keys_lvl1["bk_kb"], C.MU1)
        assert np.array_equal(out[i], O.sample_extract(1, acc)), i


@pytest.mark.parametrize("c", [0, 2, 4])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 256, 257, 512, 513, 1024, 1027])
def test_widths_agree(rotations, c, n):
    tl0, out = rotations
    assert np.array_equal(_run(tl0[:n], c), out[:n])
