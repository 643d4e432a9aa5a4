"""The NTT-backend rotation at the edges of its shares of jobs: counts that leave
CUs idle, fill rounds exactly, or make shares of two sizes, with every
jobs_per_group; every word against workgroups of one job, and those against the
oracle."""
import numpy as np
import pytest

import cufhe_amd as C
import oracle as O
from conftest import load_lvl1_keys

pytestmark = pytest.mark.gpu

MODES = {"plain": (C.BR_PLAIN, O.BR_PLAIN), "kb": (C.BR_KEY_BUNDLE, O.BR_KB),
         "bb": (C.BR_BLOCK_BINARY, O.BR_BB)}
MOST = 2305


ALONE = 100  # jobs of a batch whose workgroups have one job each


def _run(tl0, c):
    din = C.DeviceBuffer.from_numpy(tl0)
    dout = C.DeviceBuffer(tl0.shape[0] * C.TLWE1_WORDS * 4)
    C.check(C.lib().cufhe_bootstrap_lvl01(dout.ptr, din.ptr, C.MU1, tl0.shape[0], c, None), "bootstrap")
    return dout.download(np.uint32, (tl0.shape[0], C.TLWE1_WORDS))


@pytest.fixture(scope="module", params=list(MODES))
def rotations(request, keys_lvl1, keys_bb):
    name = request.param
    variant, mode = MODES[name]
    C.check(C.lib().cufhe_initialize(), "initialize")
    bk = {"plain": keys_lvl1["bk"], "kb": keys_lvl1["bk_kb"], "bb": keys_bb["bk"]}[name]
    ksk = keys_bb["ksk_subset"] if name == "bb" else keys_lvl1["ksk"]
    load_lvl1_keys(("ntt", name), bk, ksk, backend=C.BACKEND_NTT, variant=variant, subset=name == "bb")
    rng = np.random.default_rng(71)
    tl0 = rng.integers(0, 2**32, (MOST, 637), dtype=np.uint64).astype(np.uint32)
    # masks that round to 0, N and 2N - 1: roots 0, -2 and psi^-(2k+1) - 1
    tl0[0] = 0
    tl0[1] = np.uint32(1 << 31)
    tl0[2] = np.uint32(0xFFFFFFFF)
    alone = [_run(tl0[i:i + ALONE], 1) for i in range(0, MOST, ALONE)]
    return mode, bk, tl0, np.concatenate(alone)


def test_one_job_workgroups_equal_the_oracle(rotations):
    mode, bk, tl0, out = rotations
    for i in (0, 1, 2, 3, MOST - 1):
        acc = O.blind_rotate(1, O.NTT, mode, tl0[i], bk, C.MU1)
        assert np.array_equal(out[i], O.sample_extract(1, acc)), i


@pytest.mark.parametrize("c", [0, 1, 2, 6])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 513, 2047, 2048, 2049, MOST])
def test_shares_agree(rotations, c, n):
    _, _, tl0, out = rotations
    assert np.array_equal(_run(tl0[:n], c), out[:n])
