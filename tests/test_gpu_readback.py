"""Tables read back through pinned chunks: sizes around the chunk sizes, the
number of chunks and the size from which threads copy.  Values come back
bit for bit; denominators after an M-step are the constants that follow from
the counts (whole numbers, exact)."""
import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from massiveclicks_amd.model import SessionSet

pytestmark = pytest.mark.gpu

N = 40
# Entries: one chunk of 256 KB holds 65,536, eight of 1 MB 2,097,152.
SIZES = [400, 65_536, 65_537, 262_144, 524_289, 2_097_151, 2_097_152, 3_000_001]


@pytest.mark.parametrize("model", [PBM, UBM, DBN, CCM], ids=["PBM", "UBM", "DBN", "CCM"])
def test_tables_come_back_whole(model):
    rng = np.random.default_rng(model)
    pidx = np.arange(N * 10, dtype=np.int32).reshape(N, 10)
    clicks = (rng.random((N, 10)) < 0.3).astype(np.uint8)
    train = SessionSet(np.arange(N, dtype=np.int32), np.zeros((N, 10), np.int32), clicks, pidx)
    for n_qd in SIZES:
        print(f"case readback model={model} n_qd={n_qd}", flush=True)
        with ClickModel(model) as cm:
            cm.init_parameters(train, n_qd)
            tabs = [[(rng.random(size) + 1).astype(np.float32), (rng.random(size) + 3).astype(np.float32)]
                    for _, _, size in cm.get_parameter_information()]
            for t, (num, den) in enumerate(tabs):
                cm.set_parameters(t, num, den)
            for t, (num, den) in enumerate(tabs):
                got = cm.get_parameters(t)
                np.testing.assert_array_equal(got[0], num)
                np.testing.assert_array_equal(got[1], den)
            cm.em(1)
            occ, clk = np.zeros(n_qd, np.float32), np.zeros(n_qd, np.float32)
            occ[:N * 10], clk[:N * 10] = 1, clicks.reshape(-1)
            want = 2 + occ + clk if model == CCM else 2 + occ
            np.testing.assert_array_equal(cm.get_parameters(0)[1], want)
            if model == DBN:
                np.testing.assert_array_equal(cm.get_parameters(1)[1], 2 + 2 * occ - clk)
