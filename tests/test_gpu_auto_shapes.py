"""Work-item shapes that the planner chooses by itself, at sizes where its
rules change: a little over a million sessions (wider item windows, and windows
of their own for queries wider still) and small uneven DBN sets.

Bar: parameters within 1e-5 of the oracle with FP64 sums, bit-identical to the
run with a separate merge kernel."""
import os

import numpy as np
import pytest

import oracle
from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from massiveclicks_amd.model import SessionSet
from test_gpu_shapes import TOL_PARAM, check, sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}
ITERS = 5
_big = []


def large_set():
    """1,002,800 sessions: 100,000 queries of 20 documents, the first sliced,
    and one of 2,200 documents, more than any item window."""
    if not _big:
        a, na = sessions([22_000] + [9] * 99_999 + [80_009], 20, 1)
        b, nb = sessions([800], 2200, 2)
        assert nb > 2048
        _big.append((SessionSet(np.concatenate([a.query, b.query + 200_000]).astype(np.int32),
                                np.concatenate([a.docs, b.docs]), np.concatenate([a.clicks, b.clicks]),
                                np.concatenate([a.pidx, b.pidx + na]).astype(np.int32)), na + nb))
    return _big[0]


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
def test_a_million_sessions_and_a_wide_query(model):
    train, n_qd = large_set()
    assert len(train) > 1_000_000
    print(f"case automatic shape model={IDS[model]} n={len(train)} entries={n_qd}", flush=True)
    om = oracle.OracleModel(model, train.query, train.pidx, train.clicks, n_qd, accum_fp64=True,
                            n_threads=max(1, min(os.cpu_count() or 1, 16)))
    om.iterate(ITERS)
    with ClickModel(model) as a, ClickModel(model, fused_merge=False) as b:
        for cm in (a, b):
            cm.init_parameters(train, n_qd)
            cm.em(ITERS - 2)
            cm.em(2, use_graph=False)
        assert a.stream_info()["n_window_sessions"] == len(train)   # no item without a window
        for t in range(a.n_tables()):
            num, den = a.get_parameters(t)
            np.testing.assert_array_equal(num, b.get_parameters(t)[0])
            np.testing.assert_array_equal(a.get_values(t), b.get_values(t))
            err = float(np.max(np.abs(a.get_values(t) - om.get_table(t)[2])))
            assert err < TOL_PARAM, f"{a.layout_info()} table {t}: {err}"


@pytest.mark.parametrize("sizes", [[700] * 4 + [30] * 60, [5600]], ids=["64-queries", "one-query"])
def test_small_uneven_dbn_items(sizes):
    train, n_qd = sessions(sizes, 24, 6, uneven=True)
    print(f"case small uneven DBN queries={len(sizes)}", flush=True)
    lay = check(DBN, train, n_qd)
    assert 256 < lay["max_item_sessions"] <= 512, lay
