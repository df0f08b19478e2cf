"""A model that is initialised again: every device buffer of the first training
set is gone, those that later calls allocate on first use among them."""
import numpy as np
import pytest

import oracle
from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from test_gpu_shapes import ITERS, TOL_PARAM, sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
def test_set_parameters_after_a_second_init(model):
    """Caller's denominators, held-out set, host evaluation, gradient and
    logits on a small set, a much larger one and the small one again: tables
    read back as they were set, and training from the start as the oracle's."""
    rng = np.random.default_rng(model)
    with ClickModel(model) as cm:
        for queries in (30, 4000, 30):
            train, n_qd = sessions([6] * queries, 20, queries)
            print(f"case second init model={IDS[model]} entries={n_qd}", flush=True)
            cm.init_parameters(train, n_qd)
            shapes = [size for _, _, size in cm.get_parameter_information()]
            for t, size in enumerate(shapes):
                num = rng.uniform(1, 5, size).astype(np.float32)
                den = num + rng.uniform(1, 5, size).astype(np.float32)
                cm.set_parameters(t, num, den)
                got = cm.get_parameters(t)
                np.testing.assert_array_equal(got[0], num)
                np.testing.assert_array_equal(got[1], den)
            cm.set_test_set(train)
            resident = cm.evaluate_test_set()
            assert cm.evaluate(train)["llh_sum"] == pytest.approx(resident["llh_sum"], rel=1e-6)
            cm.grad_init()
            assert all(np.isfinite(g).all() for g in cm.loglik_gradient()[1])
            cm.reset_parameters()
            cm.em(ITERS)
            om = oracle.OracleModel(model, train.query, train.pidx, train.clicks, n_qd, accum_fp64=True)
            om.iterate(ITERS)
            for t in range(cm.n_tables()):
                err = float(np.max(np.abs(cm.get_values(t) - om.get_table(t)[2])))
                assert err < TOL_PARAM, f"table {t}: {err}"
