"""Lanes per work item of the gradient kernels (256, 512 or 1024 by the items
of a launch and their sessions): every choice gives the same gradient and the
same Adam steps, and the choice keeps launches of a few items more than the
GPU has CUs from taking a second round."""
import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from test_gpu_shapes import sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}
# Items on both sides of the rules' lines (256 CUs: 256, 384 and 1024 items;
# 512 and 2048 sessions in the largest).
SHAPES = {"1100-items": dict(item_sessions=64), "290-items": dict(item_sessions=220),
          "90-items": dict(item_sessions=1024), "20-items": dict(item_sessions=1 << 20, item_window=5000)}


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
def test_gradient_and_adam_with_every_choice_of_lanes(model):
    """At the same logits: per-query gradients bit for bit (integer sums of the same terms), the
    shared ones up to the rounding of FP32 lane sums (1e-6 of the sum of the
    terms' magnitudes, bounded by the sessions' ranks); Adam from the graph as
    launched one by one."""
    train, n_qd = sessions([11] * 5500 + [3000], 20, 4)
    got, items = [], []
    for name, opts in SHAPES.items():
        print(f"case gradient lanes model={IDS[model]} {name}", flush=True)
        with ClickModel(model, **opts) as cm:
            cm.init_parameters(train, n_qd)
            cm.grad_init()
            rng = np.random.default_rng(model)
            for t, (_, _, size) in enumerate(cm.get_parameter_information()):
                cm.set_logits(t, rng.normal(0.0, 1.0, size).astype(np.float32))
            items.append(cm.layout_info()["n_items"])
            got.append(cm.loglik_gradient())
            logits = []
            for use_graph in (True, False):
                cm.reset_parameters()
                cm.grad_init()
                cm.adam_configure(lr=0.02)
                cm.adam_steps(3, use_graph=use_graph)
                logits.append([cm.get_logits(t) for t in range(cm.n_tables())])
            for a, b in zip(*logits):
                np.testing.assert_array_equal(a, b)
    assert items[0] >= 1024 > items[1] > 256 > items[2] > items[3], items
    for ll, grads in got[1:]:
        assert ll == pytest.approx(got[0][0], rel=1e-6)
        for a, b in zip(grads[:-1], got[0][1][:-1]):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_allclose(grads[-1], got[0][1][-1], rtol=1e-6, atol=1e-6 * 10 * len(train))


@pytest.mark.parametrize("model", [PBM, DBN, CCM], ids=["PBM", "DBN", "CCM"])
def test_a_few_items_more_than_cus_take_no_second_round(model):
    """Adam epochs of 264 against 240 items of 372 sessions: 1.1 times the
    sessions in at most 1.25 times the time.  With 1024 lanes, of which a CU
    holds one workgroup, it takes 1.35 times."""
    us = []
    for queries in (7440, 8184):
        train, n_qd = sessions([12] * queries, 20, 5)
        print(f"case second round model={IDS[model]} queries={queries}", flush=True)
        with ClickModel(model, item_sessions=372) as cm:
            cm.init_parameters(train, n_qd)
            assert cm.layout_info()["n_items"] == queries // 31
            cm.grad_init()
            cm.adam_configure(lr=0.01)
            us.append(min(cm.adam_steps_timed(8) for _ in range(10)) / 8 * 1e3)
    print(f"  us per epoch {us}", flush=True)
    assert us[1] <= 1.25 * us[0], us
