"""Lanes of an item where the caller's window cuts the set into thousands of
items of a few sessions each."""
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from test_gpu_shapes import check, sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}
_set = []


def small_queries():
    if not _set:
        _set.extend(sessions([9] * 20_000, 50, 12))
    return _set


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
@pytest.mark.parametrize("window", [32, 128, 512])
def test_small_windows_match_the_oracle(model, window):
    train, n_qd = small_queries()
    print(f"case small windows model={IDS[model]} window={window}", flush=True)
    check(model, train, n_qd, item_window=window)


@pytest.mark.parametrize("model", [DBN, CCM], ids=["DBN", "CCM"])
def test_a_window_of_64_does_not_take_512_lanes(model):
    """At most 1.3 times the iteration with 128 lanes an item: with 512 lanes,
    most of which have no session, it takes 1.8 to 2 times."""
    train, n_qd = small_queries()
    us = []
    for opts in (dict(block=128), {}):
        with ClickModel(model, item_window=64, **opts) as cm:
            cm.init_parameters(train, n_qd)
            us.append(min(cm.em_graph_timed(20) for _ in range(6)) / 20 * 1e3)
    print(f"case lanes of small windows model={IDS[model]}: 128 lanes {us[0]:.1f} us, chosen {us[1]:.1f} us", flush=True)
    assert us[1] <= 1.3 * us[0], us
