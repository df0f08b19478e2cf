"""The shape that the planner chooses by itself as a candidate of the
autotuner, on a set of queries wider than an item window: the only shape that
keeps their sums in LDS."""
import json

import pytest

from massiveclicks_amd import PBM, UBM, ClickModel, autotune
from massiveclicks_amd._lib import MCError
from massiveclicks_amd.model import AUTO, TUNE_VERSION
from test_gpu_shapes import check, sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM"}
_set = []


def wide_set():
    if not _set:
        _set.extend(sessions([3000] * 20, 2400, 5))
    return _set


def ms_per_iteration(model, train, n_qd, opts):
    with ClickModel(model, **opts) as cm:
        cm.init_parameters(train, n_qd)
        return min(cm.em_graph_timed(20) for _ in range(5)) / 20


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
@pytest.mark.parametrize("start", [None, {"item_sessions": 8192, "item_window": 1280, "block": 256}],
                         ids=["automatic", "fixed"])
def test_tuned_is_no_slower_than_untuned(model, start):
    """At most 1.4 times the untuned iteration, for noise: without the
    planner's shape the fastest candidate takes 1.9 to 2.1 times as long."""
    train, n_qd = wide_set()
    print(f"case tuned against untuned model={IDS[model]} start={start}", flush=True)
    opts, info = autotune(model, train, n_qd, iterations=20, start=start)
    tuned, untuned = ms_per_iteration(model, train, n_qd, opts), ms_per_iteration(model, train, n_qd, {})
    print(f"  tuned {tuned * 1e3:.1f} us, untuned {untuned * 1e3:.1f} us, {opts}", flush=True)
    assert tuned <= 1.4 * untuned, (tuned, untuned, opts, info)
    assert opts["item_sessions"] >= 64 and opts["block"] in (256, 512)


def test_automatic_values_are_the_defaults():
    train, n_qd = sessions([900] * 8 + [40] * 200, 1400, 3)
    print("case automatic values", flush=True)
    auto = dict(item_sessions=AUTO, item_window=AUTO, block=AUTO)
    with ClickModel(UBM) as a, ClickModel(UBM, **auto) as b, ClickModel(UBM, item_sessions=64, item_window=64) as c:
        for cm in (a, b, c):
            cm.init_parameters(train, n_qd)
        assert a.layout_info() == b.layout_info() != c.layout_info()
        assert a.stream_info() == b.stream_info() and a.get_memory_usage() == b.get_memory_usage()
    check(UBM, train, n_qd, **auto)
    for bad in ({"item_sessions": -2}, {"item_window": -2}, {"block": -2}, {"item_sessions": 0}, {"block": 0}):
        with pytest.raises(MCError):
            ClickModel(UBM, **bad)


def test_results_of_other_versions_are_not_reused(tmp_path):
    train, n_qd = sessions([50] * 40, 24, 9)
    print("case cache of another version", flush=True)
    cache = str(tmp_path / "tune.json")
    old = {"PBM:2000:%d:0" % n_qd: {"options": {"item_sessions": 64}, "ms_per_iter": 0.0, "trials": 9}}
    with open(cache, "w") as f:
        json.dump(old, f)
    opts, info = autotune(PBM, train, n_qd, iterations=3, cache=cache)
    assert not info["cached"] and info["ms_per_iter"] > 0
    assert autotune(PBM, train, n_qd, iterations=3, cache=cache) == (opts, dict(info, cached=True))
    assert len(json.load(open(cache))) == 2 and any(k.endswith(f":v{TUNE_VERSION}") for k in json.load(open(cache)))
