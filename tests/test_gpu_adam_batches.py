"""Adam epochs replayed from a graph when a query holds several minibatches'
sessions: the minibatches behind it are empty, at the middle or the end of an
epoch, one or more in a row.

Bar: logits bit-identical to steps launched one by one, whose merges run in
every step."""
import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel
from test_gpu_shapes import sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
@pytest.mark.parametrize("sizes,batches,empty", [([4000] + [30] * 50, 6, [1, 2, 3]),
                                                 ([300] + [50] * 30 + [4200], 6, [2, 3, 4, 5]),
                                                 ([40] * 30 + [3400] + [40] * 30, 7, [2, 3, 4]),
                                                 ([2000, 3000], 4, [2, 3]), ([3500] + [30] * 50, 4, [1]),
                                                 ([5000], 3, [1, 2])],
                         ids=["first", "last", "middle", "two", "one", "only"])
@pytest.mark.parametrize("opts", [{}, {"item_sessions": 256, "item_window": 16}], ids=["window", "global"])
def test_epoch_with_empty_minibatches(model, sizes, batches, empty, opts):
    train, n_qd = sessions(sizes, 24, sum(sizes))
    print(f"case empty minibatches model={IDS[model]} batches={batches} {opts}", flush=True)
    # The first session of a query's run places the whole run.
    first = np.searchsorted(train.query, np.unique(train.query))
    used = set(np.minimum(batches - 1, first * batches // len(train)).tolist())
    assert [b for b in range(batches) if b not in used] == empty
    got = []
    for use_graph in (True, False):
        with ClickModel(model, batches=batches, **opts) as cm:
            cm.init_parameters(train, n_qd)
            cm.grad_init()
            cm.adam_configure(lr=0.05)
            for _ in range(3):
                cm.adam_steps(batches, use_graph=use_graph)
            cm.adam_steps(2 * batches, use_graph=use_graph)
            got.append([cm.get_logits(t) for t in range(cm.n_tables())]
                       + [cm.get_values(t) for t in range(cm.n_tables())])
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
