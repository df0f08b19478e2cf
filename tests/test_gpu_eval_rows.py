"""Session-major evaluation around its wavefront and block edges: the rows
of a wavefront pass through LDS, so partial wavefronts, a single block (whose
partials are the totals), the chunks that host arrays are cut into and arrays at
odd addresses are what can go wrong.

Bar: per-session values bit-identical to the resident set's kernels, which
share the per-session arithmetic; totals within 1e-6 relative (FP32 partials
over each lane's few sessions, a session's term is exact to 6e-8)."""
import ctypes as C

import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel, Dataset, _lib, synth
from massiveclicks_amd.model import SessionSet
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

NAMES = {PBM: "pbm", UBM: "ubm", DBN: "dbn", CCM: "ccm"}
SIZES = [1, 2, 63, 64, 65, 255, 256, 257, 1000, 16_384, 16_385, 32_769, 49_152, 262_145]
_models = {}


def trained(model, uneven):
    key = (model, uneven)
    if key not in _models:
        s = synth.generate(synth.SynthConfig(n_sessions=6000, n_queries=500, vocab=20000, model=NAMES[model],
                                             variable_length=uneven, seed=900 + model))
        ds = Dataset.from_sessions(s.query, s.docs, s.clicks, 0.2, length=s.length if uneven else None)
        cm = ClickModel(model)
        cm.init_from_dataset(ds)
        cm.em(5)
        _models[key] = (cm, ds)
    return _models[key]


def held_out(ds, n):
    rng = np.random.default_rng(n)
    i = rng.integers(0, len(ds.train), n)
    p = ds.train.pidx[i].copy()
    p[rng.random((n, 10)) < 0.1] = -1
    ln = None if ds.train.length is None else ds.train.length[i]
    return SessionSet(ds.train.query[i], ds.train.docs[i], ds.train.clicks[i], p, ln)


@pytest.mark.parametrize("uneven", [False, True], ids=["ten", "uneven"])
@pytest.mark.parametrize("model", list(NAMES), ids=NAMES.get)
def test_host_arrays_match_the_resident_set(model, uneven):
    cm, ds = trained(model, uneven)
    for n in SIZES:
        print(f"case rows model={model} uneven={uneven} n={n}", flush=True)
        te = held_out(ds, n)
        cm.set_test_set(te)
        want = cm.evaluate_test_set(per_session=True)
        got = cm.evaluate(te, per_session=True)
        for k in ("logp", "full", "llh"):
            np.testing.assert_array_equal(got[k], want[k])
        np.testing.assert_array_equal(got["rank_count"], want["rank_count"])
        totals = cm.evaluate(te)
        for ev in (got, totals):
            assert ev["llh_sum"] == pytest.approx(want["llh_sum"], rel=1e-6)
            np.testing.assert_allclose(ev["ppl_log2_sum"], want["ppl_log2_sum"], rtol=1e-6, atol=1e-9)
        if model in (DBN, CCM):   # the probability whose log is logp
            shown = np.arange(10)[None, :] < (te.length[:, None] if uneven else np.full((n, 1), 10))
            prob = cm.get_serp_probability(te)
            np.testing.assert_allclose(np.log(prob[shown]), want["logp"][shown], rtol=1e-5, atol=1e-6)
            assert not prob[~shown].any()


@pytest.mark.parametrize("shift", [0, 1, 3])
def test_device_arrays_at_any_element_address(shift):
    """mc_evaluate_device on arrays that start `shift` elements into their
    allocations (4-byte words and single bytes)."""
    hip = Hip()
    cm, ds = trained(UBM, True)
    n = 193
    te = held_out(ds, n)
    want = cm.evaluate(te, per_session=True)

    def at(a):
        return C.c_void_p(hip.upload(np.concatenate([np.zeros(shift, a.dtype), a.reshape(-1)])).value
                          + shift * a.itemsize)

    args = [at(te.pidx.astype(np.int32)), at(te.clicks.astype(np.uint8)), at(te.length.astype(np.uint8))]
    out = [at(np.full(n * k, 7.0, np.float32)) for k in (10, 10, 1)]
    totals = hip.empty(21 * 8)
    print(f"case device-rows shift={shift}", flush=True)
    _lib.check(_lib.lib().mc_evaluate_device(cm._h, n, *args, *out, totals))
    _lib.check(_lib.lib().mc_synchronize(cm._h))
    for p, k in zip(out, ("logp", "full", "llh")):
        np.testing.assert_array_equal(hip.download(p, want[k].shape, np.float32), want[k])
    assert hip.download(totals, 21, np.float64)[0] == want["llh_sum"]
    hip.close()
