"""The log-likelihood sum of mc_evaluate_device, whose lanes take several
sessions each from 262,144 on: FP64 from the sessions' terms on.

Bar: 1e-13 relative of the FP64 sum of the call's own per-session values.  A
lane adds up to four terms, then come at most 30 more levels of FP64 sums: 34
roundings of 1.1e-16 are 4e-15, as the terms have one sign.  FP32 lane sums
miss it by 5e-13 and more."""

import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel, Dataset, _lib, synth
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

NAMES = {PBM: "pbm", UBM: "ubm", DBN: "dbn", CCM: "ccm"}


@pytest.mark.parametrize("model", list(NAMES), ids=NAMES.get)
def test_sums_of_many_sessions_are_fp64(model):
    s = synth.generate(synth.SynthConfig(n_sessions=6000, n_queries=500, vocab=20000, model=NAMES[model], seed=70 + model))
    ds = Dataset.from_sessions(s.query, s.docs, s.clicks, 0.2)
    hip = Hip()
    with ClickModel(model) as cm:
        cm.init_from_dataset(ds)
        cm.em(5)
        for n in (262_144, 262_145, 700_001, 1_000_000):
            print(f"case evaluation sums model={NAMES[model]} n={n}", flush=True)
            i = np.random.default_rng(n).integers(0, len(ds.train), n)
            args = [hip.upload(ds.train.pidx[i]), hip.upload(ds.train.clicks[i]), None]
            llh, totals = hip.empty(4 * n), hip.empty(21 * 8)
            full = hip.empty(40 * n)
            _lib.check(_lib.lib().mc_evaluate_device(cm._h, n, *args, None, full, llh, totals))
            _lib.check(_lib.lib().mc_synchronize(cm._h))
            got = hip.download(totals, 21, np.float64)
            want = hip.download(llh, n, np.float32).astype(np.float64).sum()
            assert abs(got[0] / want - 1) < 1e-13, (got[0], want)
            # Each term a log2 in FP32.
            log2 = np.log2(hip.download(full, (n, 10), np.float32).astype(np.float64)).sum(0)
            np.testing.assert_allclose(got[1:11], log2, rtol=1e-7)
            assert (got[11:] == n).all()
            hip.close()
