"""Numerators and denominators of a table in one pass: the host fills in the
denominators that it knows while the numerators are on their way, so the two
take hardly longer than one."""
import time

import numpy as np
import pytest

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel, _lib
from test_gpu_shapes import sessions

pytestmark = pytest.mark.gpu

IDS = {PBM: "PBM", UBM: "UBM", DBN: "DBN", CCM: "CCM"}


def f32(a):
    return _lib.ptr(a, _lib.f32p)


@pytest.mark.parametrize("model", list(IDS), ids=IDS.get)
@pytest.mark.parametrize("n_qd", [1_000, 262_144, 262_145, 2_100_000])
def test_either_array_alone(model, n_qd):
    """Numerators alone and denominators alone, from the start, after an
    M-step and as the caller set them; a null pointer for the other is taken."""
    train, used = sessions([9] * 20, 14, 3)
    lib = _lib.lib()
    print(f"case either array model={IDS[model]} entries={n_qd}", flush=True)
    with ClickModel(model) as cm:
        cm.init_parameters(train, n_qd)
        for stage in ("start", "trained", "set"):
            if stage == "trained":
                cm.em(2)
            for t, (_, _, size) in enumerate(cm.get_parameter_information()):
                if stage == "set":
                    cm.set_parameters(t, np.arange(size, dtype=np.float32) + 1, np.arange(size, dtype=np.float32) + 3)
                num, den = cm.get_parameters(t)
                a, b = np.full(size, -1, np.float32), np.full(size, -1, np.float32)
                _lib.check(lib.mc_get_parameters(cm._h, t, f32(a), None))
                _lib.check(lib.mc_get_parameters(cm._h, t, None, f32(b)))
                np.testing.assert_array_equal(a, num)
                np.testing.assert_array_equal(b, den)
                _lib.check(lib.mc_get_parameters(cm._h, t, None, None))
        occ = np.bincount(train.pidx.reshape(-1), minlength=n_qd)
        assert occ[:used].min() > 0 and occ.sum() == train.pidx.size


@pytest.mark.parametrize("entries", [2_000, 90_000, 250_000])
def test_both_arrays_take_hardly_longer_than_one(entries):
    """At most 1.5 times the copy of as many logits: two passes take 1.8 to 2
    times, and the denominators alone add less than a tenth."""
    train, _ = sessions([9] * 20, 14, 3)
    lib = _lib.lib()
    with ClickModel(PBM) as cm:
        cm.init_parameters(train, entries)
        cm.em(2)
        num, den, x = (np.ones(entries, np.float32) for _ in range(3))

        def fastest(f):
            best = 1e9
            for _ in range(60):
                t = time.perf_counter()
                _lib.check(f())
                best = min(best, time.perf_counter() - t)
            return best * 1e6

        both = fastest(lambda: lib.mc_get_parameters(cm._h, 0, f32(num), f32(den)))
        cm.grad_init()
        one = fastest(lambda: lib.mc_get_logits(cm._h, 0, f32(x)))
    print(f"case both arrays entries={entries}: {both:.1f} us, one array {one:.1f} us", flush=True)
    assert both <= 1.5 * one, (both, one)
