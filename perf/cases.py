"""Timed workloads of the EM engine, through its public entry points.

Each case is one thing a program does with a click model: a training run of
EM iterations on a resident training set, a run that follows the held-out
likelihood, a fit by Adam, the likelihood gradient, and the evaluation of
sessions that lie on the host or on the device.  Click logs are synthetic:
Zipf queries, a pool of documents per query, clicks of the fitted model.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs and model, as a program has them before the call
  run(state)           one pass, returning everything it computes
  work(case)           bytes and operations that a pass cannot do without
  exact(case, seed)    what run returns, in 64-bit torch arithmetic
"""
import ctypes
import math

import numpy as np
import torch

from massiveclicks_amd import CCM, DBN, PBM, UBM, ClickModel, SessionSet, _lib

RANKS = 10
MODELS = {"pbm": PBM, "ubm": UBM, "ccm": CCM, "dbn": DBN}
TOP = float(np.float32(1.0) - np.float32(1e-6))   # Param::value's upper bound


def listed():
    return [
        # A small site's log (the 40,000-session set of the tests): every
        # iteration is a launch of a few workgroups.
        _em("em_pbm_small", "pbm", 32_000, 2_000),
        # A medium log, fitted with the largest shared table.
        _em("em_ubm_medium", "ubm", 312_457, 40_000),
        # A large log of the cascade model with three continuation parameters.
        _em("em_ccm_large", "ccm", 2_000_003, 200_000),
        # The benchmark's training set: 8M of 10M sessions, 1M queries.
        _em("em_dbn_headline", "dbn", 8_000_000, 1_000_000),
        # Result lists of 1 to 10 ranks.
        _em("em_dbn_uneven", "dbn", 3_000_000, 300_000, zipf=1.3, uneven=True),
        # Few queries with many documents each (personalised results, long
        # logs): the entries of one query exceed a work item's window.
        _em("em_ubm_wide", "ubm", 1_000_000, 1_500, pool=1_500),
        # Training that looks at the held-out likelihood after every iteration.
        _case("curve_dbn", "curve", "dbn", 500_000, 60_000, iterations=20, tests=120_000),
        # Some epochs of Adam on the likelihood gradient, minibatches of
        # query groups, from the logits of an earlier fit.
        _case("adam_dbn", "adam", "dbn", 2_000_000, 200_000, batches=4, epochs=3, item_sessions=4096),
        # One full gradient of a medium log, for an optimiser of the caller's.
        _case("gradient_ubm", "gradient", "ubm", 700_001, 80_000),
        # Scoring sessions that already lie on the device (serving loops).
        _case("score_ccm_device", "score", "ccm", 200_000, 20_000, tests=1_000_000),
        # Evaluating a held-out set given as host arrays, with its
        # per-session probabilities.
        _case("evaluate_dbn_host", "evaluate", "dbn", 400_000, 40_000, tests=100_000),
        # Click probabilities of one small batch of result pages.
        _case("serp_ubm_batch", "serp", "ubm", 50_000, 5_000, tests=256),
    ]


def _case(name, op, model, sessions, queries, pool=20, zipf=1.1, uneven=False, **more):
    case = {"op": op, "model": model, "sessions": sessions, "queries": queries, "pool": pool, "zipf": zipf,
            "uneven": uneven, **more}
    return {"name": name, **case} if name else case


def _em(name, model, sessions, queries, iterations=50, **more):
    return _case(name, "em", model, sessions, queries, iterations=iterations, **more)


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["em", "em", "em", "curve", "adam", "gradient", "score", "evaluate", "serp"])
    model = rng.choice(sorted(MODELS))
    uneven = rng.random() < 0.3
    zipf = round(rng.uniform(1.0, 1.4), 2)
    if op == "em" and rng.random() < 0.25:   # many documents per query
        pool = _spread(rng, 100, 2_000)
        sessions = _spread(rng, 50_000, 1_000_000)
        return _em(None, model, sessions, max(20, _spread(rng, 2e6, 6e6) // pool // 2), pool=pool, zipf=zipf,
                   uneven=uneven)
    sessions = _spread(rng, 5_000, 4_000_000 if op == "em" else 1_500_000)
    queries = max(50, int(sessions / rng.uniform(6, 30)))
    pool = rng.randint(12, 60)
    if op == "em":
        return _em(None, model, sessions, queries, pool=pool, zipf=zipf, uneven=uneven,
                   iterations=rng.choice([20, 50, 50, 100]))
    if op == "curve":
        return _case(None, op, model, sessions, queries, pool, zipf, uneven, iterations=rng.randint(5, 30),
                     tests=max(100, sessions // 4))
    if op == "adam":
        return _case(None, op, model, sessions, queries, pool, zipf, uneven, batches=rng.randint(1, 4),
                     epochs=rng.randint(1, 5), item_sessions=rng.choice([4096, 8192]))
    if op == "gradient":
        return _case(None, op, model, sessions, queries, pool, zipf, uneven)
    tests = {"score": (1_000, 2_000_000), "evaluate": (500, 300_000), "serp": (16, 20_000)}[op]
    return _case(None, op, model, min(sessions, 200_000), min(queries, 20_000), pool, zipf, uneven,
                 tests=_spread(rng, *tests))


# ---------------------------------------------------------------------------
# Synthetic sessions, made on the GPU
# ---------------------------------------------------------------------------

def _beta(gen, n, a, b):
    """Beta(a, b) for whole a, b as a ratio of Gamma draws."""
    x = [torch.zeros(n, device="cuda") for _ in range(2)]
    for g, k in zip(x, (a, b)):
        for _ in range(k):
            g -= torch.log(1 - torch.rand(n, generator=gen, device="cuda"))
    return x[0] / (x[0] + x[1])


def _queries(case, gen, n):
    w = torch.arange(1, case["queries"] + 1, device="cuda", dtype=torch.float64) ** -case["zipf"]
    cdf = torch.cumsum(w, 0)
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) * cdf[-1]
    return torch.clamp(torch.searchsorted(cdf, u, right=True), max=case["queries"] - 1)


def _shown(case, gen, n):
    """Ten distinct slots of the query's pool in random order, per session."""
    pool, picks, slots = case["pool"], [], []
    for r in range(RANKS):
        x = (torch.rand(n, generator=gen, device="cuda") * (pool - r)).int().clamp(max=pool - r - 1)
        for s in picks:   # ascending: step over the slots already taken
            x = x + (x >= s).int()
        slots.append(x)
        for j, s in enumerate(picks):
            picks[j], x = torch.minimum(s, x), torch.maximum(s, x)
        picks.append(x)
    return torch.stack(slots, 1).long()


def _clicks(case, gen, alpha, sigma, length):
    n, model = len(alpha), case["model"]
    u, u2, u3 = (torch.rand(n, RANKS, generator=gen, device="cuda") for _ in range(3))
    out = torch.zeros(n, RANKS, dtype=torch.bool, device="cuda")
    live = torch.ones(n, dtype=torch.bool, device="cuda")
    last = torch.full((n,), -1, device="cuda")
    for r in range(RANKS):
        a = alpha[:, r]
        if model == "pbm":
            c = u[:, r] < a / (r + 1.0) ** 0.8
        elif model == "ubm":
            c = u[:, r] < a * 0.9 * torch.exp(-0.15 * r - 0.1 * (r - last))
            last = torch.where(c, r, last)
        else:
            c = live & (u[:, r] < a)
            if model == "dbn":
                live = live & ~(c & (u2[:, r] < sigma[:, r])) & (u3[:, r] < 0.9)
            else:
                live = live & (u3[:, r] < torch.where(c, 0.6 * (1 - a) + 0.4 * a, 0.95))
        out[:, r] = c & (r < length)
    return out


def _sessions(case, gen, n, alpha, sigma, by_query):
    q = _queries(case, gen, n)
    if by_query:
        q = torch.sort(q)[0]
    pair = q[:, None] * case["pool"] + _shown(case, gen, n)
    length = (torch.randint(1, RANKS + 1, (n,), generator=gen, device="cuda") if case["uneven"]
              else torch.full((n,), RANKS, device="cuda"))
    return q, pair, _clicks(case, gen, alpha[pair], sigma[pair], length), length


def _data(case, seed):
    """Training and held-out sessions as device tensors: query, pair index
    (-1: past the list, or not seen in training), clicks, length."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 17)
    slots = case["queries"] * case["pool"]
    alpha = _beta(gen, slots, 2, 5)
    sigma = _beta(gen, slots, 2, 8)
    rank = torch.arange(RANKS, device="cuda")
    q, pair, c, length = _sessions(case, gen, case["sessions"], alpha, sigma, True)
    shown = rank < length[:, None]
    seen = torch.zeros(slots, dtype=torch.bool, device="cuda")
    seen[pair[shown]] = True
    index = torch.where(seen, torch.cumsum(seen, 0) - 1, -1)
    train = {"query": q, "pidx": torch.where(shown, index[pair], -1), "clicks": c, "length": length}
    test = None
    if case.get("tests"):
        q, pair, c, length = _sessions(case, gen, case["tests"], alpha, sigma, False)
        test = {"query": q, "pidx": torch.where(rank < length[:, None], index[pair], -1), "clicks": c,
                "length": length}
    # Tables with room for a few pairs that no training session shows, the
    # same for every seed.
    return train, test, max(int(seen.sum()), int(1.02 * _entries(case)) + 500)


def _host(case, d):
    n = len(d["query"])
    return SessionSet(query=d["query"].int().cpu().numpy(), docs=np.empty((n, 0), np.int32),
                      clicks=d["clicks"].to(torch.uint8).cpu().numpy(), pidx=d["pidx"].int().cpu().numpy(),
                      length=d["length"].to(torch.uint8).cpu().numpy() if case["uneven"] else None)


def _first_logits(case, seed, n_qd):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 18)
    return [torch.randn(len(t[0]), generator=gen, device="cuda") * 0.5 for t in _start(case["model"], n_qd)]


# Adam's eps: pairs whose gradient is down to rounding stay where they are.
EPS = 1e-4

# Iterations that a model used for scoring has been trained for.
SCORED_AFTER = 5


def prepare(case, seed):
    train, test, n_qd = _data(case, seed)
    op = case["op"]
    options = {k: case[k] for k in ("batches", "item_sessions") if k in case}
    cm = ClickModel(MODELS[case["model"]], **options)
    cm.init_parameters(_host(case, train), n_qd)
    state = {"case": case, "cm": cm}
    if op == "curve":
        cm.set_test_set(_host(case, test))
    if op in ("score", "evaluate", "serp"):
        cm.em(SCORED_AFTER)
    if op in ("evaluate", "serp"):
        state["test"] = _host(case, test)
    if op == "score":
        n = case["tests"]
        state["in"] = [test["pidx"].int().contiguous(), test["clicks"].to(torch.uint8).contiguous(),
                       test["length"].to(torch.uint8).contiguous() if case["uneven"] else None]
        state["out"] = [torch.empty(n, RANKS, device="cuda"), torch.empty(n, RANKS, device="cuda"),
                        torch.empty(n, device="cuda"), torch.empty(21, device="cuda", dtype=torch.float64)]
    if op == "gradient":
        cm.em(2)
    if op == "adam":
        cm.grad_init()
        cm.adam_configure(eps=EPS)
        for t, x in enumerate(_first_logits(case, seed, n_qd)):
            cm.set_logits(t, x.cpu().numpy())
    return state


# Sums of 32-bit log-probabilities go out in 32 bits.
def _single(x):
    return np.asarray(x, np.float32)


def _tables(cm):
    return [list(cm.get_parameters(t)) for t in range(cm.n_tables())]


def run(state):
    case, cm = state["case"], state["cm"]
    op = case["op"]
    if op == "em":
        cm.reset_parameters()
        cm.em(case["iterations"])
        return _tables(cm)
    if op == "curve":
        cm.reset_parameters()
        curve = []
        for _ in range(case["iterations"]):
            cm.em(1)
            ev = cm.evaluate_test_set()
            curve.append([ev["log_likelihood"], ev["perplexity"]])
        return {"curve": _single(curve), "tables": _tables(cm)}
    if op == "adam":
        cm.adam_steps(case["epochs"] * case["batches"])
        return [cm.get_logits(t) for t in range(cm.n_tables())]
    if op == "gradient":
        ll, grads = cm.loglik_gradient()
        return {"ll": _single(ll), "grads": grads}
    if op == "score":
        ptrs = [None if x is None else ctypes.c_void_p(x.data_ptr()) for x in state["in"] + state["out"]]
        _lib.check(_lib.lib().mc_evaluate_device(cm._h, case["tests"], *ptrs))
        _lib.check(_lib.lib().mc_synchronize(cm._h))
        logp, full, llh, totals = state["out"]
        return {"logp": logp, "full": full, "llh": llh, "totals": _single(totals.cpu().numpy())}
    if op == "evaluate":
        ev = cm.evaluate(state["test"], per_session=True)
        return {"logp": ev["logp"], "full": ev["full"], "llh": ev["llh"], "rank_count": ev["rank_count"],
                "sums": _single([ev["llh_sum"], *ev["ppl_log2_sum"]])}
    return {"prob": cm.get_serp_probability(state["test"])}


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------

def _entries(case):
    """Expected number of query-document pairs of the training set."""
    p = np.arange(1, case["queries"] + 1, dtype=np.float64) ** -case["zipf"]
    per = case["sessions"] * p / p.sum()
    miss = 1.0 - (5.5 if case["uneven"] else 10.0) / case["pool"]
    return float(np.sum(case["pool"] * (1.0 - np.power(miss, per))))


def work(case):
    """Per session 4 bytes an index and 2 bytes of clicks (a byte of length);
    per entry and per-query table of an EM iteration 16 bytes (a pair read,
    a pair written), of an Adam step 28 (logit and moments read and written,
    a value written).  Operations: about 30 a rank and pass."""
    op, T = case["op"], 2 if case["model"] == "dbn" else 1
    ranks = 5.5 if case["uneven"] else 10.0
    row = 4 * ranks + 2 + (1 if case["uneven"] else 0)
    tests = case.get("tests", 0)
    per_pass = case["sessions"] * row + 16 * T * _entries(case)
    flops = 30 * ranks * case["sessions"]
    if op == "em":
        return {"bytes": case["iterations"] * per_pass, "flops": case["iterations"] * flops}
    if op == "curve":
        held = tests * (row + 4 * T * ranks)
        return {"bytes": case["iterations"] * (per_pass + held), "flops": case["iterations"] * (flops + 30 * ranks * tests)}
    if op == "adam":
        return {"bytes": case["epochs"] * (case["sessions"] * row + 28 * T * _entries(case)), "flops": 2 * case["epochs"] * flops}
    if op == "gradient":
        return {"bytes": case["sessions"] * row + 8 * T * _entries(case), "flops": 2 * flops}
    out = {"score": 84, "evaluate": 84, "serp": 40}[op]
    return {"bytes": tests * (4 * ranks + ranks + 4 * T * ranks + out), "flops": 30 * ranks * tests}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

class _Index:
    """Reads a table at a session's ranks and sums back into it; `on` marks
    the ranks that have an index, the others read 1/2."""

    def __init__(self, index, on, size):
        self.index, self.on, self.size = torch.where(on, index, 0), on, size
        flat = torch.nonzero(on.reshape(-1))[:, 0]
        key, order = torch.sort(index.reshape(-1)[flat], stable=True)
        self.order = flat[order]
        self.ends = torch.searchsorted(key, torch.arange(size + 1, device="cuda"))

    def total(self, w):
        """Sum of w over the ranks of each index."""
        c = torch.zeros(len(self.order) + 1, dtype=torch.float64, device="cuda")
        torch.cumsum(w.reshape(-1)[self.order].double(), 0, out=c[1:])
        return c[self.ends[1:]] - c[self.ends[:-1]]

    def read(self, v):
        return _Read.apply(v, self)


class _Read(torch.autograd.Function):
    @staticmethod
    def forward(ctx, v, index):
        ctx.index = index
        return torch.where(index.on, v[index.index], 0.5)

    @staticmethod
    def backward(ctx, grad):
        return ctx.index.total(grad), None


class _Sessions64:
    """Rank-by-rank columns of a session set, as the models need them."""

    def __init__(self, case, d, n_qd):
        n = len(d["query"])
        self.n, self.n_qd, self.model = n, n_qd, case["model"]
        self.length = d["length"]
        ranks = torch.arange(RANKS, device="cuda")
        self.all_shown = ranks < d["length"][:, None]
        self.all_click = d["clicks"] & self.all_shown
        self.shown = [self.all_shown[:, r] for r in range(RANKS)]
        self.click = [self.all_click[:, r] for r in range(RANKS)]
        self.pair = _Index(d["pidx"], d["pidx"] >= 0, n_qd)
        last = torch.where(d["clicks"], ranks, -1).max(1)[0]
        self.last = torch.where(last < 0, RANKS, last)
        prev = torch.full((n,), RANKS - 1, device="cuda")
        self.slot = []
        for r in range(RANKS):
            self.slot.append(torch.full_like(prev, r) if case["model"] == "pbm" else r * (r + 1) // 2 + prev)
            prev = torch.where(self.click[r], r, prev)
        if case["model"] in ("pbm", "ubm"):
            self.exam = _Index(torch.stack(self.slot, 1), self.all_shown, _slots(case["model"]))

    def counts(self):
        return self.pair.total(self.all_shown), self.pair.total(self.all_click)

    def written(self, slots):
        """Sessions that write each examination slot (its last writer counts),
        and those that write it from a clicked rank."""
        w, wc = (torch.zeros(slots, dtype=torch.float64, device="cuda") for _ in range(2))
        for r in range(RANKS):
            lw = self.shown[r].clone()
            for q in range(r + 1, RANKS):
                lw &= ~(self.shown[q] & (self.slot[q] == self.slot[r]))
            w += torch.bincount(self.slot[r][lw], minlength=slots)
            wc += torch.bincount(self.slot[r][lw & self.click[r]], minlength=slots)
        return w, wc


def _slots(model):
    return {"pbm": 10, "ubm": 55, "ccm": 3, "dbn": 1}[model]


def _value(t):
    return torch.clamp(t[0] / t[1], max=TOP)


def _start(model, n_qd):
    sizes = [n_qd] * (2 if model == "dbn" else 1) + [_slots(model)]
    return [[torch.full((k,), v, dtype=torch.float64, device="cuda") for v in (1.0, 2.0)] for k in sizes]


def _em_step(S, tables, const):
    """One EM iteration; const: what does not change between iterations."""
    occ, clk, shared = const
    vals = [_value(t) for t in tables]
    zero = torch.zeros((), dtype=torch.float64, device="cuda")
    a = S.pair.read(vals[0])
    if S.model in ("pbm", "ubm"):
        e = S.exam.read(vals[1])
        on = S.all_shown & ~S.all_click
        attr = 1 + clk + S.pair.total(torch.where(on, a * (1 - e) / (1 - a * e), zero))
        num = shared[0] + S.exam.total(torch.where(on, e * (1 - a) / (1 - a * e), zero))
        return [[attr, 2 + occ], [num, shared[1]]]
    a = list(a.unbind(1))
    extra = [None] * RANKS   # attractiveness terms of each rank
    has = S.last < RANKS
    if S.model == "dbn":
        s = S.pair.read(vals[1]).unbind(1)
        sat = [None] * RANKS
        g = vals[2][0]
        stay = [g * (1 - a[r]) for r in range(RANKS)]
        move = [g * a[r] * (1 - s[r]) for r in range(RANKS)]
    else:
        t1, t2, t3 = vals[1]
        stay = [t1 * (1 - a[r]) for r in range(RANKS)]
        move = [a[r] * (t2 * (1 - a[r]) + t3 * a[r]) for r in range(RANKS)]
    exam, e = [], torch.ones(S.n, dtype=torch.float64, device="cuda")
    tail, G = [e], e
    for r in range(RANKS):
        exam.append(e)
        e = torch.where(S.shown[r], e * (stay[r] + move[r]), e)
        tail.append(tail[-1] - a[r] * G)
        G = G * stay[r]
    tail = torch.stack(tail, 1)
    car = torch.zeros_like(e)
    after_last = torch.zeros_like(e)   # car of the rank behind the last click
    for r in reversed(range(RANKS)):
        after_last = torch.where(S.last == r, car, after_last)
        car = torch.where(S.shown[r], a[r] + stay[r] * car, car)
        on = S.shown[r] & has & (r > S.last)
        extra[r] = torch.where(on, a[r] * (1 - exam[r]) / (1 - exam[r] * car), zero)
    E = torch.zeros_like(e)
    if S.model == "dbn":
        num, den = shared[0].clone(), shared[1].clone()
    else:
        sums = [[shared[0][k].clone(), shared[1][k].clone()] for k in range(3)]
    for r in range(RANKS):
        T = torch.gather(tail, 1, torch.clamp(S.length - 1 - r, min=0)[:, None])[:, 0]
        at = S.last == r
        on = S.shown[r] & has & (r > S.last)
        if S.model == "dbn":
            sat[r] = torch.where(at, s[r] / (1 - (1 - s[r]) * g * after_last), zero)
            f4, f5 = (1 - s[r]) * (1 - g), (1 - s[r]) * g * T
            d = f4 + f5 + s[r]
            h4, h5 = E * (1 - g), E * g * T
            dh = 1 - E + h4 + h5
            num += torch.where(at, f5 / d, zero).sum() + torch.where(on, h5 / dh, zero).sum()
            den += torch.where(at, (f4 + f5) / d, zero).sum() + torch.where(on, (h4 + h5) / dh, zero).sum()
            E = torch.where(at, g * (1 - s[r]), torch.where(on, E * stay[r] / (1 - a[r] * E), E))
        else:
            w2, w3 = (1 - a[r]) * t2, a[r] * t3
            extra[r] = torch.where(at, a[r] / (1 - (w2 + w3) * after_last), extra[r])
            early = S.shown[r] & has & S.click[r] & (r < S.last)
            x2, x3 = torch.where(early, w2 / (w2 + w3), zero).sum(), torch.where(early, w3 / (w2 + w3), zero).sum()
            f4, f6 = (1 - a[r]) * (1 - t2), a[r] * (1 - t3)
            d = f4 + w2 * T + f6 + w3 * T
            n2, n3 = torch.where(at, w2 * T / d, zero).sum(), torch.where(at, w3 * T / d, zero).sum()
            h4, h5 = E * (1 - t1), E * t1 * T
            dh = 1 - E + h4 + h5
            n1 = torch.where(on, h5 / dh, zero).sum()
            for k, (x, y) in enumerate(((n1, n1 + torch.where(on, h4 / dh, zero).sum()),
                                        (x2 + n2, x2 + n2 + torch.where(at, f4 / d, zero).sum()),
                                        (x3 + n3, x3 + n3 + torch.where(at, f6 / d, zero).sum()))):
                sums[k][0] += x
                sums[k][1] += y
            E = torch.where(at, w2 + w3, torch.where(on, E * stay[r] / (1 - a[r] * E), E))
    attr = 1 + clk + S.pair.total(torch.stack(extra, 1))
    if S.model == "dbn":
        sat = 1 + occ - clk + S.pair.total(torch.stack(sat, 1))
        return [[attr, 2 + occ], [sat, 2 + 2 * occ - clk], [num, den]]
    return [[attr, 2 + occ + clk], [torch.stack([x[i] for x in sums]) for i in (0, 1)]]


def _em_constants(S):
    occ, clk = S.counts()
    K = _slots(S.model)
    if S.model in ("pbm", "ubm"):
        w, wc = S.written(K)
        return occ, clk, [1 + wc + (S.n - w), 2 + w + 2 * (S.n - w)]
    before = torch.minimum(S.last, S.length)
    if S.model == "ccm":   # unclicked ranks before the last click
        before = sum((S.shown[r] & ~S.click[r] & (r < S.last)).long() for r in range(RANKS))
    k = torch.zeros(K, dtype=torch.float64, device="cuda")
    k[0] = before.sum().double()
    return occ, clk, [1 + k, 2 + k]


def _chain(S, vals, full):
    """Per rank the conditional probability of the observed click or skip, or
    (full) of the click bit without the session's other clicks."""
    model = S.model
    a = S.pair.read(vals[0]).unbind(1)
    sat = S.pair.read(vals[1]).unbind(1) if model == "dbn" else None
    e = S.exam.read(vals[1]).unbind(1) if model in ("pbm", "ubm") else None
    ex = torch.ones(S.n, dtype=torch.float64, device="cuda")
    out, marginal = [], []
    for r in range(RANKS):
        c = S.click[r]
        if model in ("pbm", "ubm"):
            if full and model == "ubm":
                pc = torch.zeros_like(ex)
                for j in range(-1, r):
                    skip = torch.ones_like(ex)
                    for i in range(j + 1, r):
                        skip = skip * (1 - a[i] * vals[1][i * (i + 1) // 2 + (j if j >= 0 else RANKS - 1)])
                    k = r * (r + 1) // 2 + (j if j >= 0 else RANKS - 1)
                    pc = pc + (marginal[j] if j >= 0 else 1.0) * skip * a[r] * vals[1][k]
                marginal.append(pc)
            else:
                pc = a[r] * e[r]
            out.append(torch.where(c, pc, 1 - pc))
            continue
        pc = a[r] * ex
        pr = torch.where(c, pc, 1 - pc)
        out.append(pr)
        if model == "dbn":
            g = vals[2][0]
            on, off = g * (1 - sat[r]), g * (1 - a[r])
        else:
            t1, t2, t3 = vals[1]
            on, off = t2 * (1 - a[r]) + t3 * a[r], t1 * (1 - a[r])
        ex = ex * (off + a[r] * on) if full else torch.where(c, on, ex * off / pr)
    return out


def _evaluation(S, vals):
    """logp, full, llh and the sums of a session set."""
    zero = torch.zeros((), dtype=torch.float64, device="cuda")
    cond, full = _chain(S, vals, False), _chain(S, vals, True)
    logp = torch.stack([torch.where(S.shown[r], torch.log(cond[r]), zero) for r in range(RANKS)], 1)
    fp = torch.stack([torch.where(S.shown[r], full[r], zero) for r in range(RANKS)], 1)
    llh = logp.sum(1) / S.length
    log2 = torch.stack([torch.where(S.shown[r], torch.log2(full[r]), zero).sum() for r in range(RANKS)])
    count = torch.stack([S.shown[r].sum() for r in range(RANKS)])
    return logp, fp, llh, torch.cat([llh.sum()[None], log2]), count


def _loglik_gradient(S, vals):
    """Log-likelihood and its gradient with respect to the logits."""
    leaves = [v.detach().requires_grad_() for v in vals]
    zero = torch.zeros((), dtype=torch.float64, device="cuda")
    cond = _chain(S, leaves, False)
    ll = sum(torch.where(S.shown[r], torch.log(cond[r]), zero).sum() for r in range(RANKS))
    grads = torch.autograd.grad(ll, leaves, allow_unused=True)
    return float(ll), [torch.zeros_like(v) if g is None else g * v * (1 - v) for g, v in zip(grads, vals)]


def _adam(case, seed, train, n_qd):
    """Adam over minibatches of whole query groups: the group that starts at
    session s is in batch s * batches // sessions."""
    n, B, model = case["sessions"], case["batches"], case["model"]
    _, group, size = torch.unique_consecutive(train["query"], return_inverse=True, return_counts=True)
    batch = torch.clamp((torch.cumsum(size, 0) - size)[group] * B // n, max=B - 1)
    whole = _Sessions64(case, train, n_qd)
    occ, clk = whole.counts()
    logits = [x.double() for x in _first_logits(case, seed, n_qd)]
    prior = [torch.ones_like(x) for x in logits]
    if model == "dbn":
        prior[1] += occ - clk
    if model in ("pbm", "ubm"):
        prior[-1] += n - whole.written(_slots(model))[0]
    m, v = ([torch.zeros_like(x) for x in logits] for _ in range(2))
    parts = []
    for b in range(B):
        on = batch == b
        sub = {k: x[on] for k, x in train.items()}
        used = sub["pidx"][sub["pidx"] >= 0]
        mine = torch.zeros(n_qd, dtype=torch.bool, device="cuda")
        mine[used] = True
        parts.append((_Sessions64(case, sub, n_qd), mine))
    for e in range(case["epochs"]):
        for b, (S, mine) in enumerate(parts):
            if not S.n:
                continue
            vals = [torch.sigmoid(x) for x in logits]
            _, grads = _loglik_gradient(S, vals)
            for t, g in enumerate(grads):
                last = t == len(grads) - 1
                step = e * B + b + 1 if last else e + 1
                on = torch.ones_like(g, dtype=torch.bool) if last else mine
                g = (g * (n / S.n) if last else g) + prior[t] * (1 - 2 * vals[t])
                m[t] = torch.where(on, 0.9 * m[t] + 0.1 * g, m[t])
                v[t] = torch.where(on, 0.999 * v[t] + 0.001 * g * g, v[t])
                d = torch.sqrt(v[t]) / math.sqrt(1 - 0.999 ** step) + EPS
                new = torch.clamp(logits[t] + 0.05 / (1 - 0.9 ** step) * m[t] / d, -13.8, 13.8)
                logits[t] = torch.where(on, new, logits[t])
    return logits


def exact(case, seed):
    train, test, n_qd = _data(case, seed)
    op, model = case["op"], case["model"]
    if op == "adam":
        return _adam(case, seed, train, n_qd)
    S = _Sessions64(case, train, n_qd)
    held = _Sessions64(case, test, n_qd) if test else None
    const = _em_constants(S)
    tables = _start(model, n_qd)
    curve = []
    for _ in range({"em": case.get("iterations"), "curve": case.get("iterations"), "gradient": 2}.get(op, SCORED_AFTER)):
        tables = _em_step(S, tables, const)
        if op == "curve":
            _, _, _, sums, count = _evaluation(held, [_value(t) for t in tables])
            ppl = torch.where(count > 0, 2.0 ** (-sums[1:] / count), torch.nan).mean()
            curve.append([float(sums[0]) / held.n, float(ppl)])
    if op == "em":
        return tables
    if op == "curve":
        return {"curve": np.asarray(curve), "tables": tables}
    vals = [_value(t) for t in tables]
    if op == "gradient":
        ll, grads = _loglik_gradient(S, vals)
        return {"ll": np.asarray(ll), "grads": grads}
    if op == "serp":
        zero = torch.zeros((), dtype=torch.float64, device="cuda")
        prob = _chain(held, vals, False)
        if model in ("pbm", "ubm"):   # the click probability, whatever the click
            prob = [torch.where(held.click[r], prob[r], 1 - prob[r]) for r in range(RANKS)]
        return {"prob": torch.stack([torch.where(held.shown[r], prob[r], zero) for r in range(RANKS)], 1)}
    logp, full, llh, sums, count = _evaluation(held, vals)
    out = {"logp": logp, "full": full, "llh": llh}
    if op == "score":
        return {**out, "totals": torch.cat([sums, count.double()])}
    return {**out, "rank_count": None, "sums": sums}
