"""GPU: which engine a context and a set run is a matter of their parameters alone: putting one back to the value that was
read brings the automatic choice back, and with WORKERS set the default variant's batch engine runs every matrix."""
import numpy as np
import pytest

import graphs as G
import oracle_lib as O
import parallelbatchrcm_amd as P
from test_engine_solo import CASES

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _want(rp, ci):
    _, s, it, _ = O.peripheral(rp, ci)
    return s, it, O.cm(rp, ci, s)


@pytest.mark.parametrize("workers", [0, 64])
def test_context(workers):
    """Every short-row case by the level engine, and by the default variant of the batch engine."""
    with P.RcmContext(timeout_ms=20000, workers=workers) as c:
        for name in CASES:
            rp, ci = CASES[name]()
            _say(name, workers)
            s, it, order = _want(rp, ci)
            c.load(P.CSR(rp, ci))
            assert c.order() == (s, it) and np.array_equal(c.perm(), order), name
            assert c.find_start() == s, name
            c.run(s)
            assert np.array_equal(c.perm(), order), name
            assert c.timing().workers == (workers or 1), name


@pytest.mark.parametrize("name,value", [("variant", 3), ("claim_filter", 0), ("sort", 2), ("workers", 32), ("strict", 1)])
def test_context_parameter_put_back(name, value):
    rp, ci = CASES["random1500"]()
    s, _, order = _want(rp, ci)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(P.CSR(rp, ci))
        keep = c.get_param(name)
        for v, workers in ((value, 32 if name == "workers" else 64), (keep, 1)):
            c.set_param(name, v)
            _say(name, v)
            c.run(s)
            assert np.array_equal(c.perm(), order) and c.timing().workers == workers, v


def test_set_variant_put_back():
    mats = [CASES["grid24x20"](), CASES["random1500"](), G.path(9)]
    want = [_want(*m) for m in mats]
    with P.RcmBatch(timeout_ms=20000) as b:
        b.load(P.BatchSet.from_matrices([P.CSR(*m) for m in mats]))
        few = []
        for v in (3, 4):  # 4: the default
            b.set_param("variant", v)
            _say("variant", v)
            assert not b.run([w[0] for w in want]).any()
            assert all(np.array_equal(p, w[2]) for p, w in zip(b.perms(), want))
            few.append(b.timing().workers == len(mats))
        assert few == [False, True]


@pytest.mark.parametrize("bad", ["start", "time"])
def test_set_after_a_failed_tuning(bad):
    """A tuning that ends with an error leaves the engines as they were."""
    mats = [P.workloads.config(3, scale=60000, seed=3)] * 2 + [P.CSR(*G.path(9))]
    want = [_want(m.row_offsets, m.col_ids) for m in mats]
    starts = [w[0] for w in want]
    with P.RcmBatch(timeout_ms=20000) as b:
        b.load(P.BatchSet.from_matrices(mats))
        _say("tuning", bad)
        if bad == "time":
            b.set_param("timeout_ms", 1)
        with pytest.raises(P.RcmError):
            b.autotune([-1] * 3 if bad == "start" else starts)
        b.set_param("timeout_ms", 20000)
        assert not b.run(starts).any()
        assert all(np.array_equal(p, w[2]) for p, w in zip(b.perms(), want))
        assert b.timing().workers == len(mats)


@pytest.mark.parametrize("graph", ["level", "hub"])
def test_tuning_times_the_default(graph):
    """default_ms is what a context or set with nothing chosen takes, not a variant that no default call runs."""
    m = P.workloads.config(3, scale=40000, seed=3) if graph == "level" else P.CSR(*G.hub_graph(5000, 9000, seed=1))
    s, _, order = _want(m.row_offsets, m.col_ids)
    _say(graph)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        times = []
        for _ in range(9):
            c.run(s)
            times.append(c.timing().run_kernel_ms)
        r = c.autotune(s, repeats=5)
        assert 0 < r.best_ms <= r.default_ms and min(times) / 2 < r.default_ms < 2 * max(times)
        assert r.workers > 0 or r.variant == 5
        c.run(s)
        assert np.array_equal(c.perm(), order)
    with P.RcmBatch(timeout_ms=20000) as b:
        b.load(P.BatchSet.from_matrices([m] * 3))
        times = []
        for _ in range(9):
            assert not b.run([s] * 3).any()
            times.append(b.timing().run_ms)
        r = b.autotune([s] * 3, repeats=5)
        assert 0 < r.best_ms <= r.default_ms and min(times) / 2 < r.default_ms < 2 * max(times)
        assert not b.run([s] * 3).any()
        assert all(np.array_equal(p, order) for p in b.perms())


def test_speculate_beyond_32_bits():
    """A sweep number that no search reaches means no speculation, however large."""
    rp, ci = CASES["grid24x20"]()
    _say("speculate")
    with P.RcmContext(timeout_ms=20000) as c, P.RcmBatch(timeout_ms=20000) as b:
        c.load(P.CSR(rp, ci))
        b.load(P.BatchSet.from_matrices([P.CSR(rp, ci)]))
        passes = []
        for v in (0, (1 << 32) + 1, 1):
            c.set_param("speculate", v)
            b.set_param("speculate", v)
            s, it = c.order()
            assert np.array_equal(c.perm(), O.cm(rp, ci, s))
            assert b.order()[0][0] == s and np.array_equal(b.perms()[0], c.perm())
            passes.append(c.timing().order_passes)
        assert passes[0] == passes[1] == it + 1 and passes[2] > it + 1
