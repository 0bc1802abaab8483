"""The one-workgroup engine (csrc/engine_solo.hpp) against the oracle, bit for bit: on the CPU in the wave emulator,
with a small geometry whose chunks (256 slots, 128 parents) and ring (64 entries) fill, split and overflow at small
sizes, and with the library's; on the GPU through the entry points that choose it."""
import numpy as np
import pytest

import graphs as G
import oracle_lib as O
import parallelbatchrcm_amd as P

MAXROW = 64  # the longest row the engine takes


def _stencil(kind, *dims, seed=11):
    m, _ = P.workloads.permute_symmetric(getattr(P.workloads, kind)(*dims), seed)
    return m.row_offsets, m.col_ids


def _regular(n, deg, seed):
    """Every row of exactly `deg` entries (self included): a random circulant graph."""
    rng = np.random.default_rng(seed)
    steps = rng.choice(np.arange(2, n // 2), (deg - 1) // 2 - 1, replace=False)
    steps = np.concatenate([[1], steps])
    off = np.concatenate([[0], steps, n - steps])
    rows = np.sort((np.arange(n)[:, None] + off[None, :]) % n, axis=1)
    return np.arange(0, n * rows.shape[1] + 1, rows.shape[1]).astype(np.int32), rows.reshape(-1).astype(np.int32)


CASES = {
    "path1": lambda: G.path(1),
    "path2": lambda: G.path(2),
    "path300": lambda: G.path(300),  # more levels than the level boundaries kept
    "star64": lambda: G.star(MAXROW),  # the centre's row is the longest taken
    "complete40": lambda: G.complete(40),
    "random1500": lambda: G.random_connected(1500, 9000, seed=5),  # levels of several chunks, the ring overflows
    "duplicates": lambda: G.with_duplicates(*G.random_connected(300, 500, seed=7), seed=3),
    "unsorted": lambda: G.shuffle_rows(*G.random_connected(300, 900, seed=7), seed=8),
    "grid24x20": lambda: _stencil("stencil2d", 24, 20),
    "stencil11x9x13": lambda: _stencil("stencil3d", 11, 9, 13),
    "rows63": lambda: _regular(700, 63, 1),  # chunks cut inside and at rows of nearly a slot group
}


@pytest.mark.parametrize("geo", [0, 1])
def test_emulated_order_and_search(geo):
    pytest.importorskip("emu_lib")
    import emu_lib as E

    names = list(CASES) if geo == 0 else ["path2", "star64", "duplicates", "grid24x20"]
    mats = [CASES[name]() for name in names]
    for start in (lambda n: 0, lambda n: n - 1):
        starts = [start(len(rp) - 1) for rp, _ in mats]
        perms, info = E.run_solo(mats, starts, workers=3, geo=geo)
        for k, (rp, ci) in enumerate(mats):
            assert info[k, 0] == 0 and info[k, 1] == len(rp) - 1, k
            assert np.array_equal(perms[k], O.cm(rp, ci, starts[k])), (names[k], starts[k])
    for spec in (0, 2, 3) if geo == 0 else (3,):
        perms, info = E.run_solo(mats, [-1] * len(mats), workers=3, mode=2, speculate=spec, geo=geo)
        for k, (rp, ci) in enumerate(mats):
            _, s, it, _ = O.peripheral(rp, ci)
            assert (info[k, 3], info[k, 4]) == (s, it), (names[k], spec)
            assert np.array_equal(perms[k], O.cm(rp, ci, s)), (names[k], spec)


def test_emulated_full_chunks():
    """The library's geometry on levels wider than its chunks of 4096 slots."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    mats = [CASES[name]() for name in ("rows63", "random1500", "stencil11x9x13")]
    perms, info = E.run_solo(mats, [-1] * len(mats), workers=2, mode=2, geo=1)
    for k, (rp, ci) in enumerate(mats):
        _, s, it, _ = O.peripheral(rp, ci)
        assert info[k, 0] == 0 and (info[k, 3], info[k, 4]) == (s, it), k
        assert np.array_equal(perms[k], O.cm(rp, ci, s)), k


def test_emulated_directed_and_disconnected():
    pytest.importorskip("emu_lib")
    import emu_lib as E

    directed = G.directed_with_empty_rows(2000, 1500, 24, 2)
    parts = G.from_edges(10, [(0, 1), (1, 2), (5, 6)])
    perms, info = E.run_solo([directed, parts], [0, 0], workers=2, geo=0)
    assert info[0, 0] == 0 and np.array_equal(perms[0], O.cm(*directed, 0))
    assert info[1, 0] == 0 and info[1, 1] == 3 and perms[1][:3].tolist() == [0, 1, 2]


def test_emulated_watchdog():
    """A launch past its budget still gives every matrix a status."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    _, info = E.run_solo([CASES["grid24x20"](), G.path(9)], [0, 0], workers=1, geo=0, timeout_s=0.0)
    assert (info[:, 0] == 1).all()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_emulated_give_up(mode):
    """A matrix is given up at a level too wide with too much left, in whatever pass; the others of the launch are not."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    mats = [CASES["random1500"](), CASES["path300"](), CASES["star64"]()]
    nnz = [len(ci) for _, ci in mats]
    for level, spare, wide in ((2000, 1000, True), (2000, nnz[0], False), (300, 60, True)):
        gave = [wide, False, False]
        perms, info = E.run_solo(mats, [0] * 3 if mode == 0 else [-1] * 3, workers=2, mode=mode, give_up=(level, spare))
        assert (info[:, 0] == 2).tolist() == gave, (level, spare)
        for k, (rp, ci) in enumerate(mats):
            if not gave[k]:
                s = 0 if mode == 0 else O.peripheral(rp, ci)[1]
                assert info[k, 0] == 0 and info[k, 3] == s, k
                assert mode == 1 or np.array_equal(perms[k], O.cm(rp, ci, s)), k


# unsymmetric: the sweeps from nodes 2 and 3 find eccentricities 1 and 2 in turn, and no start is ever confirmed
ENDLESS = (np.array([0, 3, 6, 9, 12], np.int32), np.array([1, 2, 3, 1, 2, 3, 0, 1, 3, 0, 1, 3], np.int32))


@pytest.mark.parametrize("mode", [1, 2])
def test_emulated_endless_search(mode):
    """A search that would go on for ever, of passes too short to look at the clock, ends by the watchdog."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    assert E.run_solo([ENDLESS], [-1], workers=1, mode=mode, timeout_s=0.2)[1][0, 0] == 1
    assert E.run_team(*ENDLESS, -1, workers=2, mode=mode, timeout_s=0.2)[1][0] == 1


@pytest.mark.parametrize("engine", ["solo", "team"])
def test_emulated_watchdog_of_each_pass(engine):
    """The budget is for each pass of a search, as where each is a launch of its own."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    def order(rp, ci, timeout_s):  # looks at the clock: two a pass, and one every 64 levels
        if engine == "solo":
            perms, info = E.run_solo([(rp, ci)], [-1], workers=1, mode=2, timeout_s=timeout_s)
            return perms[0], info[0]
        return E.run_team(rp, ci, -1, workers=1, mode=2, timeout_s=timeout_s, alone=1 << 20)

    rp, ci = G.path(300)
    _, s, it, _ = O.peripheral(rp, ci)
    try:
        E.clock(0.01)
        order(rp, ci, 100.0)
        total = E.clock(0.01)
        perm, info = order(rp, ci, 0.6 * total)
        assert info[5] >= 3  # passes of equal length but for the first, half as long: none takes 0.6 of them all
        assert info[0] == 0 and (info[3], info[4]) == (s, it) and np.array_equal(perm, O.cm(rp, ci, s))
        assert order(rp, ci, 0.1 * total)[1][0] == 1
    finally:
        E.clock(0)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [30000, 40000])
def test_gpu_watchdog_of_each_pass(rows):
    """The same for a context (one workgroup, a team) and a set: a timeout that every pass keeps but not all together."""
    m = P.CSR(*G.path(rows))
    endless = P.CSR(*ENDLESS)
    print("[case]", rows, flush=True)
    with P.RcmContext(timeout_ms=20000) as c, P.RcmBatch(timeout_ms=20000) as b:
        c.load(m)
        c.run(0)
        limit = int(1.4 * c.timing().run_kernel_ms)  # the whole search and order: 2.5 passes from an end
        s, it = c.order()
        want = c.perm()
        c.set_param("timeout_ms", limit)
        assert c.order() == (s, it) and np.array_equal(c.perm(), want)
        assert c.find_start() == s
        c.set_param("timeout_ms", max(1, limit // 4))
        assert c.run_status(0) == P.RCM_ETIMEOUT
        c.set_param("timeout_ms", 20)
        c.load(endless)
        with pytest.raises(P.RcmError) as e:
            c.order()
        assert e.value.status == P.RCM_ETIMEOUT
        b.load(P.BatchSet.from_matrices([m, m, P.CSR(*G.path(9))]))
        b.run([0, 0, 0])
        b.set_param("timeout_ms", int(1.4 * b.timing().run_ms))
        starts, iters, st = b.order()
        assert not st.any() and (starts[0], iters[0]) == (s, it)
        assert all(np.array_equal(p, want) for p in b.perms()[:2])


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES) + ["rows63x9000", "rgg65536", "grid65537"])
def test_gpu_single(name):
    """rcm_ctx (search, order, run), at the largest matrix one workgroup takes alone and just beyond it."""
    big = {"rows63x9000": lambda: _regular(9000, 63, 2), "grid65537": lambda: _stencil("stencil2d", 3, 21846),
           "rgg65536": lambda: (lambda m: (m.row_offsets, m.col_ids))(P.workloads.config(3, scale=65536, seed=6))}
    rp, ci = (CASES.get(name) or big[name])()
    m = P.CSR(rp, ci)
    _, s, it, _ = O.peripheral(rp, ci)
    want = O.cm(rp, ci, s)
    print("[case]", name, m.rows, flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        assert c.order() == (s, it)
        assert np.array_equal(c.perm(), want)
        assert c.find_start() == s and c.timing().start_iterations == it
        c.run(s, P.RCM_FLAG_REVERSE)
        assert np.array_equal(c.perm(), want[::-1])
        assert c.bandwidth() == O.bandwidth(rp, ci, want)


@pytest.mark.gpu
def test_gpu_set_with_rows_for_either_engine():
    """A set of matrices for both engines (rows up to 64 and beyond), a disconnected one and one given start."""
    mats = [f() for f in CASES.values()] + [G.star(MAXROW + 1), G.hub_graph(3000, 2000, seed=3),
                                            G.from_edges(10, [(0, 1), (1, 2), (5, 6)])]
    bs = P.BatchSet.from_matrices([P.CSR(*m) for m in mats])
    given = np.full(len(mats), -1, np.int32)
    given[4] = 7
    print("[case] set", len(mats), flush=True)
    with P.RcmBatch(timeout_ms=20000) as b:
        b.load(bs)
        starts, iters, st = b.order(given)
        assert st[-1] == P.RCM_ENOTCONNECTED and not st[:-1].any()
        perms = b.perms()
        for k, (rp, ci) in enumerate(mats[:-1]):
            s, it = (7, 0) if k == 4 else O.peripheral(rp, ci)[1:3]
            assert (starts[k], iters[k]) == (s, it), k
            assert np.array_equal(perms[k], O.cm(rp, ci, s)), k
        st = b.run(starts)
        assert st[-1] == P.RCM_ENOTCONNECTED and not st[:-1].any()
        for k, p in enumerate(b.perms()[:-1]):
            assert np.array_equal(p, perms[k]), k


# members of a set, and how many workgroups run it (None: the batch engine's)
SETS = {
    "alone": (lambda: [_stencil("stencil2d", 384, 384), CASES["path300"]()], 2),  # 147,456 rows
    "too_large": (lambda: [_stencil("stencil2d", 3, 49153), CASES["path300"]()], None),  # 147,459
    "hubs": (lambda: [_stencil("stencil2d", 60, 70), G.hub_graph(3000, 2000, seed=3), CASES["random1500"](),
                      G.star(MAXROW + 1)], None),
    "long_rows": (lambda: [CASES["grid24x20"](), _regular(3000, 81, 5)], None),  # no hub: all by the batch engine
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(SETS))
def test_gpu_set_split(name):
    """Sets on either side of the rules that split them between the engines: search and order, start search, and run,
    whose graph is replayed between them."""
    mats, workgroups = SETS[name][0](), SETS[name][1]
    bs = P.BatchSet.from_matrices([P.CSR(*m) for m in mats])
    want = []
    for rp, ci in mats:
        _, s, it, _ = O.peripheral(rp, ci)
        want.append((s, it, O.cm(rp, ci, s)))
    given = np.array([s if k % 2 else -1 for k, (s, _, _) in enumerate(want)], np.int32)
    with P.RcmBatch(timeout_ms=20000, graph=True) as b:
        b.load(bs)
        for rep in range(3):
            print("[case]", name, "repeat", rep, flush=True)
            starts, iters, st = b.order(given if rep == 2 else None)
            assert not st.any() and [int(x) for x in starts] == [s for s, _, _ in want]
            assert [int(x) for x in iters] == [0 if rep == 2 and k % 2 else it for k, (_, it, _) in enumerate(want)]
            for k, p in enumerate(b.perms()):
                assert np.array_equal(p, want[k][2]), (rep, k)
            starts, iters, st = b.find_start()
            assert not st.any() and [(int(x), int(y)) for x, y in zip(starts, iters)] == [w[:2] for w in want]
            for flags in (P.RCM_FLAG_STABLE, P.RCM_FLAG_REVERSE):
                assert not b.run(starts, flags).any()
                for k, p in enumerate(b.perms()):
                    assert np.array_equal(p, want[k][2][::-1] if flags == P.RCM_FLAG_REVERSE else want[k][2]), (rep, k)
        assert b.timing().graph_replays >= 4
        assert b.timing().workers == workgroups if workgroups else b.timing().workers > len(mats)


def _box27(a, b, c):
    """The 27-point stencil on a x b x c nodes, relabelled."""
    at = np.stack(np.meshgrid(np.arange(a), np.arange(b), np.arange(c), indexing="ij"), -1).reshape(-1, 3)
    off = np.stack(np.meshgrid(*[np.arange(-1, 2)] * 3, indexing="ij"), -1).reshape(-1, 3)
    to = at[:, None] + off[None]
    inside = ((to >= 0) & (to < (a, b, c))).all(-1)
    rp = np.concatenate([[0], np.cumsum(inside.sum(1))]).astype(np.int32)
    m, _ = P.workloads.permute_symmetric(P.CSR(rp, ((to[..., 0] * b + to[..., 1]) * c + to[..., 2])[inside].astype(np.int32)), 3)
    return m.row_offsets, m.col_ids


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["random", "box27", "bar27"])
def test_gpu_wide_levels(name):
    """Matrices that one workgroup gives up (levels of a random graph, of a 27-point stencil) and one that it does not (the
    same stencil on a bar), alone, in a set with others, in one call, and in a serving lane."""
    from hip_buffers import HipBuffers
    from test_zz_no_alloc import _noalloc

    rp, ci = {"random": lambda: G.random_connected(20000, 300000, seed=3), "box27": lambda: _box27(30, 30, 30),
              "bar27": lambda: _box27(8, 8, 400)}[name]()
    m = P.CSR(rp, ci)
    _, s, it, _ = O.peripheral(rp, ci)
    want = O.cm(rp, ci, s)
    wide = name != "bar27"
    print("[case]", name, m.rows, m.nnz, flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        assert c.order() == (s, it) and np.array_equal(c.perm(), want)
        c.run(s, P.RCM_FLAG_REVERSE)
        assert np.array_equal(c.perm(), want[::-1]) and c.timing().workers == (128 if wide else 1)
        assert c.find_start() == s
        c.load(m)  # a new matrix: one workgroup is tried again
        c.run(s)
        assert np.array_equal(c.perm(), want)
    others = [P.CSR(*CASES["grid24x20"]()), P.CSR(*CASES["path300"]())]
    mats = [others[0], m, others[1]]
    starts = [O.peripheral(x.row_offsets, x.col_ids)[1] for x in mats]
    orders = [O.cm(x.row_offsets, x.col_ids, k) for x, k in zip(mats, starts)]
    for first in ("run", "reverse", "order", "find"):
        with P.RcmBatch(timeout_ms=20000, graph=True) as b:
            b.load(P.BatchSet.from_matrices(mats))
            for rep in range(3):
                if first == "order":
                    got, iters, st = b.order()
                    assert not st.any() and got.tolist() == starts and iters[1] == it
                elif first == "find":
                    got, iters, st = b.find_start()
                    assert not st.any() and got.tolist() == starts and iters[1] == it
                    assert not b.run(got).any()
                else:
                    assert not b.run(starts, P.RCM_FLAG_REVERSE if first == "reverse" else P.RCM_FLAG_STABLE).any()
                for k, p in enumerate(b.perms()):
                    assert np.array_equal(p, orders[k][::-1] if first == "reverse" else orders[k]), (first, rep, k)
            assert not b.run(starts).any() and (b.timing().workers > 3) == wide
    perm, bw, used = P.rcm_gpu_batch(m, -1, P.RCM_FLAG_BANDWIDTH)
    assert used == s and np.array_equal(perm, want) and bw == O.bandwidth(rp, ci, want)
    with HipBuffers() as hip:
        rc, perm, bw, used = _noalloc(hip, m, -1, P.RCM_FLAG_BANDWIDTH)
        assert rc == 0 and used == s and np.array_equal(perm, want) and bw == O.bandwidth(rp, ci, want)
    with P.RcmServer(lanes=2, arena_bytes=1 << 28) as srv:
        jobs = [srv.submit(x) for x in mats]
        for j, o in zip(jobs, orders):
            rc, perm, _ = srv.wait(j)
            assert rc == 0 and np.array_equal(perm, o)


@pytest.mark.gpu
def test_gpu_set_of_the_largest():
    """Beside enough others a matrix of as many rows as the bitmap has bits goes to one workgroup; one row more, and all of
    the set to the batch engine."""
    big, more = _stencil("stencil3d", 64, 64, 64), _stencil("stencil2d", 5, 52429)
    assert len(big[0]) - 1 == 1 << 18 and len(more[0]) - 1 == (1 << 18) + 1
    want = []
    for rp, ci in (big, more):
        _, s, it, _ = O.peripheral(rp, ci)
        want.append((s, it, O.cm(rp, ci, s)))
    with P.RcmBatch(timeout_ms=20000) as b:
        for mats in ([big] * 16, [big] * 15 + [more]):
            b.load(P.BatchSet.from_matrices([P.CSR(*m) for m in mats]))
            print("[case] set", len(mats), flush=True)
            starts, iters, st = b.order()
            assert not st.any()
            for k, p in enumerate(b.perms()):
                s, it, order = want[mats[k] is more]
                assert (starts[k], iters[k]) == (s, it) and np.array_equal(p, order), k
            assert not b.run(starts).any()
            assert (b.timing().workers == 16) == (mats[-1] is big)
