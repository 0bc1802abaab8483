"""The team engine (csrc/engine_team.hpp) against the oracle, bit for bit: on the CPU in the wave emulator, with a small
geometry (64 threads, 256 slots); on the GPU through a context, from the smallest matrix it takes."""
import numpy as np
import pytest

import graphs as G
import oracle_lib as O
import parallelbatchrcm_amd as P
from test_engine_solo import CASES, _regular, _stencil

SOLO = 1 << 15  # rows up to which a context leaves a matrix to one workgroup


def _lopsided(mids, fertile, tail):
    """A level of 60 * mids nodes whose first `fertile` have 60 children each and the others none, then a path: whoever
    gets the first part of that level ends with far more than a share of the next."""
    e = [(0, 1 + k) for k in range(13)]
    e += [(1 + k % 13, 14 + k) for k in range(mids)]
    order = [14 + k for j in range(13) for k in range(j, mids, 13)]  # the mids by queue position
    base = 14 + mids
    e += [(m, base + 60 * i + j) for i, m in enumerate(order) for j in range(60)]
    leaves = base + 60 * mids
    e += [(base + i, leaves + 60 * i + j) for i in range(fertile) for j in range(60)]
    n = leaves + 60 * fertile
    e += [(n - 1 + j, n + j) for j in range(tail)]
    return G.from_edges(n + tail, e)


@pytest.mark.parametrize("workers,wide,alone", [(1, 2, 50), (4, 1, 0), (3, 0, 100)])
def test_emulated_order_and_search(workers, wide, alone):
    """A leader alone, everything shared, and levels that change from one to the other; unused workgroups."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    kw = dict(workers=workers, wide=wide, alone=alone)
    for name in ("path1", "path2", "star64", "duplicates", "unsorted", "grid24x20", "random1500"):
        rp, ci = CASES[name]()
        n = len(rp) - 1
        perm, info = E.run_team(rp, ci, n - 1, tag0=0, **kw)
        assert info[0] == 0 and info[1] == n and np.array_equal(perm, O.cm(rp, ci, n - 1)), name
        _, s, it, _ = O.peripheral(rp, ci)
        perm, info = E.run_team(rp, ci, -1, mode=2, speculate=3 if alone else 0, **kw)
        assert (info[3], info[4]) == (s, it) and np.array_equal(perm, O.cm(rp, ci, s)), name


@pytest.mark.parametrize("where", [0, 1, 2])
@pytest.mark.parametrize("member", [-1, 0, 1])
def test_emulated_slow_member(where, member):
    """A member that falls behind the others by several levels' time still reads the words meant for it."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    for name in ("star64", "grid24x20", "random1500"):
        rp, ci = CASES[name]()
        _, s, it, _ = O.peripheral(rp, ci)
        for phase in (0, 3):
            perm, info = E.run_team(rp, ci, -1, mode=2, workers=4, wide=1, linger=(where, member, phase), timeout_s=30)
            assert info[0] == 0 and (info[3], info[4]) == (s, it), (name, phase)
            assert np.array_equal(perm, O.cm(rp, ci, s)), (name, phase)


def _narrow_end():
    """A tree of 1, 10, 60 and 3 nodes by level, its root n / 2, where a search begins."""
    e = [(0, 1 + k) for k in range(10)]
    e += [(1 + k // 6, 11 + k) for k in range(60)]
    e += [(11 + 7 * k, 71 + k) for k in range(3)]
    swap = {0: 37, 37: 0}
    return G.from_edges(74, [(swap.get(a, a), swap.get(b, b)) for a, b in e])


@pytest.mark.parametrize("geo", [0, 1])
@pytest.mark.parametrize("wide", [2, 3])
def test_emulated_slow_queue_entries(geo, wide):
    """A search reads the queue entries of a last level that is redistributed (narrow: few members would do), however late
    its members store them."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    rp, ci = _narrow_end()
    _, s, it, _ = O.peripheral(rp, ci)
    for phase in (2, 4, 0, 1, 3):
        perm, info = E.run_team(rp, ci, -1, mode=2, workers=4, wide=wide, linger=(3, -1, phase), geo=geo, timeout_s=30)
        assert info[0] == 0 and (info[3], info[4]) == (s, it), phase
        assert np.array_equal(perm, O.cm(rp, ci, s)), phase


def test_emulated_several_waves():
    """Workgroups of two waves: what one wave of a member leaves for the other, at the meetings, the redistributions and
    in a part of several chunks; held up at each place."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    for name in ("star64", "duplicates", "grid24x20", "random1500"):
        rp, ci = CASES[name]()
        _, s, it, _ = O.peripheral(rp, ci)
        for where in (-1, 0, 1, 2, 3):
            perm, info = E.run_team(rp, ci, -1, mode=2, workers=3, wide=2, linger=(where, -1, 3), tag0=0, geo=1,
                                    timeout_s=30)
            assert info[0] == 0 and (info[3], info[4]) == (s, it), (name, where)
            assert np.array_equal(perm, O.cm(rp, ci, s)), (name, where)
    directed = G.directed_with_empty_rows(2000, 1500, 24, 2)
    perm, info = E.run_team(*directed, 0, geo=1)
    assert info[0] == 0 and np.array_equal(perm, O.cm(*directed, 0))
    assert E.run_team(*CASES["random1500"](), 0, cap=40, geo=1)[1][0] == 2


def test_emulated_ends():
    """Directed rows, a disconnected matrix, a stage region that is too small, and the watchdog."""
    pytest.importorskip("emu_lib")
    import emu_lib as E

    directed = G.directed_with_empty_rows(2000, 1500, 24, 2)
    perm, info = E.run_team(*directed, 0)
    assert info[0] == 0 and np.array_equal(perm, O.cm(*directed, 0))
    perm, info = E.run_team(*G.from_edges(10, [(0, 1), (1, 2), (5, 6)]), 0)
    assert info[0] == 0 and info[1] == 3 and perm[:3].tolist() == [0, 1, 2]
    assert E.run_team(*CASES["random1500"](), 0, cap=40)[1][0] == 2
    assert E.run_team(*CASES["grid24x20"](), 0, timeout_s=0.0)[1][0] == 1


GPU_CASES = {
    "grid32768": lambda: _stencil("stencil2d", 128, 256),  # one workgroup's
    "grid32769": lambda: _stencil("stencil2d", 3, 10923),  # narrow: the leader's local levels throughout
    "stencil33": lambda: _stencil("stencil3d", 33, 33, 33),
    "past_bitmap": lambda: _stencil("stencil2d", 5, 52430),  # 262,150 rows: more than the leader's bitmap has bits
    "random": lambda: G.random_connected(60000, 500000, seed=9),  # a few wide levels, of several chunks a member
    "rows63": lambda: _regular(40000, 63, 3),
    "directed": lambda: G.directed_with_empty_rows(50000, 40000, 24, 2),
    "lopsided": lambda: _lopsided(780, 520, 3000),  # a stage region overflows: the batch engine takes over
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(GPU_CASES))
def test_gpu_context(name):
    rp, ci = GPU_CASES[name]()
    m = P.CSR(rp, ci)
    print("[case]", name, m.rows, flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        if name == "directed":  # only from node 0 is every node reached
            s = 0
        else:
            _, s, it, _ = O.peripheral(rp, ci)
            assert c.order() == (s, it)
            assert np.array_equal(c.perm(), O.cm(rp, ci, s))
            assert c.find_start() == s and c.timing().start_iterations == it
        for start in (s, 0):  # stages and tags of one launch under the next
            c.run(start)
            assert np.array_equal(c.perm(), O.cm(rp, ci, start))
        team = c.timing().workers == 128
        assert team == (name not in ("grid32768", "lopsided"))


@pytest.mark.gpu
def test_gpu_growing_levels():
    """Levels that grow thirtyfold stay within the members' regions: spread before the first members have claimed most of
    the next one."""
    rp, ci = G.random_connected(200000, 3000000, seed=6)
    assert np.diff(rp).max() <= 64
    m = P.CSR(rp, ci)
    print("[case]", m.rows, m.nnz, flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        c.run(7)
        assert c.timing().workers == 128
        assert np.array_equal(c.perm(), O.cm(rp, ci, 7))


@pytest.mark.gpu
def test_gpu_memory_at_load():
    """A run allocates nothing: the team's memory is there when the matrix is loaded."""
    from hip_buffers import HipBuffers

    with P.RcmContext(timeout_ms=20000) as c, HipBuffers() as hip:
        for name in ("stencil33", "past_bitmap"):
            c.load(P.CSR(*GPU_CASES[name]()))
            print("[case]", name, flush=True)
            free = hip.free_bytes()
            c.order()
            assert c.timing().workers == 128
            assert hip.free_bytes() == free


@pytest.mark.gpu
def test_gpu_reload_and_refuse():
    """A larger matrix after a smaller one (the memory grows), a disconnected one, and the smaller one again."""
    small, big = GPU_CASES["stencil33"](), G.random_connected(300000, 300000, seed=4)
    apart = G.from_edges(SOLO + 9, [(i, i + 1) for i in range(SOLO)])
    with P.RcmContext(timeout_ms=20000) as c:
        for rp, ci in (small, big, apart, small):
            print("[case]", len(rp) - 1, flush=True)
            c.load(P.CSR(rp, ci))
            if rp is apart[0]:
                with pytest.raises(P.RcmError) as e:
                    c.order()
                assert e.value.status == P.RCM_ENOTCONNECTED
            else:
                c.run(5)
                assert np.array_equal(c.perm(), O.cm(rp, ci, 5))


@pytest.mark.gpu
@pytest.mark.parametrize("entries", [(1 << 18) - 4, 1 << 18])
def test_gpu_context_with_long_rows(entries):
    """Rows beyond the level engines, either side of the count from which the batch engine's wider variant runs."""
    n = 3000
    rng = np.random.default_rng(2)
    key = np.unique(rng.integers(0, n, 2 * entries) * n + rng.integers(0, n, 2 * entries))
    a, b = key // n, key % n
    up = a < b
    a, b = a[up], b[up]
    chain = b == a + 1  # joins every node
    keep = np.concatenate([rng.permutation(np.flatnonzero(~chain))[:(entries - 2 * (n - 1) - n) // 2]])
    a, b = np.concatenate([a[keep], np.arange(n - 1)]), np.concatenate([b[keep], np.arange(1, n)])
    r = np.concatenate([a, b, np.arange(n)])
    c = np.concatenate([b, a, np.arange(n)])
    rp, ci, _ = O.convert(n, r.astype(np.int32), c.astype(np.int32), np.ones(r.size))
    assert len(ci) == entries and (rp[1:] - rp[:-1]).max() > 64
    print("[case]", entries, flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(P.CSR(rp, ci))
        _, s, it, _ = O.peripheral(rp, ci)
        assert c.order() == (s, it)
        assert np.array_equal(c.perm(), O.cm(rp, ci, s))
        assert c.timing().workers == (256 if entries >= 1 << 18 else 64)


@pytest.mark.gpu
def test_gpu_context_with_long_rows_and_narrow_levels():
    """Rows beyond the level engines, many entries, but no hub: the batch engine's default variant."""
    a, b, c = np.meshgrid(np.arange(6), np.arange(6), np.arange(300), indexing="ij")
    at = np.stack([a, b, c], -1).reshape(-1, 3)
    off = np.stack(np.meshgrid(*[np.arange(-2, 3)] * 3, indexing="ij"), -1).reshape(-1, 3)
    to = at[:, None] + off[None]
    inside = ((to >= 0) & (to < (6, 6, 300))).all(-1)
    rp = np.concatenate([[0], np.cumsum(inside.sum(1))]).astype(np.int32)
    ci = ((to[..., 0] * 6 + to[..., 1]) * 300 + to[..., 2])[inside].astype(np.int32)
    assert len(ci) >= 1 << 18 and np.diff(rp).max() > 64
    m, _ = P.workloads.permute_symmetric(P.CSR(rp, ci), 3)
    rp, ci = m.row_offsets, m.col_ids
    print("[case]", m.rows, len(ci), flush=True)
    with P.RcmContext(timeout_ms=20000) as c:
        c.load(m)
        _, s, it, _ = O.peripheral(rp, ci)
        assert c.order() == (s, it)
        assert np.array_equal(c.perm(), O.cm(rp, ci, s))
        assert c.timing().workers == 64
