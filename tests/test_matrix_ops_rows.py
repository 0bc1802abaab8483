"""Canonicalisation where the lengths of rows matter: rows around the 64 entries that are ordered in LDS, hubs among short
rows, empty rows at the edges of the groups of 64, components linked at hubs, duplicates. Against the oracle's convert
and prepareRCM, bit for bit: on the CPU in the wave emulator, on the GPU through the library."""
import numpy as np
import pytest

import emu_lib as E
import matrix_ref as M
import oracle_lib as O
import parallelbatchrcm_amd as P


def _rows_of_length(lengths, n, rng):
    """Row i holds lengths[i] random columns (with repeats), its diagonal among them."""
    r = np.repeat(np.arange(len(lengths)), lengths)
    c = rng.integers(0, n, r.size)
    first = np.concatenate([[0], np.cumsum(lengths)[:-1]])[np.asarray(lengths) > 0]
    c[first] = r[first]
    p = rng.permutation(r.size)
    return r[p].astype(np.int32), c[p].astype(np.int32)


def _symmetric(r, c):
    key = np.unique(np.concatenate([r.astype(np.int64) << 32 | c, c.astype(np.int64) << 32 | r]))
    return (key >> 32).astype(np.int32), (key & 0xFFFFFFFF).astype(np.int32)


def _edges(rng):
    """Rows of 63, 64, 65 and 200 entries next to short ones."""
    n = 300
    ln = rng.integers(1, 6, n)
    ln[[0, 63, 64, 65, 127, 128, 299]] = [64, 65, 200, 1, 63, 64, 65]
    return n, *_rows_of_length(ln, n, rng)


def _hub_components(rng):
    """Components one after the other, some of one node, the node before a link and the linked one hubs."""
    n, r, c = 400, [], []
    bounds = [0, 1, 2, 90, 91, 192, 193, 320, 400]
    for a, b in zip(bounds[:-1], bounds[1:]):
        k = 6 * (b - a)
        hub = np.concatenate([np.full(b - a, a), np.full(b - a, b - 1)])
        r += [np.arange(a, b), rng.integers(a, b, k), hub]
        c += [np.arange(a, b), rng.integers(a, b, k), np.concatenate([np.arange(a, b)] * 2)]
    return n, *_symmetric(np.concatenate(r), np.concatenate(c))


def _triangle(rng):
    """Lower triangle with a diagonal: every pair gets its transpose."""
    n = 700
    a, b = rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n)
    keep = a != b
    key = np.unique(np.maximum(a, b)[keep].astype(np.int64) << 32 | np.minimum(a, b)[keep])
    r = np.concatenate([key >> 32, np.arange(n)])
    c = np.concatenate([key & 0xFFFFFFFF, np.arange(n)])
    p = rng.permutation(r.size)
    return n, r[p].astype(np.int32), c[p].astype(np.int32)


def _mixed(rng):
    """Pairs stored one to four times, in one direction or both, odd and even, and repeated diagonals."""
    n = 500
    r, c = _rows_of_length(rng.integers(1, 9, n), n, rng)
    again = rng.integers(0, r.size, r.size // 3)
    flip = rng.integers(0, r.size, r.size // 4)
    # doubled one-sided pairs would be unsymmetric: where that is so the directed repair is what is compared
    return n, np.concatenate([r, r[again], c[flip]]), np.concatenate([c, c[again], r[flip]])


def _one_long_row(rng):
    """Small enough for the buckets, but with a row that is not ordered by counting, full of duplicates."""
    n = 300
    r, c = np.full(150, 7), rng.integers(0, 40, 150)
    return n, *(np.concatenate(p).astype(np.int32) for p in ((r, np.arange(n)), (c, np.arange(n))))


def _past_a_bucket(rng):
    """A row that no bucket holds: the sort by digits."""
    n = 20000
    r, c = np.full(9000, 7), rng.integers(0, n, 9000)
    return n, *(np.concatenate(p).astype(np.int32) for p in ((r, np.arange(n)), (c, np.arange(n))))


def _directed_chain(rng):
    """Nothing reaches a node from below except links; row x already holds x - 1, the column that its link adds."""
    n = 200
    r = np.concatenate([np.arange(n), np.arange(1, n)])
    c = np.concatenate([np.arange(n), np.arange(n - 1)])
    return n, r.astype(np.int32), c.astype(np.int32)


CASES = {"edges": (_edges, True), "hub_components": (_hub_components, True), "hub_components_as_is": (_hub_components, False),
         "triangle": (_triangle, True), "mixed": (_mixed, True),
         "one_long_row": (_one_long_row, True), "past_a_bucket": (_past_a_bucket, True), "directed_chain": (_directed_chain, False)}


def _check(name, canonicalize):
    make, check_sym = CASES[name]
    rng = np.random.default_rng(len(name))
    n, r, c = make(rng)
    v = rng.integers(-99, 99, r.size).astype(np.float64)
    orp, oci, ov = O.convert(n, r, c, v)
    added, erp, eci, ev = O.prepare_values(orp, oci, ov, check_sym)
    assert added >= 0
    rp, ci, vv, links = canonicalize(n, r, c, v, check_sym)
    assert links == added
    np.testing.assert_array_equal(rp, erp)
    np.testing.assert_array_equal(ci, eci)
    np.testing.assert_array_equal(vv, ev)


@pytest.mark.parametrize("name", [c for c in CASES if c != "past_a_bucket"])
def test_emulated(name):
    def run(n, r, c, v, check_sym):
        rc, res = E.canonicalize(n, n, r, c, v, check_sym)
        assert rc == 0
        return res[1:]

    _check(name, run)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_gpu(name):
    print("[case]", name, flush=True)
    with P.MatrixOps() as ops:
        def run(n, r, c, v, check_sym):
            m, links = ops.canonicalize(n, n, r, c, v, check_sym)
            return m.row_offsets, m.col_ids, m.data, links

        _check(name, run)


def _permute_case(n):
    """Rows of 0 to 66 entries in unsorted order, and groups of 64 rows that divide by the 8 XCDs or leave a rest."""
    rng = np.random.default_rng(n)
    ln = rng.integers(0, 9, n)
    ln[rng.integers(0, n, 3)] = [63, 64, 66]
    rp = np.concatenate([[0], np.cumsum(ln)]).astype(np.int32)
    ci = rng.integers(0, n, rp[-1]).astype(np.int32)
    return P.CSR(rp, ci, rng.standard_normal(ci.size)), rng.permutation(n).astype(np.int32)


def _check_permuted(m, perm, rp, ci, v):
    erp, eci, ev = M.permute_ref(m.row_offsets, m.col_ids, m.data, perm)
    np.testing.assert_array_equal(rp, erp)
    np.testing.assert_array_equal(ci, eci)
    np.testing.assert_array_equal(v, ev)


@pytest.mark.parametrize("n", [5, 64, 511, 513, 1088])
def test_emulated_permute(n):
    m, perm = _permute_case(n)
    rc, rp, ci, v = E.permute(m.row_offsets, m.col_ids, m.data, perm)
    assert rc == 0
    _check_permuted(m, perm, rp, ci, v)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5, 64, 511, 513, 1088, 70001])
def test_gpu_permute(n):
    print("[case] permute", n, flush=True)
    m, perm = _permute_case(n)
    with P.MatrixOps() as ops:
        b = ops.permute(m, perm)
    _check_permuted(m, perm, b.row_offsets, b.col_ids, b.data)
