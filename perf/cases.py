"""Performance cases of the Cuthill-McKee framework: the work its users have it do, through its public entry points.

A case is a dict of plain values. `kind` names the entry point:

  run      rcm_ctx_run: one order of a resident matrix from a known start (the headline measurement of bench.py)
  order    rcm_ctx_order: start search and order of a resident matrix, the order read back to the host
  batch    rcm_batch_run: every matrix of a resident set from known starts (bench.py's batched leg)
  border   rcm_batch_order: start search and order of every matrix of a set, the orders read back
  serve    rcm_server_submit / rcm_server_wait: a burst of borrowed requests, every order returned
  oneshot  rcm_gpu_batch: host CSR in, reversed order and bandwidth out
  canon    rcm_ops_canonicalize_device: shuffled lower-triangle triples to a symmetric, connected CSR
  permute  rcm_ops_permute_device: B = P A P^T with values, P the reversed order of A

`graph` names the matrix: "2d" (5-point, a x b), "3d" (7-point, a x b x c), "rgg" (random geometric, n points of mean
degree deg), "rmat" (2^scale nodes, edge factor ef, power-law hubs, components linked), or for sets "mix" (count
matrices of n_lo..n_hi rows, half stencils, half geometric graphs). All are relabelled at random from the seed, as
bench.py's are; the graph itself is the case's, so every seed gives matrices of the same size. Sizes come from
bench.py, the tests and the benchmark configurations, or are generic.
"""
import ctypes as C
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import parallelbatchrcm_amd as P
from parallelbatchrcm_amd import _native

HOST_THREADS = 16
GRAPH_SEED = 4


# ---------------------------------------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest matrices of the batched mix, one at a time: an inner solver reordering small blocks
        {"name": "run_2d_31x33", "kind": "run", "graph": "2d", "a": 31, "b": 33},
        # the 100 x 100 configuration: a user's first, small problem, start unknown
        {"name": "order_2d_100x100", "kind": "order", "graph": "2d", "a": 100, "b": 100},
        # the headline benchmark: the 128^3 stencil, one order
        {"name": "run_3d_128", "kind": "run", "graph": "3d", "a": 128, "b": 128, "c": 128},
        # the million-point geometric graph: an unstructured mesh, start unknown
        {"name": "order_rgg_1m", "kind": "order", "graph": "rgg", "n": 1000000, "deg": 12.0},
        # the serving stream's power-law member: hub rows of thousands of entries
        {"name": "order_rmat_18", "kind": "order", "graph": "rmat", "scale": 18, "ef": 16},
        # an eighth of the batched benchmark's mix, starts known
        {"name": "batch_mix_512", "kind": "batch", "graph": "mix", "count": 512, "n_lo": 1000, "n_hi": 200000},
        # a handful of small subdomain matrices, starts unknown
        {"name": "border_small_60", "kind": "border", "graph": "mix", "count": 60, "n_lo": 1000, "n_hi": 16000},
        # a burst at a reorder service
        {"name": "serve_burst_48", "kind": "serve", "graph": "mix", "count": 48, "n_lo": 1000, "n_hi": 100000},
        # one call from a host program that keeps nothing on the GPU
        {"name": "oneshot_3d_48", "kind": "oneshot", "graph": "3d", "a": 48, "b": 48, "c": 48},
        # loading the headline matrix from triples, double values
        {"name": "canon_3d_128_f64", "kind": "canon", "graph": "3d", "a": 128, "b": 128, "c": 128, "vb": 8},
        # the same for a power-law graph with many components, single values
        {"name": "canon_rmat_16_f32", "kind": "canon", "graph": "rmat", "scale": 16, "ef": 16, "vb": 4},
        # applying the headline order, double values
        {"name": "permute_3d_128_f64", "kind": "permute", "graph": "3d", "a": 128, "b": 128, "c": 128, "vb": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "order", "batch", "border", "serve", "oneshot", "canon", "permute"])
    case = {"kind": kind}
    if kind in ("batch", "border", "serve"):
        case["graph"] = "mix"
        case["count"] = _log(rng, 3, {"batch": 400, "border": 60, "serve": 48}[kind])
        case["n_lo"] = _log(rng, 500, 2000)
        case["n_hi"] = _log(rng, 4000, 150000)
        return case
    n = _log(rng, 900, 1200000)
    if kind == "oneshot":
        n = _log(rng, 900, 300000)
    case["graph"] = g = rng.choice(["2d", "3d", "rgg", "rmat"])
    if g == "2d":
        case["a"] = max(3, int(math.sqrt(n) * rng.uniform(0.5, 1.5)))
        case["b"] = max(3, n // case["a"])
    elif g == "3d":
        case["a"] = max(3, int(n ** (1 / 3) * rng.uniform(0.7, 1.3)))
        case["b"] = max(3, int(n ** (1 / 3) * rng.uniform(0.7, 1.3)))
        case["c"] = max(3, n // (case["a"] * case["b"]))
    elif g == "rgg":
        case["n"] = min(n, 800000)
        case["deg"] = round(rng.uniform(6, 14), 2)
    else:
        case["scale"] = min(17, max(10, n.bit_length() - 1))
        case["ef"] = rng.choice([4, 8, 16])
    if kind in ("canon", "permute"):
        case["vb"] = rng.choice([0, 4, 8])
    return case


# ---------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------
def _matrix(case, seed):
    g = case["graph"]
    if g == "2d":
        m = P.workloads.stencil2d(case["a"], case["b"])
    elif g == "3d":
        m = P.workloads.stencil3d(case["a"], case["b"], case["c"])
    elif g == "rgg":
        m = P.workloads.rgg(case["n"], case["deg"], GRAPH_SEED)
    else:
        m = P.workloads.rmat(case["scale"], case["ef"], seed=GRAPH_SEED)
    m, _ = P.workloads.permute_symmetric(m, seed + 1)
    return m if g in ("2d", "3d") else P.connect_components(m)[0]


def _set(case, seed):
    """The mix with every matrix relabelled from the seed."""
    bs = P.workloads.batch_mix(case["count"], case["n_lo"], case["n_hi"], GRAPH_SEED, HOST_THREADS)

    def relabelled(k):
        return P.workloads.permute_symmetric(bs.matrix(k), seed * 1000003 + k)[0]

    with ThreadPoolExecutor(HOST_THREADS) as pool:
        return list(pool.map(relabelled, range(len(bs))))


def _values(nnz, vb, seed):
    if not vb:
        return None
    g = torch.Generator().manual_seed(seed)
    return torch.randn(nnz, generator=g, dtype=torch.float64 if vb == 8 else torch.float32)


def _triples(case, seed):
    """The lower triangle (diagonal included) of a relabelled matrix, shuffled, as host tensors. The power-law graph
    keeps its components apart: the repair links them."""
    if case["graph"] == "rmat":
        m = P.workloads.rmat(case["scale"], case["ef"], seed=GRAPH_SEED)
        m, _ = P.workloads.permute_symmetric(m, seed + 1)
    else:
        m = _matrix(case, seed)
    n = m.rows
    rows = torch.repeat_interleave(torch.arange(n, dtype=torch.int32),
                                   torch.from_numpy(np.diff(m.row_offsets)).long())
    cols = torch.from_numpy(m.col_ids)
    low = cols <= rows
    rows, cols = rows[low], cols[low]
    p = torch.randperm(rows.numel(), generator=torch.Generator().manual_seed(seed))
    return n, rows[p].contiguous(), cols[p].contiguous(), _values(rows.numel(), case["vb"], seed + 2)


class _DeviceArray:
    """A device pointer of the library as something torch can view; it keeps the object that owns the memory."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, ptr, count, typestr="<i4"):
    t = torch.as_tensor(_DeviceArray(owner, ptr, count, typestr), device="cuda")
    t.owner = owner  # the view outlives whoever made the call
    return t


def _ptr(t):
    return C.c_void_p(t.data_ptr() if t is not None else None)


def _check(rc, what):
    if rc != P.RCM_OK:
        raise P.RcmError(rc, what)


def _resident(m):
    """A context with m loaded."""
    ctx = P.RcmContext()
    ctx.load(m)
    return ctx


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind}
    if kind in ("batch", "border", "serve"):
        mats = _set(case, seed)
        if kind == "serve":
            st["requests"] = mats
            st["server"] = P.RcmServer(arena_bytes=4 << 30)
            return st
        bs = P.BatchSet.from_matrices(mats)
        b = P.RcmBatch()
        b.load(bs)
        st["batch"] = b
        st["orders"] = np.empty(int(bs.n.astype(np.int64).sum()), np.int32)
        if kind == "batch":
            st["starts"] = b.order()[0]
        return st
    if kind == "canon":
        n, r, c, v = _triples(case, seed)
        st.update(n=n, vb=case["vb"], r=r.cuda(), c=c.cuda(), v=None if v is None else v.cuda(), ops=P.MatrixOps())
        return st
    m = _matrix(case, seed)
    if kind == "oneshot":
        st["m"] = m
        return st
    ctx = _resident(m)
    st["ctx"] = ctx
    if kind == "run":
        st["start"] = ctx.find_start()
    elif kind == "permute":
        ctx.order(-1, P.RCM_FLAG_REVERSE)
        v = _values(m.nnz, case["vb"], seed + 2)
        st.update(n=m.rows, nnz=m.nnz, vb=case["vb"], rp=torch.from_numpy(m.row_offsets).cuda(),
                  ci=torch.from_numpy(m.col_ids).cuda(), v=None if v is None else v.cuda(),
                  perm=torch.from_numpy(ctx.perm()).cuda(), ops=P.MatrixOps())
        st["rp_out"] = torch.empty_like(st["rp"])
        st["ci_out"] = torch.empty_like(st["ci"])
        st["v_out"] = None if v is None else torch.empty_like(st["v"])
        del st["ctx"]
        ctx.close()
    return st


# ---------------------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------------------
def run(st):
    kind, lib = st["kind"], _native.lib()
    if kind == "run":
        ctx = st["ctx"]
        ctx.run(st["start"])
        d = C.c_void_p()
        _check(lib.rcm_ctx_perm_device(ctx._h, C.byref(d)), "perm_device")
        return _view(ctx, d.value, ctx.n)
    if kind == "order":
        start, sweeps = st["ctx"].order()
        return {"perm": st["ctx"].perm(), "start": start, "sweeps": sweeps}
    if kind == "batch":
        b = st["batch"]
        _check(int(np.abs(b.run(st["starts"])).max()), "batch run")
        d = C.c_void_p()
        # the set's orders lie back to back from matrix 0's on, in load order
        _check(lib.rcm_batch_perm_device(b._h, 0, C.byref(d)), "batch_perm_device")
        return _view(b, d.value, st["orders"].size)
    if kind == "border":
        b = st["batch"]
        starts, sweeps, status = b.order()
        _check(lib.rcm_batch_read_perm(b._h, None, st["orders"].ctypes.data_as(_native.I32P)), "read_perm")
        return {"perm": st["orders"], "starts": starts, "sweeps": sweeps, "status": status}
    if kind == "serve":
        srv = st["server"]
        ids = [srv.submit(m, borrow=True) for m in st["requests"]]
        out = []
        for j in ids:
            rc, perm, _ = srv.wait(j)
            _check(rc, "serve")
            out.append(perm)
        return out
    if kind == "oneshot":
        perm, bw, start = P.rcm_gpu_batch(st["m"], -1, P.RCM_FLAG_REVERSE | P.RCM_FLAG_BANDWIDTH)
        return {"perm": perm, "bandwidth": bw, "start": start}
    ops = st["ops"]._h
    if kind == "canon":
        links = C.c_int64()
        _check(lib.rcm_ops_canonicalize_device(ops, st["n"], st["n"], st["r"].numel(), _ptr(st["r"]), _ptr(st["c"]),
                                               _ptr(st["v"]), st["vb"], 1, C.byref(links)), "canonicalize_device")
        n, nnz, rp, ci, v = C.c_int32(), C.c_int64(), C.c_void_p(), C.c_void_p(), C.c_void_p()
        _check(lib.rcm_ops_result(ops, C.byref(n), C.byref(nnz), C.byref(rp), C.byref(ci), C.byref(v)), "ops_result")
        out = {"links": links.value, "row_ptr": _view(st["ops"], rp.value, n.value + 1),
               "col_idx": _view(st["ops"], ci.value, nnz.value)}
        if st["vb"]:
            out["values"] = _view(st["ops"], v.value, nnz.value, "<f8" if st["vb"] == 8 else "<f4")
        return out
    _check(lib.rcm_ops_permute_device(ops, st["n"], st["nnz"], _ptr(st["rp"]), _ptr(st["ci"]), _ptr(st["v"]),
                                      st["vb"], _ptr(st["perm"]), _ptr(st["rp_out"]), _ptr(st["ci_out"]),
                                      _ptr(st["v_out"])), "permute_device")
    out = {"row_ptr": st["rp_out"], "col_idx": st["ci_out"]}
    if st["vb"]:
        out["values"] = st["v_out"]
    return out


# ---------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------
def _sizes(case):
    """(rows, entries), exact for the stencils, expected values for the random graphs."""
    g = case["graph"]
    if g == "2d":
        a, b = case["a"], case["b"]
        return a * b, 5 * a * b - 2 * (a + b)
    if g == "3d":
        a, b, c = case["a"], case["b"], case["c"]
        return a * b * c, 7 * a * b * c - 2 * (a * b + b * c + a * c)
    if g == "rgg":
        return case["n"], int(case["n"] * (case["deg"] + 1))
    if g == "rmat":
        return 1 << case["scale"], int((1 << case["scale"]) * (1 + 1.75 * case["ef"]))
    lo, hi = case["n_lo"], case["n_hi"]
    n = int(case["count"] * (hi - lo) / math.log(hi / lo))
    return n, int(8.46 * n)


def work(case):
    n, nnz = _sizes(case)
    kind, vb = case["kind"], case.get("vb", 0)
    if kind == "canon":  # the triples in, the CSR out
        low = (nnz + n) // 2
        return {"bytes": low * (8 + vb) + 4 * (n + 1) + nnz * (4 + vb), "flops": 0}
    if kind == "permute":  # CSR and permutation in, CSR out
        return {"bytes": 2 * (4 * (n + 1) + nnz * (4 + vb)) + 4 * n, "flops": 0}
    return {"bytes": 4 * (n + 1) + 4 * nnz + 4 * n, "flops": 0}  # CSR in, order out


# ---------------------------------------------------------------------------------------------------------
# What run() returns, from plain torch in 64 bits: the values, for the kinds that carry them. Orders, starts and
# row structures are whole numbers.
# ---------------------------------------------------------------------------------------------------------
def _component_roots(n, r, c):
    """Smallest node of every node's component."""
    root = torch.arange(n)
    while True:
        new = root.clone()
        new.scatter_reduce_(0, root[r], root[c], "amin")
        new.scatter_reduce_(0, root[c], root[r], "amin")
        new = torch.minimum(new, new[new])
        while True:
            flat = new[new]
            if torch.equal(flat, new):
                break
            new = flat
        if torch.equal(new, root):
            return root
        root = new


def exact(case, seed):
    if not case.get("vb"):
        return None
    if case["kind"] == "canon":
        n, r, c, v = _triples(case, seed)
        r, c, v = r.long(), c.long(), v.double()
        off = r != c
        root = _component_roots(n, r, c)
        heads = torch.arange(1, n)[root[1:] == torch.arange(1, n)]
        rows = torch.cat([r, c[off], heads - 1, heads])
        cols = torch.cat([c, r[off], heads, heads - 1])
        vals = torch.cat([v, v[off], torch.ones(2 * heads.numel(), dtype=torch.float64)])
        return {"links": None, "row_ptr": None, "col_idx": None, "values": vals[torch.argsort(rows * n + cols)]}
    if case["kind"] == "permute":
        m = _matrix(case, seed)
        ctx = _resident(m)  # the permutation is an input of the pass: the same whole numbers as prepare()'s
        ctx.order(-1, P.RCM_FLAG_REVERSE)
        perm = torch.from_numpy(ctx.perm()).long()
        ctx.close()
        n = m.rows
        inv = torch.empty_like(perm)
        inv[perm] = torch.arange(n)
        rows = torch.repeat_interleave(torch.arange(n), torch.from_numpy(np.diff(m.row_offsets)).long())
        key = inv[rows] * n + inv[torch.from_numpy(m.col_ids).long()]
        v = _values(m.nnz, case["vb"], seed + 2).double()
        return {"row_ptr": None, "col_idx": None, "values": v[torch.argsort(key)]}
    return None
