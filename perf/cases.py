"""Performance cases: what a DMRG or exact-diagonalisation program has this library do.

A DMRG step builds the superblock of two renormalised blocks and two sites, solves for its
ground state (Kronecker form, assembled CRS or the matrix-free product), truncates
the left half through its density matrices, renormalises the block operators and, for
expectation values, applies operators that change the sector.  Beside it stand batches of
exact-diagonalisation problems.  Every case is one such call, through the entry points that
programs use, from the arrays that they hold.

The blocks come from the superblocks of recorded DMRG runs (XXZ, Hubbard and Kondo lattice
chains, tests/golden/): a case with m kept states takes the m states of highest weight of the
recorded block, so that any size up to the recorded one has a block's real quantum
numbers, operator sparsity and spectrum.  The seed sets the couplings.
"""
import ctypes as C
import functools
import math
import os

import numpy as np
import torch

import dmrg_c_amd as D
from dmrg_c_amd import ed, engine, snapshot

GOLDEN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(D.__file__))), "tests", "golden")
RECORDED = {"xxz": "xxz_L64_m300_s31", "hubbard": "hubbard_L64_m400_s31", "klm": "klm_L48_m800_s23"}
# states of the recorded blocks, and products (Lanczos steps + CG iterations) of their solves
M_MAX = {"xxz": 162, "hubbard": 396, "klm": 799}
PRODUCTS = {"xxz": 200, "hubbard": 250, "klm": 780}


# --------------------------------------------------------------------------- the cases
def listed():
    return [
        # early steps of a run: superblocks of about a thousand states, where a solve is a long
        # chain of very short products
        {"name": "kron_hubbard_m32", "path": "kron", "model": "hubbard", "m": 32},
        # steps of a production spin chain and of a Hubbard chain at m = 400
        {"name": "kron_xxz_m162", "path": "kron", "model": "xxz", "m": 162},
        {"name": "kron_hubbard_m396", "path": "kron", "model": "hubbard", "m": 396},
        # the largest superblock: Kondo lattice at m = 800, two million states
        {"name": "kron_klm_m799", "path": "kron", "model": "klm", "m": 799},
        # the reference's own structure: the CRS assembled on the device, then the same solve
        {"name": "crs_xxz_m162", "path": "crs", "model": "xxz", "m": 162, "precision": 0},
        # assembly of a large CRS (13 million stored elements) and one product with it
        {"name": "assemble_hubbard_m396", "path": "assemble", "model": "hubbard", "m": 396},
        # one product with a CRS far larger than the caches (0.7 billion elements), in the form
        # that the schedule tuner picks for it
        {"name": "product_klm_m799", "path": "product", "model": "klm", "m": 799, "tuned": True},
        # truncation of the m = 400 step: density matrices, their eigenpairs, the kept states
        {"name": "truncate_hubbard_m396", "path": "truncate", "model": "hubbard", "m": 396},
        # renormalisation of one block operator of that step, T^dagger O T
        {"name": "renormalise_hubbard_m396", "path": "renormalise", "model": "hubbard", "m": 396},
        # an operator that takes the ground state into the sector of one spin flip
        {"name": "sector_hubbard_m396", "path": "sector", "model": "hubbard", "m": 396},
        # the matrix-free path, for superblocks whose CRS a program does not want to hold
        {"name": "matrix_free_xxz_m100", "path": "matrix_free", "model": "xxz", "m": 100},
        # a sweep over couplings by exact diagonalisation: chains of mixed lengths, FP32 values
        # with FP64 refinement
        {"name": "ed_batch_32", "path": "ed_batch", "count": 32, "l_max": 18, "precision": 1},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["kron", "kron", "crs", "assemble", "product", "truncate", "renormalise", "sector",
                       "matrix_free", "ed_batch"])
    if path == "ed_batch":
        return {"path": path, "count": log_int(2, 32), "l_max": rng.choice([12, 14, 16, 18]),
                "precision": rng.choice([0, 1])}
    if path == "matrix_free":
        return {"path": path, "model": "xxz", "m": log_int(12, 100)}
    model = rng.choice(["xxz", "hubbard", "klm"])
    # the largest block of a draw: where the case would cost more than the listed ones, less
    top = {"kron": {}, "crs": {"hubbard": 200, "klm": 100}, "assemble": {"klm": 200}, "product": {},
           "truncate": {"klm": 250}, "renormalise": {"klm": 250}, "sector": {"klm": 250}}[path]
    case = {"path": path, "model": model, "m": log_int(16, top.get(model, M_MAX[model]))}
    if path == "crs":
        case["precision"] = rng.choice([0, 0, 1, 2])
    if path == "product":
        case["tuned"] = rng.choice([False, True])
    return case


# ------------------------------------------------------------- blocks and their operators
@functools.lru_cache(maxsize=None)
def _recorded(model):
    s = snapshot.load(os.path.join(GOLDEN, RECORDED[model] + ".npz"))
    z = np.load(os.path.join(GOLDEN, "qn_" + RECORDED[model] + ".npz"))
    q = {k: z[k].astype(np.int32) for k in ("sz_LL", "ele_LL", "sz_RR", "ele_RR", "sz_site", "ele_site")}
    n_qn, _, _, _, t_sz, t_ele = (int(v) for v in z["header"])
    q.update(n_qn=n_qn, target_sz=t_sz, target_ele=t_ele)
    return s, q


def _heaviest(sz, ele, m):
    """The m states kept first: within a quantum number the recorded block lists its states by
    falling weight."""
    rank = np.zeros(len(sz))
    keys = ele.astype(np.int64) * 1000 + sz
    for k in np.unique(keys):
        at = np.nonzero(keys == k)[0]
        rank[at] = (np.arange(len(at)) + 0.5) / len(at)
    return np.sort(np.argsort(rank, kind="stable")[:m])


def _sub_crs(o, keep):
    a = o.to_dense()[np.ix_(keep, keep)]
    r, c = np.nonzero(a)
    row = np.zeros(len(keep) + 1, np.int64)
    np.add.at(row, r + 1, 1)
    return snapshot.Crs(len(keep), len(keep), np.cumsum(row), c.astype(np.int32), a[r, c])


@functools.lru_cache(maxsize=4)
def _block(model, m):
    """(operators, parity arrays, terms, quantum numbers) of the superblock with m states a side."""
    s, q = _recorded(model)
    keep = _heaviest(q["sz_LL"], q["ele_LL"], m)
    ops = [_sub_crs(o, keep) if o.row_dim == s.dim_LL else o for o in s.ops]
    eles = [e[keep] if len(e) == s.dim_LL else e for e in s.eles]
    q = dict(q)
    for k in ("sz_LL", "ele_LL", "sz_RR", "ele_RR"):
        q[k] = q[k][keep]
    return ops, eles, s.terms, q


def _superblock(case, seed):
    """The snapshot and quantum numbers that a program hands over, with the seed's couplings."""
    ops, eles, terms, q = _block(case["model"], case["m"])
    rng = np.random.default_rng(seed)
    terms = terms.copy()
    one, left, right, mid = rng.uniform(0.9, 1.1, 4)
    for k, f in (("LL", 1.0), ("RR", 1.0), ("LR", one), ("RL", one), ("LLLR", left), ("RRRL", right), ("LRRL", mid)):
        terms["coeff"][terms["kind"] == snapshot.KIND_NAMES.index(k)] *= f
    m, d = case["m"], len(q["sz_site"])
    none = np.zeros(0, np.int16)
    return snapshot.Snapshot(0, m, m, d, 0, 0, 0, none, none, none, none, ops, eles, terms), q


def _halves(q, side):
    """Quantum numbers of the (block, site) states of one half, block-major."""
    d = len(q["sz_site"])
    m = len(q["sz_" + side])
    site = np.tile(np.arange(d), m)
    block = np.repeat(np.arange(m), d)
    return block, site, q["ele_" + side][block] + q["ele_site"][site], q["sz_" + side][block] + q["sz_site"][site]


def _sectors(q, target=None):
    """The superblock basis as a program's GET_BASIS_SUPERBLOCK has it: per quantum number of the
    left half (electrons, then spin) its left states and the right states that complete it."""
    te, ts = target if target else (q["target_ele"], q["target_sz"])
    _, _, ea, sa = _halves(q, "LL")
    _, _, eb, sb = _halves(q, "RR")
    out = []
    for e, s in sorted(set(zip(ea.tolist(), sa.tolist()))):
        left = np.nonzero((ea == e) & (sa == s))[0]
        right = np.nonzero((eb == te - e) & (sb == ts - s))[0]
        if len(left) and len(right):
            out.append((e, s, left, right))
    return out


def _basis_arrays(q, target=None):
    """LL, LR, RR, RL of every superblock state."""
    d = len(q["sz_site"])
    a = np.concatenate([np.repeat(x, len(y)) for _, _, x, y in _sectors(q, target)])
    b = np.concatenate([np.tile(y, len(x)) for _, _, x, y in _sectors(q, target)])
    return [np.ascontiguousarray(v, np.int16) for v in (a // d, a % d, b // d, b % d)]


def _dims(case):
    q = _block(case["model"], case["m"])[3]
    return [(len(x), len(y)) for _, _, x, y in _sectors(q)]


# ------------------------------------------------------------------------ ground states
def _aligned(vec, like):
    """An eigenvector is defined up to its sign; a program that follows a state from step to step
    keeps the sign of the one before."""
    if np.dot(vec, like) < 0.0:
        np.negative(vec, out=vec)
    return vec


def _prepare_solve(case, seed):
    snap, q = _superblock(case, seed)
    n = sum(a * b for a, b in _dims(case))
    return {"snap": snap, "qn": q, "like": np.random.default_rng([seed, 1]).standard_normal(n)}


def _run_kron(s):
    sb = D.Superblock(s["snap"], s["qn"])
    K = sb.kron()
    energy, vec, _ = K.ground_state()
    K.free()
    sb.free()
    return {"energy": energy, "vec": _aligned(vec, s["like"])}


def _run_crs(s):
    sb = D.Superblock(s["snap"], s["qn"])
    A = sb.assemble()
    energy, vec, _ = A.ground_state(precision=s["precision"])
    A.free()
    sb.free()
    return {"energy": energy, "vec": _aligned(vec, s["like"])}


# ------------------------------------------------------------------- CRS and its product
def _prepare_assemble(case, seed):
    s = _prepare_solve(case, seed)
    s["x"] = torch.from_numpy(s.pop("like")).cuda()
    s["y"] = torch.empty_like(s["x"])
    s["sb"] = D.Superblock(s["snap"], s["qn"])
    return s


def _product(A, x, y):
    D.check(D.lib().dmrgx_spmv_device(A.handle, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr())))
    return y


def _run_assemble(s):
    A = s["sb"].assemble()
    y = _product(A, s["x"], s["y"])
    A.free()
    return y


def _prepare_product(case, seed):
    s = _prepare_assemble(case, seed)
    s["A"] = s["sb"].assemble()
    s["sb"].free()
    if case["tuned"]:   # sliced form, 16-bit columns, non-temporal loads one group ahead
        s["A"].set_schedule(1, 8192, 91)
    _product(s["A"], s["x"], s["y"])   # the form's arrays are laid out once per matrix
    return s


def _run_product(s):
    return _product(s["A"], s["x"], s["y"])


# ------------------------------------------------- truncation, renormalisation, sectors
def _dmrg_basis(q):
    """DMRG_BASIS with the superblock, its inverse and the LLLR states."""
    d, m = len(q["sz_site"]), len(q["sz_LL"])
    LL, LR, RR, RL = _basis_arrays(q)
    dims = (m, d, m, d)
    inv = np.full(int(np.prod(dims)), -1, np.int32)
    inv[np.ravel_multi_index([a.astype(np.int64) for a in (LL, LR, RR, RL)], dims)] = np.arange(len(LL), dtype=np.int32)
    left = np.concatenate([x for _, _, x, _ in _sectors(q)])
    hold = {"LL_LLLRRRRL": LL, "LR_LLLRRRRL": LR, "RR_LLLRRRRL": RR, "RL_LLLRRRRL": RL, "Inv_LLLRRRRL": inv,
            "LL_LLLR": np.ascontiguousarray(left // d, np.int16), "LR_LLLR": np.ascontiguousarray(left % d, np.int16),
            "Sum_LLLR": np.concatenate([np.full(len(x), len(y), np.int32) for _, _, x, y in _sectors(q)])}
    B = D.DMRG_BASIS()
    for k, a in hold.items():
        setattr(B, k, a.ctypes.data_as(C.POINTER(C.c_int if a.dtype == np.int32 else C.c_short)))
    B.dim_LLLRRRRL, B.dim_LL, B.dim_RR, B.dim_onsite, B.dim_LLLR = len(LL), m, m, d, len(left)
    q1 = np.concatenate([np.full(len(x), e, np.int32) for e, _, x, _ in _sectors(q)])
    q2 = np.concatenate([np.full(len(x), s, np.int32) for _, s, x, _ in _sectors(q)])
    return B, hold, q1, q2


def _reflected(rng, rows, cols, diag):
    """A rows x cols matrix with the singular values diag, its singular vectors mixed by three
    reflections a side."""
    a = np.zeros((rows, cols))
    np.fill_diagonal(a, diag)
    for _ in range(3):
        u, v = rng.standard_normal(rows), rng.standard_normal(cols)
        a -= np.outer(u * (2.0 / u.dot(u)), u @ a)
        a -= np.outer(a @ v, v * (2.0 / v.dot(v)))
    return a


def _schmidt_state(q, seed):
    """A normalised state whose Schmidt values fall off as a ground state's do: fast within each
    quantum number, and away from the middle one.  The values are the case's, the states the
    seed's."""
    rng, values = np.random.default_rng([seed, 2]), np.random.default_rng(len(q["sz_LL"]))
    out = []
    e0, s0 = q["target_ele"] / 2.0, q["target_sz"] / 2.0
    for e, s, left, right in _sectors(q):
        k = min(len(left), len(right))
        w = math.exp(-0.25 * ((e - e0) ** 2 + (s - s0) ** 2))
        sv = w * 10.0 ** (-4.0 * (np.arange(k) + values.uniform(0.0, 0.5, k)) / k)
        out.append(_reflected(rng, len(left), len(right), sv).ravel())
    v = np.concatenate(out)
    return v / np.linalg.norm(v)


def _prepare_truncate(case, seed):
    q = _block(case["model"], case["m"])[3]
    B, hold, q1, q2 = _dmrg_basis(q)
    L = D.lib()
    L.dmrgx_get_system_info.argtypes = [C.c_int32, C.c_void_p, C.c_void_p, C.POINTER(D.DMRG_BASIS), C.c_void_p,
                                        C.c_int32, C.POINTER(C.POINTER(D.DMRG_SYSTEM_INFO))]
    L.dmrgx_free_system_info.argtypes = [C.POINTER(D.DMRG_SYSTEM_INFO)]
    return {"B": B, "hold": hold, "q1": q1, "q2": q2, "vec": _schmidt_state(q, seed), "m": case["m"]}


def _run_truncate(s):
    L = D.lib()
    out = C.POINTER(D.DMRG_SYSTEM_INFO)()
    D.check(L.dmrgx_get_system_info(2, s["q1"].ctypes.data, s["q2"].ctypes.data, C.byref(s["B"]),
                                    s["vec"].ctypes.data, s["m"], C.byref(out)))
    S = out.contents
    k, T = S.dim_renorm, S.Trans_Matrix.contents
    arr = np.ctypeslib.as_array
    col = arr(T.Col, (k + 1,)).copy()
    res = {"weights": arr(S.Val_DM_Dist, (S.dim_LLLR,)).copy(), "discarded": S.tr_error, "kept": k,
           "q1": arr(S.Q_Number1, (k,)).copy(), "q2": arr(S.Q_Number2, (k,)).copy(), "col": col,
           "row": arr(T.Row, (int(col[k]),)).copy(),
           # a kept state is defined up to its sign
           "val": np.abs(arr(T.Val, (int(col[k]),)))}
    L.dmrgx_free_system_info(out)
    return res


def _left_operator(case, seed):
    """The Hamiltonian of block and site as one CRS on the left half's states, sector by sector."""
    snap, q = _superblock(case, seed)
    h = _half_dense(snap, q, "LL", "cpu").numpy()
    left = np.concatenate([x for _, _, x, _ in _sectors(q)])
    return h[np.ix_(left, left)], q


def _prepare_renormalise(case, seed):
    h, q = _left_operator(case, seed)
    rng = np.random.default_rng([seed, 3])
    n = h.shape[0]
    share = case["m"] / n
    cols, at = [], 0
    for _, _, left, _ in _sectors(q):
        d, k = len(left), max(1, int(round(share * len(left))))
        block = np.zeros((n, k))
        block[at:at + d] = _reflected(rng, d, k, np.ones(k))
        cols.append(block)
        at += d
    T = np.concatenate(cols, axis=1)
    k = T.shape[1]

    def crs(a):
        r, c = np.nonzero(a)
        ptr = np.zeros(a.shape[0] + 1, np.int64)
        np.add.at(ptr, r + 1, 1)
        return [np.cumsum(ptr), c.astype(np.int32), np.ascontiguousarray(a[r, c])]

    t, o = crs(T.T), crs(h)   # the CCS of T is the CRS of its transpose
    i32, i64 = C.POINTER(C.c_int), C.POINTER(C.c_long)

    def struct(kind, a, rows, cols_, rank, outer):
        ptr, idx, val = a
        ip, pp, vp = idx.ctypes.data_as(i32), ptr.ctypes.data_as(i64), val.ctypes.data_as(C.POINTER(C.c_double))
        x = kind(len(val), outer + 1, rows, cols_)
        x.Val = vp
        x.Col, x.Row = (ip, pp) if rank == "crs" else (pp, ip)
        return x

    res = [np.zeros(k + 1, np.int64), np.zeros(k * k + 1, np.int32), np.zeros(k * k + 1)]
    work = [np.zeros(k + 1, np.int64), np.zeros(n * k + 1, np.int32), np.zeros(n * k + 1)]
    fn = D.lib().CRS_CRS_CCS_PRODUCT
    fn.argtypes = [C.POINTER(D.CRS1), C.POINTER(D.CRS1), C.POINTER(D.CCS1), C.POINTER(D.CRS1), C.POINTER(D.CCS1),
                   C.c_void_p]
    fn.restype = None
    return {"k": k, "hold": (t, o, work), "res": res, "vec": np.zeros(n), "T": T, "h": h,
            "m1": struct(D.CRS1, t, k, n, "crs", k), "m2": struct(D.CRS1, o, n, n, "crs", n),
            "m3": struct(D.CCS1, t, n, k, "ccs", k), "out": struct(D.CRS1, res, 0, 0, "crs", k),
            "work": struct(D.CCS1, work, 0, 0, "ccs", k)}


def _run_renormalise(s):
    D.lib().CRS_CRS_CCS_PRODUCT(C.byref(s["m1"]), C.byref(s["m2"]), C.byref(s["m3"]), C.byref(s["out"]),
                                C.byref(s["work"]), s["vec"].ctypes.data)
    row, col, val = s["res"]
    n = int(row[s["k"]])
    return {"row": row, "col": col[:n], "val": val[:n]}


def _raised(q):
    """The sector that one spin flip leads to."""
    return q["target_ele"], q["target_sz"] + 2


def _raising(q, seed):
    """A block operator with the pattern of S^+: same electrons, S^z up by one."""
    rng = np.random.default_rng([seed, 4])
    e, s = q["ele_LL"], q["sz_LL"]
    mask = (e[:, None] == e[None, :]) & (s[:, None] == s[None, :] + 2)
    return np.where(mask, rng.uniform(-1.0, 1.0, mask.shape), 0.0)


def _prepare_sector(case, seed):
    q = _block(case["model"], case["m"])[3]
    d, m = len(q["sz_site"]), case["m"]
    dims = (m, d, m, d)
    inv = np.full(int(np.prod(dims)), -1, np.int32)
    basis = {}
    for name, target in (("in", None), ("out", _raised(q))):
        basis[name] = _basis_arrays(q, target)
        flat = np.ravel_multi_index([a.astype(np.int64) for a in basis[name]], dims)
        inv[flat] = np.arange(len(flat), dtype=np.int32)
    W = D.WholeBasis(m, m, d, inv)
    op = _raising(q, seed)
    r, c = np.nonzero(op)
    row = np.zeros(m + 1, np.int64)
    np.add.at(row, r + 1, 1)
    x = np.random.default_rng([seed, 5]).standard_normal(len(basis["in"][0]))
    return {"W": W, "sector": W.add_sector(*basis["out"]), "op": (np.cumsum(row), c.astype(np.int32), op[r, c]),
            "x": x / np.linalg.norm(x)}


def _run_sector(s):
    return s["W"].v_m(0, s["op"], s["sector"], s["x"])


# ---------------------------------------------------------------------- matrix-free path
def _prepare_matrix_free(case, seed):
    snap, q = _superblock(case, seed)
    B, hold, _, _ = _dmrg_basis(q)
    d, m = len(q["sz_site"]), case["m"]

    def sub(block, site, inv_rows, inv_cols, name):
        """Sub-basis in its first-appearance order, with its inverse."""
        key = block.astype(np.int64) * inv_cols + site
        _, first = np.unique(key, return_index=True)
        order = key[np.sort(first)]
        inv = np.full((inv_rows, inv_cols), -1, np.int32)
        inv.ravel()[order] = np.arange(len(order), dtype=np.int32)
        a, b = (np.ascontiguousarray(v, np.int16) for v in (order // inv_cols, order % inv_cols))
        rows = (C.POINTER(C.c_int) * inv_rows)(*[inv[i].ctypes.data_as(C.POINTER(C.c_int)) for i in range(inv_rows)])
        hold[name] = (a, b, inv, rows)
        return a, b, order, C.cast(rows, C.POINTER(C.POINTER(C.c_int)))

    short = lambda a: a.ctypes.data_as(C.POINTER(C.c_short))  # noqa: E731
    LL, LR, RR, RL = (hold[k + "_LLLRRRRL"] for k in ("LL", "LR", "RR", "RL"))
    a, b, left, B.Inv_LLLR = sub(LL, LR, m, d, "LLLR")
    B.LL_LLLR, B.LR_LLLR, B.dim_LLLR = short(a), short(b), len(left)
    a, b, mid, B.Inv_LRRL = sub(LR, RL, d, d, "LRRL")
    B.LR_LRRL, B.RL_LRRL, B.dim_LRRL = short(a), short(b), len(mid)
    a, b, right, B.Inv_RRRL = sub(RR, RL, m, d, "RRRL")
    B.RR_RRRL, B.RL_RRRL, B.dim_RRRL = short(a), short(b), len(right)

    def crs(a):
        r, c = np.nonzero(a)
        row = np.zeros(a.shape[0] + 1, np.int64)
        np.add.at(row, r + 1, 1)
        return D.HostCRS(np.cumsum(row), c.astype(np.int32), a[r, c], a.shape[0])

    mats = {"LLLR": crs(_half_dense(snap, q, "LL", "cpu").numpy()[np.ix_(left, left)]),
            "RRRL": crs(_half_dense(snap, q, "RR", "cpu").numpy()[np.ix_(right, right)]),
            "LRRL": crs(_middle_dense(snap)[np.ix_(mid, mid)]),
            "sign": D.HostCRS(np.zeros(len(left) + 1, np.int64), np.zeros(1, np.int32), np.zeros(1), len(left))}
    n = B.dim_LLLRRRRL
    ele = np.zeros(max(m, len(right)), np.int32)
    like = np.random.default_rng([seed, 1]).standard_normal(n)
    return {"B": B, "hold": hold, "mats": mats, "ele": ele, "n": n, "like": like}


def _run_matrix_free(s):
    L = D.lib()
    vec, energy = np.zeros(s["n"]), np.zeros(1)
    dp = C.POINTER(C.c_double)
    box = D.DMRG_BOX_LAN()
    box.Eig_Vec, box.eig_val = vec.ctypes.data_as(dp), energy.ctypes.data_as(dp)
    box.acc, box.min_step, box.max_step, box.p_threads = 1e-14, 1, 800, 1
    box.Guess, box.Type = b"No", b"Normal"
    box.M_LLLR, box.M_LRRL, box.M_LRRL_Sign, box.M_RRRL = (s["mats"][k].ptr for k in ("LLLR", "LRRL", "sign", "RRRL"))
    box.Ele_RR = s["ele"].ctypes.data_as(C.POINTER(C.c_int))
    box.Dmrg_Basis = C.pointer(s["B"])
    L.DMRG_LANCZOS_SLOW_OBC(C.byref(box))
    return {"energy": float(energy[0]), "vec": _aligned(vec, s["like"])}


# ------------------------------------------------------------------ exact diagonalisation
def _ed_models(case, seed):
    """Chains of mixed lengths: XXZ at S^z = 0 up to l_max sites, Hubbard at half filling up to
    half as many."""
    shape = np.random.default_rng(case["count"] * 100 + case["l_max"])   # lengths: the case's
    coup = np.random.default_rng([seed, 6])                              # couplings: the seed's
    out = []
    for i in range(case["count"]):
        h = float(coup.uniform(0.05, 0.5))
        if i % 2 == 0:
            L = int(shape.choice(np.arange(8, case["l_max"] + 1, 2)))
            out.append(ed.Model("xxz", L=L, sz=0, J_z=float(coup.uniform(0.5, 1.5)), h_z=h))
        else:
            L = int(shape.choice(np.arange(4, case["l_max"] // 2 + 1, 2)))
            out.append(ed.Model("hubbard", L=L, N=L, sz=0, t=-1.0, U=float(coup.uniform(3.0, 5.0)), h_z=h))
    return out


def _ed_dim(m):
    return math.comb(m.L, m.L // 2) ** (2 if m.model == "hubbard" else 1)


def _prepare_ed(case, seed):
    models = _ed_models(case, seed)
    like = [np.random.default_rng([seed, 7, i]).standard_normal(_ed_dim(m)) for i, m in enumerate(models)]
    return {"models": models, "like": like}


def _run_ed(s):
    mats = []
    for m in s["models"]:
        P = ed.EdProblem.from_model(m)
        mats.append(P.assemble())
        P.free()
    res = engine.ground_state_batch(mats, engine.default_params(precision=s["precision"]))
    for A in mats:
        A.free()
    return {"energy": np.array([r[0] for r in res]),
            "vec": np.concatenate([_aligned(r[1], like) for r, like in zip(res, s["like"])])}


# --------------------------------------------------------------------------- entry points
_PREPARE = {"kron": _prepare_solve, "crs": _prepare_solve, "assemble": _prepare_assemble,
            "product": _prepare_product, "truncate": _prepare_truncate, "renormalise": _prepare_renormalise,
            "sector": _prepare_sector, "matrix_free": _prepare_matrix_free, "ed_batch": _prepare_ed}
_RUN = {"kron": _run_kron, "crs": _run_crs, "assemble": _run_assemble, "product": _run_product,
        "truncate": _run_truncate, "renormalise": _run_renormalise, "sector": _run_sector,
        "matrix_free": _run_matrix_free, "ed_batch": _run_ed}


def prepare(case, seed):
    os.environ["DMRGX_SML_OUT"] = "0"   # no step-count files
    s = _PREPARE[case["path"]](case, seed)
    s["path"], s["precision"] = case["path"], case.get("precision", 0)
    return s


def run(state):
    return _RUN[state["path"]](state)


def work(case):
    path = case["path"]
    if path == "ed_batch":
        models = _ed_models(case, 0)
        rows = sum(_ed_dim(m) for m in models)
        nnz = sum(_ed_dim(m) * (m.L / 2 if m.model == "xxz" else m.L) for m in models)
        # about 100 products of each matrix, vectors read and written once a product
        return {"bytes": 100.0 * 16 * rows + 12.0 * nnz + 8 * rows, "flops": 100.0 * 2 * nnz}
    q = _block(case["model"], case["m"])[3]
    dims = np.array(_dims(case), np.float64)
    n, dense = float(np.sum(dims[:, 0] * dims[:, 1])), float(np.sum(dims ** 2))
    flops = float(np.sum(2.0 * dims[:, 0] * dims[:, 1] * (dims[:, 0] + dims[:, 1])))
    # elements of the full CRS: the left and right Hamiltonians' rows on every state
    fill = {"xxz": 0.77, "hubbard": 0.78, "klm": 0.42}[case["model"]]
    nnz = fill * flops / 2.0
    if path == "kron":
        p = PRODUCTS[case["model"]]
        return {"bytes": 8.0 * dense + p * 16.0 * n, "flops": p * flops}
    if path == "crs":
        p = PRODUCTS[case["model"]]
        return {"bytes": 12.0 * nnz + p * (12.0 * nnz + 16.0 * n), "flops": p * 2.0 * nnz}
    if path == "assemble":
        return {"bytes": 24.0 * nnz + 16.0 * n, "flops": 2.0 * nnz}
    if path == "product":
        return {"bytes": 12.0 * nnz + 16.0 * n, "flops": 2.0 * nnz}
    if path == "truncate":
        d = dims[:, 0]
        return {"bytes": 8.0 * n + 16.0 * float(np.sum(d ** 2)),
                "flops": float(np.sum(d ** 2 * dims[:, 1] + 4.0 / 3.0 * d ** 3))}
    if path == "renormalise":
        d = dims[:, 0]
        share = case["m"] / float(np.sum(d))
        k = share * d
        return {"bytes": float(np.sum(12.0 * (d * d * 0.5 + 2 * d * k + k * k))),
                "flops": float(np.sum(d * d * k + 2.0 * d * k * k))}
    if path == "sector":
        n_out = float(sum(len(x) * len(y) for _, _, x, y in _sectors(q, _raised(q))))
        per_row = float(np.count_nonzero(_raising(q, 0))) / case["m"]
        return {"bytes": 8.0 * (n + n_out) + 12.0 * per_row * case["m"], "flops": 2.0 * per_row * n_out}
    return {"bytes": 8.0 * dense + 100 * 16.0 * n, "flops": 100 * flops}   # matrix_free


def tolerance(case):
    """Measured against the 64-bit results (`exact`), about four times the largest seen."""
    path = case["path"]
    if path in ("kron", "crs", "ed_batch"):   # a residual below 1e-9 over the gap
        return {"rel": 2e-9, "max": 1e-7}
    if path == "matrix_free":   # Lanczos alone: the vector's error is the root of the energy's
        return {"rel": 2e-6, "max": 4e-5}
    if path in ("assemble", "product"):
        return {"rel": 3e-15, "max": 2e-14}
    if path == "truncate":   # the weights' order and the states' gaps: 1e-13 of the weights
        return {"rel": 1e-10, "max": 1e-8}
    if path == "renormalise":
        return {"rel": 2e-15, "max": 4e-14}
    return {"rel": 2e-15, "max": 1e-14}   # sector


# ----------------------------------------------------------------------- 64-bit results
def _signs(eles, t, ids, block, site):
    """(-1)^p of a term's sign rule on the states (block, site); ids: which parity arrays are
    read at the block's and at the site's state."""
    p = np.zeros(len(block), np.int64)
    for name, at in ids:
        p += eles[int(t[name])][block if at == "block" else site]
    return 1.0 - 2.0 * (p % 2)


def _constant(t):
    return float(t["coeff"]) * (-1.0 if int(t["sign_mode"]) == 1 else 1.0)


def _half_dense(snap, q, side, device):
    """Dense Hamiltonian of one half (block, site), block-major."""
    block, site, _, _ = _halves(q, side)
    d, m = snap.dim_onsite, snap.dim_LL
    kinds = {"LL": ("LL", "LR", "LLLR"), "RR": ("RR", "RL", "RRRL")}[side]
    h = torch.zeros(m * d, m * d, dtype=torch.float64, device=device)
    for t in snap.terms:
        k = snapshot.KIND_NAMES[int(t["kind"])]
        if k not in kinds or t["coeff"] == 0.0:
            continue
        a = torch.from_numpy(snap.ops[int(t["op1"])].to_dense()).to(device)
        if k == kinds[0]:
            h += t["coeff"] * torch.kron(a, torch.eye(d, dtype=torch.float64, device=device))
        elif k == kinds[1]:
            h += t["coeff"] * torch.kron(torch.eye(m, dtype=torch.float64, device=device), a)
        else:
            b = torch.from_numpy(snap.ops[int(t["op2"])].to_dense()).to(device)
            ab = torch.kron(a, b)
            if int(t["sign_mode"]):
                ab *= torch.from_numpy(_signs(snap.eles, t, [("ele0", "block")], block, site)).to(device)[:, None]
            h += _constant(t) * ab
    return h


def _middle_dense(snap):
    """The coupling of the two middle sites (no fermion signs)."""
    d = snap.dim_onsite
    h = np.zeros((d * d, d * d))
    for t in snap.terms:
        if snapshot.KIND_NAMES[int(t["kind"])] == "LRRL" and t["coeff"] != 0.0:
            h += t["coeff"] * np.kron(snap.ops[int(t["op1"])].to_dense(), snap.ops[int(t["op2"])].to_dense())
    return h


def _exact_operator(case, seed):
    """x -> H x on the GPU in 64 bits: dense halves per sector, the middle coupling by index."""
    snap, q = _superblock(case, seed)
    d, m = snap.dim_onsite, snap.dim_LL
    dev = "cuda"
    hl, hr = _half_dense(snap, q, "LL", dev), _half_dense(snap, q, "RR", dev)
    blocks, at = [], 0
    for _, _, x, y in _sectors(q):
        ix, iy = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)
        blocks.append((at, len(x), len(y), hl[ix][:, ix].contiguous(), hr[iy][:, iy].contiguous()))
        at += len(x) * len(y)
    n = at
    basis = [torch.from_numpy(a.astype(np.int64)).to(dev) for a in _basis_arrays(q)]
    dims = (m, d, m, d)
    inv = torch.full((int(np.prod(dims)),), -1, dtype=torch.int64, device=dev)
    code = ((basis[0] * d + basis[1]) * m + basis[2]) * d + basis[3]
    inv[code] = torch.arange(n, device=dev)
    hops = []
    for t in snap.terms:
        if snapshot.KIND_NAMES[int(t["kind"])] != "LRRL" or t["coeff"] == 0.0:
            continue
        a, b = (snap.ops[int(t[k])].to_dense() for k in ("op1", "op2"))
        sign = None
        if int(t["sign_mode"]):
            e0, e1 = (torch.from_numpy(snap.eles[int(t[k])].astype(np.int64)).to(dev) for k in ("ele0", "ele1"))
            sign = 1.0 - 2.0 * ((e0[basis[2]] + e1[basis[1]]) % 2).double()
        for i, i2 in np.argwhere(a):
            for j, j2 in np.argwhere(b):
                rows = torch.nonzero((basis[1] == int(i)) & (basis[3] == int(j))).ravel()
                cols = inv[((basis[0][rows] * d + int(i2)) * m + basis[2][rows]) * d + int(j2)]
                ok = cols >= 0
                rows, cols = rows[ok], cols[ok]
                v = torch.full((len(rows),), _constant(t) * a[i, i2] * b[j, j2], dtype=torch.float64, device=dev)
                if len(rows):
                    hops.append((rows, cols, v * sign[rows] if sign is not None else v))

    def apply(x):
        y = torch.empty_like(x)
        for off, da, db, ml, mr in blocks:
            X = x[off:off + da * db].view(da, db)
            y[off:off + da * db].view(da, db).copy_(ml @ X + X @ mr.T.contiguous())
        for rows, cols, v in hops:
            y[rows] += v * x[cols]
        return y

    return n, apply


def _lowest(n, apply, dev, gen_seed=12345):
    """Lowest eigenpair by Lanczos with full reorthogonalisation, to a residual of 1e-12."""
    if n == 1:
        one = torch.ones(1, dtype=torch.float64, device=dev)
        return float(apply(one)[0]), one
    g = torch.Generator(device=dev)
    g.manual_seed(gen_seed)
    v = torch.randn(n, dtype=torch.float64, device=dev, generator=g)
    cap = min(n, 900)
    V = torch.empty(cap, n, dtype=torch.float64, device=dev)
    al, be = [], []
    v /= v.norm()
    for k in range(cap):
        V[k] = v
        w = apply(v)
        al.append(float(w @ v))
        for _ in range(2):
            w -= V[:k + 1].T @ (V[:k + 1] @ w)
        b = float(w.norm())
        last = k == cap - 1 or b < 1e-13 * max(1.0, abs(al[0]))
        if last or k % 20 == 19:
            T = np.diag(al) + np.diag(be, 1) + np.diag(be, -1)
            lam, s = np.linalg.eigh(T)
            if last or abs(b * s[-1, 0]) < 1e-12 * max(1.0, abs(lam[0])):
                x = V[:k + 1].T @ torch.from_numpy(s[:, 0].copy()).to(dev)
                return float(lam[0]), x / x.norm()
        be.append(b)
        v = w / b


def _exact_solve(case, seed):
    n, apply = _exact_operator(case, seed)
    energy, v = _lowest(n, apply, "cuda")
    like = np.random.default_rng([seed, 1]).standard_normal(n)
    return {"energy": energy, "vec": _aligned(v.cpu().numpy(), like)}


def _exact_product(case, seed):
    n, apply = _exact_operator(case, seed)
    return apply(torch.from_numpy(np.random.default_rng([seed, 1]).standard_normal(n)).cuda())


def _exact_truncate(case, seed):
    q = _block(case["model"], case["m"])[3]
    v = torch.from_numpy(_schmidt_state(q, seed)).cuda()
    states, at, row0 = [], 0, 0
    for e, s, left, right in _sectors(q):
        psi = v[at:at + len(left) * len(right)].view(len(left), len(right))
        u, sv, _ = torch.linalg.svd(psi, full_matrices=True)
        w = torch.zeros(len(left), dtype=torch.float64, device=v.device)
        w[:len(sv)] = sv * sv
        u, w = u.abs().T.cpu().numpy(), w.cpu().numpy()
        states += [(w[i], e, s, row0, u[i]) for i in range(len(left))]
        at += len(left) * len(right)
        row0 += len(left)
    states.sort(key=lambda t: -t[0])
    if len(states) <= case["m"]:
        kept = sum(1 for t in states if t[0] > 1e-15)
    else:
        kept = next(i for i in range(case["m"], 0, -1)
                    if abs(states[i - 1][0] - states[i][0]) > 1e-15 and states[i - 1][0] > 1e-15)
    keep = sorted(sorted(states[:kept], key=lambda t: t[2]), key=lambda t: t[1])
    return {"weights": np.array([t[0] for t in states]), "discarded": float(sum(t[0] for t in reversed(states[kept:]))), "kept": kept,
            "q1": np.array([t[1] for t in keep], np.int32), "q2": np.array([t[2] for t in keep], np.int32),
            "col": np.cumsum([0] + [len(t[4]) for t in keep]),
            "row": np.concatenate([t[3] + np.arange(len(t[4])) for t in keep]).astype(np.int32),
            "val": np.concatenate([t[4] for t in keep])}


def _exact_renormalise(case, seed):
    s = _prepare_renormalise(case, seed)
    T, h = (torch.from_numpy(s[k]).cuda() for k in ("T", "h"))
    r = (T.T.contiguous() @ (h @ T)).cpu().numpy()
    r[np.abs(r) <= 1e-15] = 0.0
    i, j = np.nonzero(r)
    row = np.zeros(r.shape[0] + 1, np.int64)
    np.add.at(row, i + 1, 1)
    return {"row": np.cumsum(row), "col": j.astype(np.int32), "val": r[i, j]}


def _exact_sector(case, seed):
    q = _block(case["model"], case["m"])[3]
    d, m = len(q["sz_site"]), case["m"]
    x = np.random.default_rng([seed, 5]).standard_normal(len(_basis_arrays(q)[0]))
    flat = {k: torch.from_numpy(np.ravel_multi_index([a.astype(np.int64) for a in _basis_arrays(q, t)],
                                                     (m, d, m, d))).cuda()
            for k, t in (("in", None), ("out", _raised(q)))}
    psi = torch.zeros(m * d * m * d, dtype=torch.float64, device="cuda")
    psi[flat["in"]] = torch.from_numpy(x / np.linalg.norm(x)).cuda()
    out = torch.from_numpy(_raising(q, seed)).cuda() @ psi.view(m, d * m * d)
    return out.reshape(-1)[flat["out"]].cpu().numpy()


def _ed_exact_one(m):
    """Ground state of one chain from its bond terms, codes ascending, site 0 the lowest digit."""
    d = 2 if m.model == "xxz" else 4
    codes = np.arange(d ** m.L, dtype=np.int64)
    digit = [(codes // d ** i) % d for i in range(m.L)]
    ele, sz = np.array([0, 1, 1, 2]), np.array([0, 1, -1, 0])
    if d == 2:
        ok = sum(digit) * 2 == m.L
    else:
        ok = (sum(ele[x] for x in digit) == m.N) & (sum(sz[x] for x in digit) == m.sz)
    codes = codes[ok]
    digit = [x[ok] for x in digit]
    n = len(codes)
    diag = np.zeros(n)
    if d == 2:
        z = [0.5 - x for x in digit]
        for i in range(m.L):
            diag += m.h_z * z[i]
        pairs = [(np.array([[0, 1.0], [0, 0]]), np.array([[0, 0], [1.0, 0]]), 0.5 * m.J_xy, False)]
        for i in range(m.L - 1):
            diag += m.J_z * z[i] * z[i + 1]
    else:
        for i in range(m.L):
            diag += m.h_z * 0.5 * sz[digit[i]] + m.U * (digit[i] == 3)
        up, dn = np.zeros((4, 4)), np.zeros((4, 4))   # annihilation, both = c+_up c+_down |0>
        up[0, 1] = up[2, 3] = 1.0
        dn[0, 2], dn[1, 3] = 1.0, -1.0
        pairs = [(up.T, up, m.t, True), (dn.T, dn, m.t, True)]
    cols, vals = [], []
    for i in range(m.L - 1):
        for a, b, c, fermi in pairs:
            for (p, r), swap in (((a, b), 1.0), ((b, a), -1.0 if fermi else 1.0)):
                # operators with at most one element a row
                pc, rc = np.abs(p).argmax(1), np.abs(r).argmax(1)
                pv, rv = p[np.arange(d), pc], r[np.arange(d), rc]
                x, y = digit[i], digit[i + 1]
                v = c * pv[x] * rv[y]
                if fermi:
                    v = v * swap * np.where(ele[x] % 2 == 1, 1.0, -1.0)
                target = codes + (pc[x] - x) * d ** i + (rc[y] - y) * d ** (i + 1)
                at = np.searchsorted(codes, target).clip(0, n - 1)
                v = np.where(codes[at] == target, v, 0.0)
                cols.append(np.where(v != 0.0, at, 0))
                vals.append(v)
    cols, vals, diag = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (np.array(cols), np.array(vals), diag))

    def apply(x):
        return diag * x + (vals * x[cols]).sum(0)

    return _lowest(n, apply, "cuda")


def _exact_ed(case, seed):
    models = _ed_models(case, seed)
    res = [_ed_exact_one(m) for m in models]
    return {"energy": np.array([r[0] for r in res]),
            "vec": np.concatenate([_aligned(v.cpu().numpy(), np.random.default_rng([seed, 7, i]).standard_normal(len(v)))
                                   for i, (_, v) in enumerate(res)])}


_EXACT = {"kron": _exact_solve, "crs": _exact_solve, "matrix_free": _exact_solve, "assemble": _exact_product,
          "product": _exact_product, "truncate": _exact_truncate, "renormalise": _exact_renormalise,
          "sector": _exact_sector, "ed_batch": _exact_ed}


def exact(case, seed):
    return _EXACT[case["path"]](case, seed)
