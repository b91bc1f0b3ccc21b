"""Kronecker form of the superblock Hamiltonian (dmrgx_superblock_kron): per sector of the
superblock basis, the LL/LR/LLLR terms as a dense matrix on the rows of the sector's block of
the vector and the RR/RL/RRRL terms as one on its columns, the coupling terms row by row.

The operator is the one GET_HAM_LLLRRRRL assembles (main/dmrg/<model>_vf/src/allocations/
GET_HAM_LLLRRRRL.c:11-114), so its product must equal the product with the reference's own
CRS (expanded to full) to rounding, on every golden superblock of the three models, and its
ground state must be the reference's within the FP64 bounds."""
import os

import numpy as np
import pytest

from conftest import GOLDEN, golden_ids, golden_snapshots

SNAPS = golden_snapshots()
BIG = [os.path.join(GOLDEN, f) for f in ("hubbard_L64_m400_s31.npz", "xxz_L64_m300_s31.npz")]


def _ref_full(s):
    import scipy.sparse as sp
    L = sp.csr_matrix((s.ham.val, s.ham.col, s.ham.row), shape=(s.n, s.n))
    return (L + L.T - sp.diags(L.diagonal())).tocsr()


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [0, 1, 2], ids=["16x16", "by-size", "32x32"])
@pytest.mark.parametrize("path", SNAPS + BIG, ids=golden_ids(SNAPS + BIG))
def test_gpu_kron_product_equals_reference_crs(path, variant):
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(path)
    sb = D.Superblock(s)
    K = sb.kron()
    K.set_kernel(variant)
    try:
        x = np.random.default_rng(11).standard_normal(s.n)
        y = K.matvec(x)
        if s.ham is not None:
            y_ref = _ref_full(s) @ x
        else:   # no dumped CRS: the device assembly (bit-exact with the reference's)
            A = sb.assemble()
            y_ref = A.matvec(x)
            A.free()
        scale = np.abs(y_ref).max()
        assert np.abs(y - y_ref).max() <= 1e-12 * scale, np.abs(y - y_ref).max() / scale
    finally:
        K.free()
        sb.free()


@pytest.mark.gpu
@pytest.mark.parametrize("path", SNAPS + BIG[:1], ids=golden_ids(SNAPS + BIG[:1]))
def test_gpu_kron_ground_state(path):
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(path)
    sb = D.Superblock(s)
    K = sb.kron()
    try:
        E, vec, st = K.ground_state()
    finally:
        K.free()
        sb.free()
    e_ref = float(s.meta["gs_energy"][0])
    assert abs(E - e_ref) <= 1e-10 * max(1.0, abs(e_ref)), (E, e_ref)
    assert st.gs_error < 1e-9
    if "gs_vec" in s.meta:
        ref = s.meta["gs_vec"]
        assert np.abs(vec - np.sign(vec @ ref) * ref).max() <= 1e-8


@pytest.mark.gpu
def test_gpu_kron_autotune_and_bad_variant():
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(BIG[0])
    sb = D.Superblock(s)
    K = sb.kron()
    try:
        v, us = K.autotune()
        assert 0 <= v < K.VARIANTS and us > 0
        for bad in (-1, K.VARIANTS):
            with pytest.raises(D.DmrgxError):
                K.set_kernel(bad)
        E, _, _ = K.ground_state()
        e_ref = float(s.meta["gs_energy"][0])
        assert abs(E - e_ref) <= 1e-10 * abs(e_ref)
    finally:
        K.free()
        sb.free()


@pytest.mark.gpu
def test_gpu_kron_kernel_numbers():
    """3 to 15 are accepted and give the default kernel's bits."""
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(SNAPS[-1])
    sb = D.Superblock(s)
    K = sb.kron()
    try:
        x = np.random.default_rng(11).standard_normal(s.n)
        y = K.matvec(x)
        for variant in range(3, K.VARIANTS):
            K.set_kernel(variant)
            assert np.array_equal(K.matvec(x), y), variant
    finally:
        K.free()
        sb.free()


@pytest.mark.gpu
def test_gpu_kron_rejects_fp32():
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(SNAPS[-1])
    sb = D.Superblock(s)
    K = sb.kron()
    try:
        with pytest.raises(D.DmrgxError):
            K.ground_state(precision=1)
    finally:
        K.free()
        sb.free()


@pytest.mark.gpu
@pytest.mark.parametrize("path", SNAPS[-3:] + BIG[:1], ids=golden_ids(SNAPS[-3:] + BIG[:1]))
def test_gpu_residual_stop(path):
    """lan_type 2 ("Residual", no reference counterpart): Lanczos until the Ritz pair's residual
    bound is below ii_acc / (2 sqrt(n)); the reference's L1 residual test then decides.  The
    energy within the FP64 bound of the reference's, on the Kronecker form and the CRS."""
    import dmrg_c_amd as D
    from dmrg_c_amd import snapshot
    s = snapshot.load(path)
    e_ref = float(s.meta["gs_energy"][0])
    sb = D.Superblock(s)
    K = sb.kron()
    A = sb.assemble()
    try:
        for solver in (K, A):
            E, vec, st = solver.ground_state(lan_type=2)
            assert abs(E - e_ref) <= 1e-10 * max(1.0, abs(e_ref)), (E, e_ref)
            assert st.gs_error < 1e-9
            _, _, st0 = solver.ground_state()
            assert st.spmv_calls <= st0.spmv_calls + 2
        with pytest.raises(D.DmrgxError):
            A.ground_state(lan_type=3)
    finally:
        K.free()
        A.free()
        sb.free()


def _random_superblock(left, right, middle, seed, far=False):
    """A spin-1/2 superblock with left[i] / right[i] block states of 2 S^z = left0 + 2 i, random
    block operators of the right selection rules, and the terms of an XXZ chain; with far also
    couplings of block to block and of block to site, whose operators take a state to many."""
    from dmrg_c_amd import snapshot as S
    rng = np.random.default_rng(seed)
    qa = np.repeat(np.arange(len(left)), left) * 2 - (len(left) - 1)
    qb = np.repeat(np.arange(len(right)), right) * 2 - (len(right) - 1)
    site = np.array([1, -1])

    def op(q, dq, sym=False):
        a = np.where(q[:, None] == q[None, :] + dq, rng.uniform(-1, 1, (len(q), len(q))), 0.0)
        return a + a.T if sym else a

    def crs(a):
        r, c = np.nonzero(a)
        row = np.zeros(len(a) + 1, np.int64)
        np.add.at(row, r + 1, 1)
        return S.Crs(len(a), len(a), np.cumsum(row), c.astype(np.int32), a[r, c])
    sp = np.array([[0.0, 1.0], [0.0, 0.0]])
    sz = np.diag([0.5, -0.5])
    pa, pb = op(qa, 2), op(qb, 2)
    mats = [op(qa, 0, True), op(qb, 0, True), sz, sp, sp.T, pa, pa.T, pb, pb.T]
    rows = [("LL", 0, -1, 1.0), ("RR", 1, -1, 0.7), ("LR", 2, -1, 0.3), ("RL", 2, -1, -0.2),
            ("LLLR", 5, 4, 0.5), ("LLLR", 6, 3, 0.5), ("RRRL", 7, 4, 0.4), ("RRRL", 8, 3, 0.4)]
    if middle:
        rows += [("LRRL", 3, 4, 0.5), ("LRRL", 4, 3, 0.5), ("LRRL", 2, 2, 1.1)]
    if far:
        rows += [("LLRR", 5, 8, 0.25), ("LLRR", 6, 7, 0.25), ("LLRL", 5, 4, 0.1), ("LLRL", 6, 3, 0.1),
                 ("LRRR", 3, 8, 0.2), ("LRRR", 4, 7, 0.2)]
    rows += [("ZERO", -1, -1, 0.0)]
    terms = np.zeros(len(rows), S.TERM_DTYPE)
    for t, (kind, o1, o2, c) in zip(terms, rows):
        t["kind"], t["op1"], t["op2"], t["coeff"] = S.KIND_NAMES.index(kind), o1, o2, c
        t["ele0"] = t["ele1"] = t["ele2"] = -1
    sa, sb = (qa[:, None] + site).ravel(), (qb[:, None] + site).ravel()
    states = [(x, y) for s in np.unique(sa) for x in np.nonzero(sa == s)[0] for y in np.nonzero(sb == -s)[0]]
    x, y = np.array(states).T
    basis = [np.ascontiguousarray(v, np.int16) for v in (x // 2, x % 2, y // 2, y % 2)]
    return S.Snapshot(len(x), len(qa), len(qb), 2, 0, 0, 0, *basis, [crs(m) for m in mats], [], terms)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [0, 1, 2], ids=["16x16", "by-size", "32x32"])
@pytest.mark.parametrize("left,right,far", [([1], [1], False), ([1, 1], [1, 1], False), ([1, 14, 2], [2, 13, 1], False),
                                            ([8, 9, 8], [7, 9, 8], True), ([1, 15, 16, 17], [33, 1, 15, 30], False),
                                            ([10, 34, 5], [3, 36, 17], True)],
                         ids=["1", "2", "edge16", "far17", "edge32", "far"])
def test_gpu_kron_tile_edges(left, right, far, variant):
    """Sectors of one state, of one below, at and one above 16 and 32 states on either side (the
    shifted last slab, partly filled tiles), and couplings in their general form, against the
    product with the oracle's CRS."""
    import dmrg_c_amd as D
    import oracle_py as O
    import scipy.sparse as sp
    s = _random_superblock(left, right, True, 7, far)
    row, col, val = O.assemble(s)
    A = sp.csr_matrix((val, col, row), shape=(s.n, s.n))
    A = (A + A.T - sp.diags(A.diagonal())).tocsr()
    sb = D.Superblock(s)
    K = sb.kron()
    K.set_kernel(variant)
    try:
        x = np.random.default_rng(3).standard_normal(s.n)
        y, y_ref = K.matvec(x), A @ x
        # each element sums at most a few hundred products of numbers below 2
        assert np.abs(y - y_ref).max() <= 1e-13 * np.abs(x).max() * abs(A).sum(axis=1).max()
        if s.n < 3000:
            E, _, _ = K.ground_state()
            w = np.linalg.eigvalsh(A.toarray())
            assert abs(E - w[0]) <= 1e-10 * max(1.0, abs(w[0]))
    finally:
        K.free()
        sb.free()



@pytest.mark.gpu
def test_gpu_kron_repeated_operator_columns():
    """Operators whose rows hold columns out of order and twice (both entries count, as the element
    makers add them): the sector matrices' general build."""
    import dmrg_c_amd as D
    import oracle_py as O
    import scipy.sparse as sp
    from dmrg_c_amd import snapshot as S
    s = _random_superblock([3, 12, 5], [2, 14, 3], True, 9)
    for k in (0, 5, 6):
        o = s.ops[k]
        rows = [list(zip(o.col[a:b], o.val[a:b])) for a, b in zip(o.row[:-1], o.row[1:])]
        rows = [[(c, 0.25 * v) for c, v in r] + [(c, 0.75 * v) for c, v in reversed(r)] for r in rows]
        flat = [e for r in rows for e in r]
        s.ops[k] = S.Crs(o.row_dim, o.col_dim, np.cumsum([0] + [len(r) for r in rows]).astype(np.int64),
                         np.array([c for c, _ in flat], np.int32), np.array([v for _, v in flat]))
    row, col, val = O.assemble(s)
    A = sp.csr_matrix((val, col, row), shape=(s.n, s.n))
    A = (A + A.T - sp.diags(A.diagonal())).tocsr()
    sb = D.Superblock(s)
    K = sb.kron()
    try:
        x = np.random.default_rng(3).standard_normal(s.n)
        y = K.matvec(x)
        assert np.abs(y - A @ x).max() <= 1e-13 * np.abs(x).max() * abs(A).sum(axis=1).max()
    finally:
        K.free()
        sb.free()
