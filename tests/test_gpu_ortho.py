"""orthoQS (block SVD truncation) on the device vs the CPU oracle (GPU tests).

Bar: the structure of both results (label records, block order, dims,
itags), the kept count, Ntot and flag bit-exact; singular values, svd2tr,
sv2tot and sfac within 1e-12 (relative to the largest singular value /
themselves); singular vectors up to the sign of each column (the SVD's own
gauge), within 1e-9, and gauge-free: A1 . A2 equals the oracle's product
within 1e-12, A1 is an isometry within 1e-12.
"""
import numpy as np
import pytest

import oracle as O
import qspace_amd as Q
from qspace_amd import gen
from helpers import assert_same_structure, oracle_ortho
from test_oracle_blockops import u1_rank4

pytestmark = pytest.mark.gpu


def _tensor(kind):
    if kind == "psi":
        return gen.u1_two_site_psi(seed=3, Lq=(-4, -2, 0, 2, 4), Rq=(-4, -2, 0, 2, 4), dmin=2, dmax=7)
    if kind == "rank4":
        return u1_rank4(5, nq=2, dmin=1, dmax=5)
    if kind == "mps":
        return gen.u1_mps(seed=9, Lq=(-4, -2, 0, 2, 4), Rq=(-3, -1, 1, 3), dmin=2, dmax=6)
    if kind == "psi_full":  # every group matrix in LDS (dims up to 2 x 32)
        return gen.u1_two_site_psi(seed=1007)
    if kind == "psi_wide":  # group matrices beyond the LDS capacity
        return gen.u1_two_site_psi(seed=1008, Lq=(-4, -2, 0, 2, 4), Rq=(-4, -2, 0, 2, 4), dmin=60, dmax=110)
    raise KeyError(kind)


def _group_mats(T):
    """per new-leg label: the blocks of T stacked along their fused leading
    legs (T's last leg is the new one) -> {label: matrix}"""
    out = {}
    dims = T.dims()
    for i, d in enumerate(T.data):
        key = tuple(T.Q[T.rank - 1][i])
        out.setdefault(key, []).append(np.asarray(d).reshape(-1, int(dims[i, -1]), order="F"))
    return {k: np.vstack(v) for k, v in out.items()}


def _check(P, K, **kw):
    A1, A2, info = Q.orthoQS(P, K, **kw)
    R1, R2, rinfo = oracle_ortho(P, K, **kw)
    print(f"orthoQS K={K} {kw} blocks={P.nblk} groups={info['ngroups']} sweeps={info['sweeps']} "
          f"keep={info['Nkeep']}/{info['Ntot']}", flush=True)
    assert_same_structure(A1, R1)
    assert_same_structure(A2, R2)
    for k in ("Nkeep", "Ntot", "flag"):
        assert info[k] == rinfo[k], k
    smax = float(rinfo["svd"][0])
    assert np.abs(info["svd"] - rinfo["svd"]).max() <= 1e-12 * smax
    for k in ("sfac", "sv2tot"):
        assert info[k] == pytest.approx(rinfo[k], rel=1e-12), k
    assert info["svd2tr"] == pytest.approx(rinfo["svd2tr"], rel=1e-9, abs=1e-15)
    # singular vectors up to a sign per column
    U, UR = _group_mats(A1), _group_mats(R1)
    V, VR = _group_mats(A2), _group_mats(R2)
    for key in UR:
        sgn = np.sign(np.sum(U[key] * UR[key], axis=0))
        assert np.all(sgn != 0)
        assert np.abs(U[key] * sgn - UR[key]).max() < 1e-9
        if key in VR:
            assert np.abs(V[key] * sgn - VR[key]).max() < 1e-9 * smax
    # gauge-free: the product and the isometry
    if A1.nblk and A2.nblk:
        X = O.contract(A1, [K], A2, [P.rank - K])
        XR = O.contract(R1, [K], R2, [P.rank - K])
        assert_same_structure(X, XR)
        num = sum(float(np.sum((a - b) ** 2)) for a, b in zip(X.data, XR.data))
        den = sum(float(np.sum(b * b)) for b in XR.data)
        assert np.sqrt(num / den) < 1e-12
        G = O.contract(A1, list(range(K)), A1, list(range(K)), conjA=1)
        for d in G.data:
            assert np.abs(d - np.eye(d.shape[0])).max() < 1e-12
    return A1, A2, info


CASES = [("psi", 2, {}), ("psi", 1, {}), ("psi", 2, {"Nkeep": 9}), ("psi", 2, {"Nkeep": 100, "stol": 0.5}),
         ("psi", 2, {"Nkeep": 100, "stol": 0.5, "Nkmin": 14, "itag": "X"}), ("rank4", 2, {"Nkeep": 12}),
         ("rank4", 1, {}), ("mps", 2, {"Nkeep": 10}), ("mps", 1, {"stol": 0.3})]


@pytest.mark.parametrize("kind,K,kw", CASES)
def test_ortho_matches_oracle(gpu, kind, K, kw):
    _check(_tensor(kind), K, **kw)


@pytest.mark.parametrize("kind", ["psi_full", "psi_wide"])
def test_ortho_full_size(gpu, kind):
    """the two-site psi at full size (LDS path) and with group matrices
    beyond the LDS (the in-place path): parity, and A1 . A2 = PSI when all
    states are kept"""
    P = _tensor(kind)
    _check(P, 2, Nkeep=400)
    A1, A2, info = Q.orthoQS(P, 2)
    assert info["Nkeep"] == info["Ntot"] and info["sfac"] == 1.0
    X = O.contract(A1, [2], A2, [2])
    got = {tuple(X.QIDX[i]): d for i, d in enumerate(X.data)}
    assert sorted(got) == sorted(tuple(r) for r in P.QIDX)
    num = sum(float(np.sum((got[tuple(P.QIDX[i])] - d) ** 2)) for i, d in enumerate(P.data))
    den = sum(float(np.sum(d * d)) for d in P.data)
    assert np.sqrt(num / den) < 1e-12


def test_ortho_unsupported_flip(gpu):
    M = gen.u1_mps(seed=2, Lq=(-2, 0, 2), Rq=(-1, 1), dmin=2, dmax=3)
    M2 = Q.QSpace(M.Q, M.data, "A", ["L", "s", "R"])
    with pytest.raises(Q.QsxError) as e:
        Q.orthoQS(M2, 2)
    assert e.value.code == 5


def test_ortho_edge_cases(gpu):
    """nothing kept (Nkeep = 0; stol above every value), a group with a zero
    block, a rank-2 block-diagonal psi (K = 1 = r-1)"""
    from test_oracle_ortho import u1_rank2
    P = _tensor("psi")
    for kw in ({"Nkeep": 0}, {"Nkeep": 50, "stol": 1e3}):
        A1, A2, info = _check(P, 2, **kw)
        assert A1.nblk == 0 and A2.nblk == 0 and info["Nkeep"] == 0
    Z = gen.u1_two_site_psi(seed=5, Lq=(-4, -2, 0, 2, 4), Rq=(-4, -2, 0, 2, 4), dmin=2, dmax=7)
    Z = Q.QSpace(Z.Q, [np.zeros_like(d) if i == 3 else d for i, d in enumerate(Z.data)], Z.qtype, Z.itags)
    _check(Z, 2, Nkeep=20)
    _check(u1_rank2(), 1, Nkeep=5)
    _check(u1_rank2(seed=6, qs=(-4, -2, 0, 2, 4), dmin=20, dmax=150), 1, Nkeep=200, stol=1e-3)


def test_ortho_rank_deficient_groups(gpu):
    """group matrices of exactly deficient rank (every block of a two-site
    psi a product of thin factors, several blocks per group): the zero
    singular values come out at rounding level, the sweeps end (a column of
    rounding noise is not rotated against a larger one), and the truncated
    and the full products agree with the oracle"""
    rng = np.random.RandomState(17)
    P = gen.u1_two_site_psi(seed=6, Lq=(-4, -2, 0, 2, 4), Rq=(-4, -2, 0, 2, 4), dmin=3, dmax=7)
    data = []
    for d in P.data:
        s = d.shape
        L = rng.standard_normal((s[0] * s[1], 2))
        R = rng.standard_normal((2, s[2] * s[3]))
        data.append(np.asfortranarray((L @ R).reshape(s, order="F")))
    D = Q.QSpace(P.Q, data, P.qtype, P.itags)
    for kw in ({}, {"Nkeep": 6}):
        A1, A2, info = Q.orthoQS(D, 2, **kw)
        R1, R2, rinfo = oracle_ortho(D, 2, **kw)
        assert (info["Nkeep"], info["Ntot"]) == (rinfo["Nkeep"], rinfo["Ntot"])
        sv, rsv = np.asarray(info["svd"]), np.asarray(rinfo["svd"])
        assert np.abs(sv - rsv).max() <= 1e-12 * rsv.max()
        assert (rsv < 1e-13 * rsv.max()).sum() > 0  # the draw is rank-deficient
        X = O.contract(A1, [2], A2, [2], skip_zero=0)
        XR = O.contract(R1, [2], R2, [2], skip_zero=0)
        assert_same_structure(X, XR)
        num = sum(float(np.sum((a - b) ** 2)) for a, b in zip(X.data, XR.data))
        den = sum(float(np.sum(b * b)) for b in XR.data)
        assert np.sqrt(num / den) < 1e-12


# group matrices (rows, columns) at the edges of the SVD's paths: panels of 16
# columns, the in-LDS / column-block line (n = 96 / 97), register rows of the
# cross rounds (multiples of 32), row buckets of the QR (256, 512, 1024 rows),
# the line beyond which the matrix itself is swept (n = 257, m = 1025) and, of
# those, the ones in one workgroup's LDS (m n + n^2 <= 20224, among them the
# single columns that no pair of column blocks has room for) and the first
# beyond it; small ones are swept as they are too (n <= 6, or n <= 24 and
# m n <= 5120)
SHAPES = [(1, 1), (2, 2), (5, 2), (16, 16), (17, 16), (40, 17), (33, 32), (96, 96), (97, 97), (130, 96), (128, 97),
          (129, 128), (140, 129), (256, 193), (257, 225), (256, 256), (513, 60), (600, 100), (1024, 33), (1025, 20),
          (258, 257), (512, 257), (513, 258), (300, 1), (24, 24), (25, 25), (1024, 6), (1024, 7), (640, 8), (641, 8), (213, 24), (214, 24), (2000, 8), (2520, 8), (2521, 8), (1045, 19), (1046, 19), (10111, 1), (12000, 1), (20223, 1)]


@pytest.mark.parametrize("kind", ["random", "graded", "deficient", "scaled"])
@pytest.mark.parametrize("wide", [False, True])
def test_svd_shapes(gpu, kind, wide):
    """singular values, A1 . A2 = psi and the isometry of A1 over the shapes
    where the decomposition changes path; graded: values over six decades,
    deficient: half the columns repeated and one zero, scaled: entries near
    2^+-400.  Tolerance: an element takes about n rotations a sweep, over at
    most 10 sweeps of a preconditioned matrix and 60 (the limit) of one swept
    as it is, each rounding at 2 eps of its row: a random walk of
    2 sqrt(sweeps (m + n)) eps, times 4.  Deficient matrices beyond the QRs:
    test_svd_deficient_beyond_qr."""
    rng = np.random.default_rng(23 + wide)
    for k, (m, n) in enumerate(SHAPES):
        if kind == "deficient" and n > 256:
            continue
        if kind == "graded":
            M = (rng.standard_normal((m, n)) / np.sqrt(m) * np.exp(-14.0 * np.arange(n) / n)) @ \
                (rng.standard_normal((n, n)) / np.sqrt(n))
        elif kind == "deficient":
            M = _deficient(rng, m, n)
        else:
            M = rng.standard_normal((m, n))
        if kind == "scaled":
            M = np.ldexp(M, 400 if k % 2 else -400)
        if wide:
            M = M.T
        P = Q.QSpace([np.array([[0]]), np.array([[0]])], [M], "A", ["L", "R*"])
        print(kind, M.shape, flush=True)
        A1, A2, info = Q.orthoQS(P, 1, stol=0.0)
        _check_group(M, A1, A2, 0, info["svd"])


def _deficient(rng, m, n):
    M = rng.standard_normal((m, n))
    M[:, n // 2:] = M[:, :n - n // 2]
    M[:, -1] = 0.0
    return M


def _check_group(M, A1, A2, i, svd):
    """block i of A1 and A2 against its matrix: the product, the isometry over
    the columns of singular values above rounding (all, unless M is deficient;
    a zero one has a zero column, one of rounding an arbitrary one), and, if
    given, the singular values"""
    m, n = max(M.shape), min(M.shape)
    s = np.linalg.svd(M, compute_uv=False)
    tol = 8.0 * np.sqrt((60.0 if n > 256 or m > 1024 else 10.0) * (m + n)) * np.finfo(float).eps
    if svd is not None:
        assert np.abs(svd - s).max() <= tol * max(s[0], 1e-300)
    if not A2.nblk:
        assert s[0] == 0.0
        return
    U, V = A1.data[i], A2.data[i]
    # A2 is (R, new): psi = U V^T; V's columns carry the singular values
    assert np.linalg.norm(U @ V.T - M) <= tol * np.linalg.norm(M)
    sv = np.linalg.norm(V, axis=0)
    big = sv > tol * sv.max()
    assert big.sum() == (s > tol * s[0]).sum()
    G = U[:, big].T @ U[:, big]
    assert np.abs(G - np.eye(big.sum())).max(initial=0.0) <= tol


@pytest.mark.xfail(strict=True, raises=Q.QsxError,
                   reason="swept as they are, half-rank matrices of more than 256 columns do not end in 60 sweeps")
def test_svd_deficient_beyond_qr(gpu):
    M = _deficient(np.random.default_rng(3), 300, 260)
    Q.orthoQS(Q.QSpace([np.array([[0]]), np.array([[0]])], [M], "A", ["L", "R*"]), 1, stol=0.0)


# groups of every path in one call: in LDS and by rounds of column blocks after
# the QRs, as they are by column blocks and in one workgroup's LDS (beside small
# ones, that take the QRs here); all small, as they are
@pytest.mark.parametrize("shapes", [[(40, 30), (130, 110), (300, 260), (2000, 8), (20, 1), (96, 96), (97, 97), (9, 9)],
                                    [(130, 110), (256, 200), (12000, 1)], [(5, 4), (1, 1), (24, 24), (800, 6), (3, 90)]])
def test_svd_mixed_groups(gpu, shapes):
    rng = np.random.default_rng(len(shapes))
    mats = [rng.standard_normal(s if k % 2 else s[::-1]) for k, s in enumerate(shapes)]
    lab = [np.arange(len(mats))[:, None]] * 2
    A1, A2, info = Q.orthoQS(Q.QSpace(lab, mats, "A", ["L", "R*"]), 1, stol=0.0)
    assert info["ngroups"] == len(mats)
    for i, M in enumerate(mats):
        _check_group(M, A1, A2, i, None)
    s = np.sort(np.concatenate([np.linalg.svd(M, compute_uv=False) for M in mats]))[::-1]
    assert np.abs(info["svd"] - s).max() <= 1e-12 * s[0]


# group matrices that are swept as they are (8 x 6), in LDS after the QRs (60 x
# 40), by rounds of column blocks (130 x 110) and, beyond the QRs, as they are
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("m,n", [(8, 6), (60, 40), (130, 110), (300, 200), (300, 260)])
def test_svd_non_finite(gpu, m, n, bad):
    """a NaN or an infinity in one column of a group leaves the other columns'
    decomposition and the other groups finite.  Tolerance as in
    test_svd_shapes."""
    rng = np.random.default_rng(m + n)
    M, other = rng.standard_normal((m, n)), rng.standard_normal((50, 40))
    M[m // 3, n // 2] = bad
    P = Q.QSpace([np.array([[0], [1]]), np.array([[0], [1]])], [M, other], "A", ["L", "R*"])
    A1, A2, info = Q.orthoQS(P, 1, stol=0.0)
    svd = np.asarray(info["svd"])
    fin = np.sort(svd[np.isfinite(svd)])
    ref = np.sort(np.concatenate([np.linalg.svd(np.delete(M, n // 2, 1), compute_uv=False),
                                  np.linalg.svd(other, compute_uv=False)]))
    tol = 8.0 * np.sqrt(60.0 * (m + n)) * np.finfo(float).eps
    assert len(svd) == n + 40 and len(fin) == n + 39
    assert np.abs(fin - ref).max() <= tol * ref[-1]
    U = A1.data[0][:, np.isfinite(A1.data[0]).all(axis=0)]
    assert U.shape == (m, n - 1) and np.abs(U.T @ U - np.eye(n - 1)).max() <= tol
    assert np.linalg.norm(A1.data[1] @ A2.data[1].T - other) <= tol * np.linalg.norm(other)
