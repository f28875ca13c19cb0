"""Performance cases: what a DMRG program asks of this framework at one site
of a sweep -- H*psi on device vectors, the eigensolvers around it, the
truncation of the result, the environment update and the contractions
between -- over the sizes, symmetries and modes of this repository's own
workloads.

A case is a dict of plain values.  Its sector layout (labels and block
dimensions) follows from the case alone (``layout`` seeds it); the block
entries follow from the seed of ``prepare``.  ``exact`` restates every path
in numpy from the labels and blocks alone: Clebsch-Gordan tensors from the
closed forms of coupling to spin 0, 1/2 and 1, contractions block by block,
LAPACK singular values.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import qspace_amd as Q
from qspace_amd import gen

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # The smallest call: overlap matrix of a U(1) MPS tensor with itself,
        # contractQS(A,'12*',A,'12'), blocks of 4..32 states in host memory
        # in, host memory out.  Latency, launches and copies.
        dict(name="overlap_u1", kind="overlap", nq=11, dmin=4, dmax=32, layout=1001),
        # One environment step L.A.conj(A) of an SU(2) MPS with ~600
        # multiplets per bond, as two contraction plans on device buffers.
        dict(name="env_step_su2", kind="envstep", nl=17, dmin=8, dmax=64, layout=1002),
        # Environment update {A,'!2*',{{A,HK},W}} of a U(1) MPS (about 1700
        # states per bond, MPO bond 3 per charge): the cell form, host in and out.
        dict(name="env_update_u1", kind="envupdate", nq=21, dmin=40, dmax=120, dw=3, layout=1006),
        # Small H*psi, pseudo-MPO form (block Hamiltonians and two operator
        # pairs): the sites near the ends of a chain and the warm-up sweeps.
        dict(name="hpsi_pseudo_300", kind="hpsi", model="pseudo", D=300, nop=2, mode="batched", layout=1008),
        # The two-site H*psi of the Heisenberg chain at 4000 multiplets.
        dict(name="hpsi_heis_4000", kind="hpsi", model="heis", D=4000, nop=0, mode="batched", layout=1003),
        # The same at a production bond, the largest H*psi.
        dict(name="hpsi_heis_16000", kind="hpsi", model="heis", D=16000, nop=0, mode="batched", layout=1003),
        # Hubbard chain, two symmetries, parity signs, larger and more ragged blocks.
        dict(name="hpsi_hubbard_4000", kind="hpsi", model="hubbard", D=4000, nop=0, mode="batched", layout=1005),
        # Split precision (BF16 slices, the mode's default count).
        dict(name="hpsi_bf16_4000", kind="hpsi", model="heis", D=4000, nop=0, mode="split_bf16", layout=1003),
        # The eigensolver of one site update, both methods.
        dict(name="lanczos20_heis_2000", kind="eig", model="heis", D=2000, nop=0, method="lanczos", niter=20,
             layout=1003),
        dict(name="davidson30_hubbard_4000", kind="eig", model="hubbard", D=4000, nop=0, method="davidson", niter=30,
             layout=1005),
        # The truncation after it and the truncated wave function A1.A2: a
        # U(1) two-site psi with about 1000 states per bond (group matrices
        # up to 250 x 190) whose singular values fall over six decades ...
        dict(name="ortho_u1_1000", kind="ortho", form="u1", nq=11, dmin=40, dmax=140, decay=14.0, keep=512,
             layout=1009),
        # ... and an SU(2) MPS tensor with 17 multiplets per bond (group
        # matrices up to 128 x 64), left-orthonormalised.
        dict(name="ortho_su2_left", kind="ortho", form="su2_left", nq=17, dmin=8, dmax=64, decay=14.0, keep=64,
             layout=1002),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """one more case of the ranges above: bonds of 100..16000 multiplets (D*),
    3..21 sectors per bond, blocks of one to 140 states, both eigensolvers
    with 6..30 iterations, FP64 and the split modes"""
    layout = rng.randint(1, 10**6)
    kind = rng.choice(["overlap", "envstep", "envupdate", "hpsi", "hpsi", "hpsi", "hpsi", "eig", "eig", "ortho",
                       "ortho"])
    if kind == "overlap":
        dmin = rng.randint(1, 12)
        return dict(kind=kind, nq=rng.randint(3, 21), dmin=dmin, dmax=dmin + rng.randint(2, 60), layout=layout)
    if kind == "envstep":
        dmin = rng.randint(1, 16)
        return dict(kind=kind, nl=rng.randint(3, 25), dmin=dmin, dmax=dmin + rng.randint(4, 80), layout=layout)
    if kind == "envupdate":
        dmin = _logint(rng, 2, 40)
        return dict(kind=kind, nq=rng.randint(5, 21), dmin=dmin, dmax=dmin + _logint(rng, 4, 75), dw=rng.randint(1, 3),
                    layout=layout)
    if kind in ("hpsi", "eig"):
        model = rng.choice(["heis", "heis", "hubbard", "pseudo"])
        top = 4000 if kind == "eig" or model != "heis" else 16000
        c = dict(kind=kind, model=model, D=_logint(rng, 100, top), nop=rng.randint(1, 4) if model == "pseudo" else 0,
                 layout=layout)
        if kind == "eig":
            c.update(method=rng.choice(["lanczos", "davidson"]), niter=rng.randint(6, 24))
        else:
            c["mode"] = "batched" if model == "pseudo" or c["D"] > 4000 else \
                rng.choice(["batched", "batched", "batched", "split_bf16", "split_f32"])
        return c
    form = rng.choice(["u1", "u1", "su2_left", "su2_right"])
    dmin = _logint(rng, 2, 30)
    dmax = dmin + _logint(rng, 4, 80 if form == "u1" else 50)
    return dict(kind=kind, form=form, nq=rng.randint(4, 11) if form == "u1" else rng.randint(4, 17), dmin=dmin,
                dmax=dmax, decay=rng.choice([0.0, 7.0, 14.0]), keep=rng.randint(16, 512), layout=layout)


# ----------------------------------------------------------- layouts and data


def _charges(n):
    return tuple(range(-(n - 1), n, 2))


@functools.lru_cache(maxsize=8)
def _layout(key):
    """the tensors of a case with the generator's entries: labels, block
    dimensions and itags are used, the entries are replaced by _filled"""
    c = dict(key)
    kind, seed = c["kind"], c["layout"]
    if kind == "overlap":
        L = _charges(c["nq"])
        return (gen.u1_mps(seed=seed, Lq=L, Rq=tuple(q - 1 for q in L) + (L[-1] + 1,), dmin=c["dmin"],
                           dmax=c["dmax"]),)
    if kind == "envstep":
        A, L = gen.su2_mps(seed=seed, tS=tuple(range(c["nl"])), dmin=c["dmin"], dmax=c["dmax"])
        return L, A
    if kind == "envupdate":
        L = _charges(c["nq"])
        return gen.u1_env_update(seed=seed, Lq=L, Rq=tuple(q - 1 for q in L) + (L[-1] + 1,), dmin=c["dmin"],
                                 dmax=c["dmax"], dw=c["dw"])
    if kind in ("hpsi", "eig"):
        if c["model"] == "heis":
            return gen.heis_hpsi(seed=seed, Dstar=c["D"])
        if c["model"] == "hubbard":
            return gen.hubbard_hpsi(seed=seed, Dstar=c["D"])
        HKL, psi, HKR, OPL, OPR = gen.heis_pseudo_hpsi(seed=seed, Dstar=c["D"], nop=c["nop"])
        return (HKL, psi, HKR, *OPL, *OPR)
    if c["form"] == "u1":
        L = _charges(c["nq"])
        return (gen.u1_two_site_psi(seed=seed, Lq=L, Rq=L, dmin=c["dmin"], dmax=c["dmax"]),)
    return (gen.su2_mps(seed=seed, tS=tuple(range(c["nq"])), dmin=c["dmin"], dmax=c["dmax"])[0],)


def _templates(case):
    return _layout(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "mode", "method", "niter", "keep",
                                                                             "decay"))))


def _filled(T, rng, scale=1.0):
    return T.with_packed(scale * rng.standard_normal(T.numel()))


def _rows_cols(P, K):
    """groups of a wave function split after K legs: {label of the new leg:
    (row records, column records, [(block, row, column)])}, the group label
    read off the incoming legs (their sum; the last leg for K = r-1, the
    first for K = 1)"""
    groups = {}
    for i in range(P.nblk):
        rec = [tuple(int(x) for x in P.Q[k][i]) for k in range(P.rank)]
        if K == 1:
            g = rec[0]
        elif K == P.rank - 1:
            g = rec[-1]
        else:
            g = tuple(sum(r[c] for r in rec[:K]) for c in range(P.qdim))
        rows, cols, blk = groups.setdefault(g, ({}, {}, []))
        d = P.data[i].shape
        rows[tuple(rec[:K])] = int(np.prod(d[:K]))
        cols[tuple(rec[K:])] = int(np.prod(d[K:]))
        blk.append((i, tuple(rec[:K]), tuple(rec[K:])))
    return groups


def _offsets(d):
    off, o = {}, 0
    for r in sorted(d):
        off[r] = o
        o += d[r]
    return off, o


def _wave_function(P, K, decay, rng):
    """psi with singular values exp(-decay k/n) (k < n) in every group, as a
    ground state has them; decay = 0: N(0,1) entries"""
    if decay == 0.0:
        return _filled(P, rng)
    data = [None] * P.nblk
    for g, (rows, cols, blk) in sorted(_rows_cols(P, K).items()):
        ro, m = _offsets(rows)
        co, n = _offsets(cols)
        r = min(m, n)
        X = rng.standard_normal((m, r)) / math.sqrt(m)
        Y = rng.standard_normal((r, n)) / math.sqrt(n)
        M = (X * np.exp(-decay * np.arange(r) / r)) @ Y
        for i, a, b in blk:
            data[i] = M[ro[a]: ro[a] + rows[a], co[b]: co[b] + cols[b]].reshape(P.data[i].shape, order="F")
    return P.with_packed(np.concatenate([d.ravel(order="F") for d in data]))


def _inputs(case, seed):
    """the tensors of a case with entries from the seed, and for H*psi and
    the eigensolvers the normalised vector they act on"""
    rng = np.random.default_rng([int(seed), case["layout"]])
    T = _templates(case)
    if case["kind"] in ("hpsi", "eig"):
        k = 1  # psi's position
        T = [t if i == k else _filled(t, rng) for i, t in enumerate(T)]
        if case["model"] == "pseudo":  # block Hamiltonians are symmetric
            for i in (0, 2):
                T[i] = T[i].with_packed(np.concatenate([(0.5 * (d + d.T)).ravel(order="F") for d in T[i].data]))
        x = rng.standard_normal(T[k].numel())
        return T, x / np.linalg.norm(x)
    if case["kind"] == "ortho":
        return [_wave_function(T[0], _split(case), case["decay"], rng)], None
    return [_filled(t, rng) for t in T], None


def _split(case):
    return 1 if case["form"] == "su2_right" else 2


# ---------------------------------------------------------- prepare and run


class DeviceArray:
    """device vector of doubles as the plans take it (an object with .ptr)"""

    def __init__(self, a):
        self.t = a if isinstance(a, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(a)).cuda()
        self.ptr = ctypes.c_void_p(self.t.data_ptr())

    @classmethod
    def empty(cls, n):
        return cls(torch.zeros(n, dtype=torch.float64, device="cuda"))


def _hpsi_plan(case, T):
    mode = case.get("mode", "batched")
    if case["model"] == "pseudo":
        n = case["nop"]
        return Q.HPsi.pseudo(T[0], T[1], T[2], T[3:3 + n], T[3 + n:], mode=mode)
    ferm = gen.fermion_parity_signs(T[0]) if case["model"] == "hubbard" else None
    return Q.HPsi(T[0], T[1], T[2], hconj=1, fermA=ferm, mode=mode)


def prepare(case, seed):
    T, x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "envstep":
        L, A = T
        P1 = Q.CtrPlan(L, "2", A, "1")
        P2 = Q.CtrPlan(P1.out, "12", A, "12*")
        return dict(kind=kind, P1=P1, P2=P2, L=DeviceArray(L.packed()), A=DeviceArray(A.packed()),
                    X=DeviceArray.empty(P1.nout), C=DeviceArray.empty(P2.nout))
    if kind == "hpsi":
        return dict(kind=kind, H=_hpsi_plan(case, T), x=DeviceArray(x), y=DeviceArray.empty(x.size))
    if kind == "eig":
        H = _hpsi_plan(case, T)
        return dict(kind=kind, solve=getattr(H, case["method"]), x=x, niter=case["niter"])
    if kind == "ortho":
        return dict(kind=kind, psi=T[0], K=_split(case), keep=case["keep"])
    return dict(kind=kind, T=T)


def run(state):
    kind = state["kind"]
    if kind == "overlap":
        A, = state["T"]
        return Q.contractQS(A, "12*", A, "12").data
    if kind == "envstep":
        state["P1"].execute(state["L"], state["A"], state["X"])
        state["P2"].execute(state["X"], state["A"], state["C"])
        return state["X"].t, state["C"].t
    if kind == "envupdate":
        A, HK, W = state["T"]
        return Q.contractQS([A, "!2*", [[A, HK], W]]).data
    if kind == "hpsi":
        state["H"].apply_dev(state["x"], state["y"])
        return state["y"].t
    if kind == "eig":
        e0, ritz, gs = state["solve"](state["x"], state["niter"])
        return dict(e0=e0, ritz=ritz, gs=gs)
    # ortho: the singular vectors are defined up to their signs; what a
    # program goes on with is the truncated wave function A1.A2
    psi, K = state["psi"], state["K"]
    A1, A2, info = Q.orthoQS(psi, K, Nkeep=state["keep"])
    return dict(svd=info["svd"], psi=Q.contractQS(A1, [K + 1], A2, [psi.rank - K + 1]).data)


# ------------------------------------------------------------ work, tolerance


def _dims(T):
    return {tuple(tuple(int(x) for x in T.Q[k][i]) for k in range(T.rank)): T.data[i].shape[:T.rank]
            for i in range(T.nblk)}


def _pair_flops(A, ia, B, ib, keep=None):
    """2 M N K over the block pairs whose contracted labels match (and whose
    result labels `keep` takes), and the result's {labels: dims} (kept legs
    of A, then of B)"""
    ka = [k for k in range(len(next(iter(A)))) if k not in ia]
    kb = [k for k in range(len(next(iter(B)))) if k not in ib]
    by = {}
    for r, d in B.items():
        by.setdefault(tuple(r[k] for k in ib), []).append((r, d))
    fl, out = 0.0, {}
    for r, d in A.items():
        for s, e in by.get(tuple(r[k] for k in ia), ()):
            key = tuple(r[k] for k in ka) + tuple(s[k] for k in kb)
            if keep and not keep(key):
                continue
            dim = tuple(d[k] for k in ka) + tuple(e[k] for k in kb)
            fl += 2.0 * float(np.prod(dim)) * float(np.prod([d[k] for k in ia]))
            out[key] = dim
    return fl, out


def _numel(A):
    return sum(float(np.prod(d)) for d in A.values())


def work(case):
    T = [_dims(t) for t in _templates(case)]
    kind = case["kind"]
    if kind == "overlap":
        fl, C = _pair_flops(T[0], (0, 1), T[0], (0, 1))
        return dict(bytes=8.0 * (_numel(T[0]) + _numel(C)), flops=fl)
    if kind == "envstep":
        f1, X = _pair_flops(T[0], (1,), T[1], (0,))
        f2, C = _pair_flops(X, (0, 1), T[1], (0, 1), lambda r: r[0] == r[1])  # an SU(2) scalar's blocks
        return dict(bytes=8.0 * (_numel(T[0]) + _numel(T[1]) + _numel(X) + _numel(C)), flops=f1 + f2)
    if kind == "envupdate":
        A, HK, W = T
        f1, X = _pair_flops(A, (0,), HK, (0,))                    # (R, s, L, w)
        f2, Y = _pair_flops(X, (3, 1), W, (0, 2))                 # (R, L, w2, s)
        f3, C = _pair_flops(A, (0, 2), Y, (1, 3))                 # (R, R, w2)
        return dict(bytes=8.0 * (_numel(A) + _numel(HK) + _numel(W) + _numel(C)), flops=f1 + f2 + f3)
    if kind in ("hpsi", "eig"):
        fl = _hpsi_flops(case)
        ops = sum(_numel(t) for i, t in enumerate(T) if i != 1)
        n = _numel(T[1])
        if kind == "hpsi":
            return dict(bytes=8.0 * (ops + 2 * n), flops=fl)
        k = case["niter"]
        # k H*psi, and against a growing basis two Gram-Schmidt passes of a
        # dot product and an update each
        return dict(bytes=8.0 * (ops + 2 * n), flops=k * fl + 4.0 * n * k * (k + 1))
    P, K = _templates(case)[0], _split(case)
    fl = 0.0
    for rows, cols, _ in _rows_cols(P, K).values():
        m, n = sorted((sum(rows.values()), sum(cols.values())), reverse=True)
        fl += 6.0 * m * n * n + 20.0 * n**3  # SVD with both sets of vectors (Golub, Van Loan, R-SVD)
    return dict(bytes=8.0 * 3 * P.numel(), flops=fl)


def tolerance(case):
    """about four times the largest error against ``exact`` seen over the
    listed and drawn cases"""
    kind = case["kind"]
    if kind == "hpsi" and case["mode"] == "split_bf16":
        return {"rel": 4e-14}
    if kind == "hpsi" and case["mode"] == "split_f32":
        return {"rel": 6e-10}
    if kind == "eig":  # rounding grows along the Krylov space
        return {"rel": 2e-13}
    if kind == "ortho":
        return {"rel": 8e-13}
    return {"rel": 3e-15}


# ------------------------------------------------------- SU(2) in closed form
# A block's Clebsch-Gordan tensor: the unit-norm invariant tensor of its
# labels (2S per leg, directions +1 / -1) whose first non-zero entry in the
# canonical leg order (majority direction first, ascending labels) is
# positive; index i = S - m, the first leg fastest.


def _cg_small(a, ma, s, ms, b, mb):
    """<a ma; s ms | b mb> for s = 0, 1/2, 1, all arguments doubled"""
    if ma + ms != mb or abs(ma) > a or abs(ms) > s or abs(mb) > b:
        return 0.0
    if s == 0:
        return 1.0 if a == b else 0.0
    j, M = a / 2.0, mb / 2.0
    if s == 1:
        up, dn = math.sqrt((j + M + 0.5) / (2 * j + 1)), math.sqrt(max(0.0, j - M + 0.5) / (2 * j + 1))
        if b == a + 1:
            return up if ms > 0 else dn
        return -dn if ms > 0 else up
    k = ms // 2
    if b == a + 2:
        if k == 1:
            return math.sqrt((j + M) * (j + M + 1) / ((2 * j + 1) * (2 * j + 2)))
        if k == 0:
            return math.sqrt((j - M + 1) * (j + M + 1) / ((2 * j + 1) * (j + 1)))
        return math.sqrt((j - M) * (j - M + 1) / ((2 * j + 1) * (2 * j + 2)))
    if b == a:
        if k == 1:
            return -math.sqrt((j + M) * (j - M + 1) / (2 * j * (j + 1)))
        if k == 0:
            return M / math.sqrt(j * (j + 1))
        return math.sqrt((j - M) * (j + M + 1) / (2 * j * (j + 1)))
    if k == 1:
        return math.sqrt((j - M) * (j - M + 1) / (2 * j * (2 * j + 1)))
    if k == 0:
        return -math.sqrt((j - M) * (j + M) / (j * (2 * j + 1)))
    return math.sqrt((j + M + 1) * (j + M) / (2 * j * (2 * j + 1)))


def _threej(t, m):
    """3j symbol of three labels of which one is at most 1, up to a factor
    that does not depend on m"""
    k = min(range(3), key=lambda i: t[i])
    a, b = [i for i in range(3) if i != k]
    ph = -1.0 if ((t[b] - m[b]) // 2) % 2 else 1.0
    return ph * _cg_small(t[a], m[a], t[k], m[k], t[b], -m[b])


@functools.lru_cache(maxsize=None)
def _canon(t, d):
    """(canonical leg order, flags, sign / norm) of a block's CG tensor"""
    r = len(t)
    nin = sum(x > 0 for x in d)
    flip = nin < (r + 1) // 2
    fl = [(0 if d[k] > 0 else 1) ^ int(flip) for k in range(r)]
    o = sorted(range(r), key=lambda k: (fl[k], t[k]))
    if r == 2:
        if fl[0] != fl[1] and t[o[0]] > t[o[1]]:
            o.reverse()
        same = fl[0] == fl[1]
        sign = -1.0 if same and t[0] % 2 else 1.0
        return tuple(o), same, sign / math.sqrt(t[0] + 1)
    alike = fl[0] == fl[1] == fl[2]
    c = [t[k] for k in o]
    k = min(range(3), key=lambda i: c[i])
    b = max(i for i in range(3) if i != k)
    norm = math.sqrt(c[b] + 1)  # the sum of the squared entries is 2S + 1 of the coupled leg
    for m2 in range(c[2], -c[2] - 1, -2):
        for m1 in range(c[1], -c[1] - 1, -2):
            m0 = -m1 - m2 if alike else m2 - m1
            if abs(m0) > c[0]:
                continue
            v = _raw3(c, (m0, m1, m2), alike)
            if abs(v) > 1e-14 * norm:
                return tuple(o), alike, (1.0 if v > 0 else -1.0) / norm
    raise ValueError("vanishing CG tensor")


def _raw3(c, m, alike):
    if alike:
        return _threej(c, m)
    ph = -1.0 if ((c[2] - m[2]) // 2) % 2 else 1.0
    return ph * _threej(c, (m[0], m[1], -m[2]))


def _entry(t, d, m):
    """entry of the block's CG tensor at doubled m"""
    if len(t) < 2:
        return 1.0
    o, alike, f = _canon(t, d)
    mm = tuple(m[k] for k in o)
    c = [t[k] for k in o]
    if len(t) == 2:
        if alike:
            return 0.0 if mm[0] != -mm[1] else -f if ((c[0] - mm[0]) // 2) % 2 else f
        return f if mm[0] == mm[1] else 0.0
    if (mm[0] + mm[1] + mm[2] if alike else mm[0] + mm[1] - mm[2]) != 0:
        return 0.0
    return f * _raw3(c, mm, alike)


def _weight(t, d):
    """external norm of a block's CG tensor (rank <= 3)"""
    r = len(t)
    if r == 0 or all(x == 0 for x in t):
        return 1.0
    if r == 3:
        nin = sum(x > 0 for x in d)
        if nin in (0, 3):
            return 1.0
        odd = next(k for k in range(3) if (d[k] < 0) == (nin == 2))
        return math.sqrt(t[odd] + 1)
    return math.sqrt(max(t) + 1)


@functools.lru_cache(maxsize=None)
def _factor(ta, da, ia, tb, db, ib):
    """factor of a block product: the two CG tensors contracted, relative to
    the result's CG tensor, with the external norms"""
    ka = [k for k in range(len(ta)) if k not in ia]
    kb = [k for k in range(len(tb)) if k not in ib]
    tc = tuple(ta[k] for k in ka) + tuple(tb[k] for k in kb)
    dc = tuple(da[k] for k in ka) + tuple(db[k] for k in kb)
    if len(tc) == 2 and tc[0] != tc[1] or len(tc) == 3 and not (
            abs(tc[0] - tc[1]) <= tc[2] <= tc[0] + tc[1] and sum(tc) % 2 == 0):
        return 0.0
    # an entry of the result's tensor that is not small
    best, mc = 0.0, None
    o, alike, _ = _canon(tc, dc)
    if len(tc) == 2:
        mc = (tc[0], -tc[0] if alike else tc[0])
        best = _entry(tc, dc, mc)
    else:
        k = min(range(3), key=lambda i: tc[i])
        a, b = [i for i in range(3) if i != k]
        sg = [1 if alike else (1 if i != o[2] else -1) for i in range(3)]
        for mk in range(tc[k], -tc[k] - 1, -2):
            for ma in range(tc[a], max(-tc[a], tc[a] - 8) - 1, -2):
                mb = -(sg[k] * mk + sg[a] * ma) * sg[b]
                m = [0, 0, 0]
                m[k], m[a], m[b] = mk, ma, mb
                if abs(mb) <= tc[b] and abs(v := _entry(tc, dc, tuple(m))) > abs(best):
                    best, mc = v, tuple(m)
    ma, mb = [0] * len(ta), [0] * len(tb)
    for k, v in zip(ka, mc):
        ma[k] = v
    for k, v in zip(kb, mc[len(ka):]):
        mb[k] = v
    acc = 0.0
    big = max(range(len(ia)), key=lambda q: ta[ia[q]])

    def fill(q):
        nonlocal acc
        if q == len(ia):
            # the largest contracted label's m from each value that conserves m
            t = ta[ia[big]]
            for v in {s * sum(f) for f in _signs(ma, ia[big]) for s in (1, -1)}:
                if abs(v) <= t and (v - t) % 2 == 0:
                    ma[ia[big]] = mb[ib[big]] = v
                    e = _entry(ta, da, tuple(ma))
                    if e:
                        acc += e * _entry(tb, db, tuple(mb))
            return
        if q == big:
            fill(q + 1)
            return
        for v in range(ta[ia[q]], -ta[ia[q]] - 1, -2):
            ma[ia[q]] = mb[ib[q]] = v
            fill(q + 1)

    fill(0)
    return acc / best * _weight(ta, da) * _weight(tb, db) / _weight(tc, dc)


def _signs(m, skip):
    """the other legs' m with every choice of signs"""
    out = [()]
    for i, v in enumerate(m):
        if i != skip:
            out = [f + (s * v,) for f in out for s in ((1, -1) if v else (1,))]
    return out


def _su2_cols(T):
    return [j for j, s in enumerate((T.qtype or "").split(",")) if s.strip() == "SU2"]


def _dirs(T, conj=0):
    return tuple((-1 if t.endswith("*") else 1) * (-1 if conj else 1) for t in T.itags)


def _pair_factor(A, ra, da, ia, B, rb, db, ib):
    f = 1.0
    for j in _su2_cols(A):
        f *= _factor(tuple(x[j] for x in ra), da, tuple(ia), tuple(x[j] for x in rb), db, tuple(ib))
    return f


def _recs(T):
    return [tuple(tuple(int(x) for x in T.Q[k][i]) for k in range(T.rank)) for i in range(T.nblk)]


def _contract(A, da, ia, B, db, ib):
    """{labels: block} of two block-sparse tensors given as (recs, data, T)"""
    recA, datA, TA = A
    recB, datB, TB = B
    ka = [k for k in range(len(recA[0])) if k not in ia]
    kb = [k for k in range(len(recB[0])) if k not in ib]
    by = {}
    for j, r in enumerate(recB):
        by.setdefault(tuple(r[k] for k in ib), []).append(j)
    out = {}
    for i, r in enumerate(recA):
        for j in by.get(tuple(r[k] for k in ia), ()):
            f = _pair_factor(TA, r, da, ia, TB, recB[j], db, ib)
            if f == 0.0:
                continue
            key = tuple(r[k] for k in ka) + tuple(recB[j][k] for k in kb)
            x = f * np.tensordot(datA[i], datB[j], axes=(ia, ib))
            out[key] = out[key] + x if key in out else x
    dc = tuple(da[k] for k in ka) + tuple(db[k] for k in kb)
    keys = sorted(out)
    return (keys, [out[k] for k in keys], TA), dc


# ------------------------------------------------------------- H*psi, restated


@functools.lru_cache(maxsize=8)
def _entries_of(key):
    """H*psi of a case as a list of (out block, in block, operators and the
    leg of each that meets psi, factor)"""
    case = dict(key)
    T = _layout(tuple(sorted((k, v) for k, v in case.items())))
    psi = T[1]
    pr = _recs(psi)
    left = {r[0]: i for i, r in enumerate(pr)}
    dp = _dirs(psi)
    out = []
    if case["model"] == "pseudo":
        n = case["nop"]
        terms = [(3 + j, 1, 3 + n + j, 0) for j in range(n)] + [(3 + j, 0, 3 + n + j, 1) for j in range(n)]
        for i, r in enumerate(pr):  # block Hamiltonians: the CG tensors are identities
            out.append((i, i, 0, 1, None, 0, 1.0))
            out.append((i, i, None, 0, 2, 1, 1.0))
    else:
        terms = [(0, 0, 2, 0), (0, 1, 2, 1)]
    for li, cl, ri, cr in terms:
        L, R = T[li], T[ri]
        dl, dr = _dirs(L, cl), _dirs(R, cr)
        la, ra = int(not cl), int(not cr)  # the outgoing bond leg meets psi
        rr = {(r[ra], r[2], r[1 - ra]): j for j, r in enumerate(_recs(R))}
        for k, r in enumerate(_recs(L)):
            j = left.get(r[la])
            i = left.get(r[1 - la])
            if i is None or j is None:
                continue
            rec = (pr[j][1], r[2], pr[i][1])
            m = rr.get(rec)
            if m is None:
                continue
            f = 1.0
            for c in _su2_cols(psi):
                tl, tp = tuple(x[c] for x in r), tuple(x[c] for x in pr[j])
                tr = [0, 0, rec[1][c]]
                tr[ra], tr[1 - ra] = rec[0][c], rec[2][c]
                f *= _factor(tl, dl, (la,), tp, dp, (0,))
                # T's legs: L's kept legs in order, then psi's right leg
                tt = (tl[1 - la], tl[2], tp[1])
                dt = (dl[1 - la], dl[2], dp[1])
                f *= _factor(tt, dt, (1, 2), tuple(tr), dr, (2, ra))
            if f != 0.0:
                out.append((i, j, li, la, ri, ra, f, k, m))
    return out


def _entries(case):
    return _entries_of(tuple(sorted((k, v) for k, v in case.items()
                                    if k not in ("name", "mode", "method", "niter"))))


def _hpsi_flops(case):
    T = _templates(case)
    psi, fl = [d.shape for d in T[1].data], 0.0
    for e in _entries(case):
        (a, b), (a1, b1) = psi[e[0]], psi[e[1]]
        if len(e) == 7:
            fl += 2.0 * a * b * (a if e[2] is not None else b)
        else:
            w = T[e[2]].data[e[7]].shape[2]
            fl += 2.0 * a * a1 * w * b1 + 2.0 * a * b1 * w * b
    return fl


def _operator(case, T):
    """y = H x in numpy (x, y: psi's blocks back to back, column-major)"""
    psi = T[1]
    shapes = [d.shape for d in psi.data]
    offs = np.concatenate([[0], np.cumsum([d.size for d in psi.data])])
    sign = None
    if case["model"] == "hubbard":  # Jordan-Wigner: odd operators meet odd kets
        sign = [-1.0 if (int(T[0].Q[2][i][1]) % 2) * (int(T[0].Q[1][i][1]) % 2) else 1.0 for i in range(T[0].nblk)]

    def apply(x):
        X = [x[offs[i]: offs[i + 1]].reshape(s, order="F") for i, s in enumerate(shapes)]
        Y = [np.zeros(s) for s in shapes]
        for e in _entries(case):
            if len(e) == 7:
                i, j, li, la, ri, ra, f = e
                # HK_L(a, a') psi and psi HK_R: the legs that match psi's are the outgoing ones
                Y[i] += T[li].data[i] @ X[j] if li is not None else X[j] @ T[ri].data[i].T
                continue
            i, j, li, la, ri, ra, f, k, m = e
            if sign is not None:
                f = f * sign[k]
            L, R = T[li].data[k], T[ri].data[m]
            if la == 0:
                L = L.transpose(1, 0, 2)
            if ra == 0:
                R = R.transpose(1, 0, 2)
            for w in range(L.shape[2]):  # L (a, a', w), R (b, b', w)
                Y[i] += f * (L[:, :, w] @ X[j] @ R[:, :, w].T)
        return np.concatenate([y.ravel(order="F") for y in Y])

    return apply


def _multiplets(psi):
    """full-space weight of every element: the multiplet dimension"""
    c = _su2_cols(psi)
    return np.concatenate([np.full(d.size, float(np.prod([int(psi.Q[0][i][j]) + 1 for j in c])))
                           for i, d in enumerate(psi.data)])


def _orthogonalise(V, r):
    for _ in range(2):
        r = r - V.T @ (V @ r)
    return r


def _lanczos(apply, x, w, niter):
    s = np.sqrt(w)
    V = [s * x / np.linalg.norm(s * x)]
    al, be = [], []
    for _ in range(niter):
        r = s * apply(V[-1] / s)
        al.append(float(V[-1] @ r))
        r = _orthogonalise(np.array(V), r)
        be.append(float(np.linalg.norm(r)))
        V.append(r / be[-1])
    ritz = []
    for k in range(1, niter + 1):
        lam, y = np.linalg.eigh(np.diag(al[:k]) + np.diag(be[:k - 1], 1) + np.diag(be[:k - 1], -1))
        ritz.append(lam[0])
    y = y[:, 0] * (1.0 if y[:, 0].sum() >= 0 else -1.0)
    return dict(e0=float(ritz[-1]), ritz=np.array(ritz), gs=(np.array(V[:niter]).T @ y) / s)


def _davidson(apply, x, w, niter):
    s = np.sqrt(w)
    V = [s * x / np.linalg.norm(s * x)]
    HV = [s * apply(V[0] / s)]
    ritz = []
    while True:
        A, B = np.array(V), np.array(HV)
        lam, y = np.linalg.eigh(0.5 * (A @ B.T + B @ A.T))
        ritz.append(lam[0])
        if len(ritz) == niter:
            break
        r = _orthogonalise(A, B.T @ y[:, 0] - lam[0] * (A.T @ y[:, 0]))
        V.append(r / np.linalg.norm(r))
        HV.append(s * apply(V[-1] / s))
    return dict(e0=float(ritz[-1]), ritz=np.array(ritz), gs=None)  # the vector's sign is not fixed


# ------------------------------------------------------------------- exact


def _truncated(P, K, keep):
    """singular values (descending) and psi cut to the largest `keep` of
    them, its norm restored"""
    su2 = _su2_cols(P)
    d = _dirs(P)
    parts = []
    for g, (rows, cols, blk) in sorted(_rows_cols(P, K).items()):
        qd = float(np.prod([g[c] + 1 for c in su2])) if su2 else 1.0
        ro, m = _offsets(rows)
        co, n = _offsets(cols)
        M = np.zeros((m, n))
        for i, a, b in blk:
            f = np.prod([_weight(tuple(x[c] for x in a + b), d) for c in su2]) / math.sqrt(qd) if su2 else 1.0
            M[ro[a]: ro[a] + rows[a], co[b]: co[b] + cols[b]] = f * P.data[i].reshape(rows[a], cols[b], order="F")
        parts.append((blk, rows, cols, ro, co, qd, *np.linalg.svd(M, full_matrices=False)))
    S = np.concatenate([p[7] for p in parts])
    D = np.concatenate([np.full(p[7].size, p[5]) for p in parts])
    cut = np.sort(S)[::-1][min(keep, S.size) - 1]
    tot, kept = float((S**2 * D).sum()), float((S[S >= cut]**2 * D[S >= cut]).sum())
    out = {}
    for blk, rows, cols, ro, co, qd, U, s, Vt in parts:
        n = int((s >= cut).sum())
        if n == 0:
            continue
        M = (U[:, :n] * s[:n]) @ Vt[:n] * math.sqrt(tot / kept)
        for a in rows:
            for b in cols:
                t = a + b
                if su2 and any(not (abs(t[0][c] - t[1][c]) <= t[2][c] <= t[0][c] + t[1][c]) for c in su2):
                    continue
                f = np.prod([_weight(tuple(x[c] for x in t), d) for c in su2]) / math.sqrt(qd) if su2 else 1.0
                i = next((q for q, x, y in blk if (x, y) == (a, b)), None)
                x = M[ro[a]: ro[a] + rows[a], co[b]: co[b] + cols[b]] / f
                out[t] = x.reshape(P.data[i].shape if i is not None else x.shape, order="F")
    return dict(svd=np.sort(S)[::-1].copy(), psi=[out[k] for k in sorted(out)])


def exact(case, seed):
    T, x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "overlap":
        A = (_recs(T[0]), T[0].data, T[0])
        return _contract(A, _dirs(T[0], 1), (0, 1), A, _dirs(T[0]), (0, 1))[0][1]
    if kind == "envstep":
        L, A = T
        tA = (_recs(A), A.data, A)
        X, dx = _contract((_recs(L), L.data, L), _dirs(L), (1,), tA, _dirs(A), (0,))
        C, _ = _contract(X, dx, (0, 1), tA, _dirs(A, 1), (0, 1))
        pack = lambda t: np.concatenate([b.ravel(order="F") for b in t[1]])
        return pack(X), pack(C)
    if kind == "envupdate":
        A, HK, W = [(_recs(t), t.data, t) for t in T]
        X, dx = _contract(A, _dirs(T[0]), (0,), HK, _dirs(T[1]), (0,))       # (R, s, L, w)
        Y, dy = _contract(X, dx, (3, 1), W, _dirs(T[2]), (0, 2))             # (R, L, w2, s)
        return _contract(A, _dirs(T[0], 1), (0, 2), Y, dy, (1, 3))[0][1]
    if kind == "hpsi":
        return _operator(case, T)(x)
    if kind == "eig":
        return (_lanczos if case["method"] == "lanczos" else _davidson)(_operator(case, T), x, _multiplets(T[1]),
                                                                        case["niter"])
    return _truncated(T[0], _split(case), case["keep"])
