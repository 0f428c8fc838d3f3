"""Performance cases of the tt-fort local-solver path on one GPU.

What is timed is what programs built on this library call: the projected
local operator in its precisions, the rank truncation, the local linear
solve with its block preconditioner, the learned preconditioner (inference
and training gradient), and whole driver calls (a time step and a block
eigensolve).  `listed()` names fixed cases, `draw()` gives more of the same
ranges, `prepare()` makes the inputs on the device from a seed, `run()` is
one pass, `work()` the operations and bytes of a pass and `exact()` the
result in 64 bits by plain numpy.

Flat arrays are column-major, as in the C ABI (include/ttfort_amd.h).
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "tt-fort_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import ttfort  # noqa: E402

DTYPES = {"f64": np.float64, "f32": np.float32, "c128": np.complex128, "c64": np.complex64}
MATVEC = {"f64": "ttf_dbfun3", "f32": "ttf_sbfun3", "c128": "ttf_zbfun3", "c64": "ttf_cbfun3"}


# ------------------------------------------------------------------- cases
def matvec(name, dtype, rx1, m, rx2, ra1, ra2, nvec, ry1=None, n=None, ry2=None):
    return {"name": name, "kind": "matvec", "dtype": dtype, "rx1": rx1, "m": m, "rx2": rx2, "ry1": ry1 or rx1,
            "n": n or m, "ry2": ry2 or rx2, "ra1": ra1, "ra2": ra2, "nvec": nvec}


def listed():
    return [
        # the second site of a spin chain: what a sweep does at the chain's
        # ends, and every solver's smallest call
        matvec("matvec_chain_end", "f64", 2, 2, 4, 5, 5, 1),
        # the largest local problem of the d = 64 Heisenberg sweep (rank 128,
        # MPO rank 5), applied to the block eigensolver's 8 vectors
        matvec("matvec_eig_block", "f64", 128, 2, 128, 5, 5, 8),
        # the local problem of the 6-D diffusion solve (64 points, rank 64,
        # operator rank 6), one Krylov vector
        matvec("matvec_amen", "f64", 64, 64, 64, 6, 6, 1),
        # the same operator in the mixed-precision solver, odd ranks
        matvec("matvec_amen_f32_odd", "f32", 61, 64, 57, 6, 6, 1),
        # the local problem of the TFIM time step (rank 64, MPO rank 3)
        matvec("matvec_ksl", "c128", 64, 2, 64, 3, 3, 1),
        # a large bond dimension, one block of vectors
        matvec("matvec_large", "f64", 512, 2, 512, 5, 5, 8),
        # truncation of the eigensolver's rank-128 unfolding with 5
        # eigenvectors: (r n) x (r B), singular values and left vectors
        {"name": "truncation_eig", "kind": "truncation", "r": 128, "n": 2, "B": 5, "side": "L"},
        # one local solve of the 6-D diffusion problem: block-Jacobi set-up,
        # GMRES to the local tolerance, the solution
        {"name": "local_solve_amen", "kind": "solve", "rx1": 64, "n": 64, "rx2": 64, "ra": 6, "tol": 1e-10},
        # one apply of the trained block preconditioner to that problem
        {"name": "learned_precond", "kind": "precond", "rx1": 64, "rx2": 64, "ra": 6},
        # one training batch of that network: loss and gradient
        {"name": "learned_gradient", "kind": "gradient", "M": 1024},
        # one time step of a TFIM chain at fixed rank (half of it right to
        # left, half left to right)
        {"name": "ksl_step", "kind": "ksl", "d": 20, "r": 32, "order": 20, "tau": 0.05},
        # the three lowest states of a disordered XXZ chain, to convergence
        {"name": "eigb_chain", "kind": "eigb", "d": 12, "B": 3, "rmax": 96, "eps": 1e-11, "seed": 0},
    ]


def _loguni(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_matvec(rng):
    form = rng.choice(["spin", "spin", "grid", "rect"])
    dtype = rng.choice(["f64", "f64", "f32", "c128", "c64"])
    if form == "spin":      # small modes, large ranks, blocks of vectors in the (real) eigensolver
        m, ra = rng.choice([2, 2, 3, 4]), rng.randint(2, 6)
        c = matvec("", dtype, _loguni(rng, 2, 512), m, _loguni(rng, 2, 512), ra, ra,
                   1 if dtype[0] == "c" else rng.choice([1, 3, 8]))
    elif form == "grid":    # large modes, one vector
        m, ra = _loguni(rng, 8, 64), rng.randint(2, 6)
        c = matvec("", dtype, _loguni(rng, 4, 64), m, _loguni(rng, 4, 64), ra, ra, 1)
    else:                   # the projection of a product: other ranks and modes for y than for x
        c = matvec("", dtype, _loguni(rng, 2, 96), rng.randint(2, 20), _loguni(rng, 2, 96), rng.randint(2, 6),
                   rng.randint(2, 6), 1, _loguni(rng, 2, 96), rng.randint(2, 20), _loguni(rng, 2, 96))
    del c["name"]
    return c


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "matvec", "matvec", "truncation", "solve", "precond", "gradient", "ksl",
                       "eigb"])
    if kind == "matvec":
        while True:
            c = _draw_matvec(rng)
            if work(c)["flops"] <= 4e10:
                return c
    if kind == "truncation":
        if rng.random() < 0.5:
            return {"kind": kind, "r": _loguni(rng, 8, 120), "n": rng.choice([2, 2, 3]) if rng.random() < 0.3 else 2,
                    "B": rng.randint(1, 5), "side": rng.choice(["L", "R"])}
        return {"kind": kind, "r": _loguni(rng, 8, 64), "n": _loguni(rng, 16, 64), "B": 1,
                "side": rng.choice(["L", "R"])}
    if kind == "solve":
        return {"kind": kind, "rx1": _loguni(rng, 4, 64), "n": _loguni(rng, 8, 64), "rx2": _loguni(rng, 4, 64),
                "ra": 2 * rng.randint(1, 3), "tol": 1e-10}
    if kind == "precond":
        return {"kind": kind, "rx1": _loguni(rng, 3, 64), "rx2": _loguni(rng, 3, 64), "ra": 2 * rng.randint(1, 3)}
    if kind == "gradient":
        return {"kind": kind, "M": _loguni(rng, 48, 4096)}
    if kind == "ksl":
        return {"kind": kind, "d": rng.randint(6, 20), "r": _loguni(rng, 4, 32), "order": rng.randint(8, 20),
                "tau": 0.05}
    return {"kind": kind, "d": rng.randint(9, 12), "B": rng.randint(1, 3), "rmax": 96, "eps": 1e-11,
            "seed": rng.randint(1, 1 << 20)}


# ------------------------------------------------------------------ inputs
def _normal(rng, dt, *shape):
    dt = np.dtype(dt)
    if dt.kind == "c":
        return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * math.sqrt(0.5)
    return rng.standard_normal(shape)


def _interfaces(c, rng, dt):
    """Projections of an operator onto orthonormal interface bases: the first
    MPO component carries the identity (when the ranks agree), the others
    have entries of order 1 / sqrt(rank)."""
    p1 = _normal(rng, dt, c["ry1"], c["rx1"], c["ra1"]) / math.sqrt(c["rx1"])
    p2 = _normal(rng, dt, c["rx2"], c["ra2"], c["ry2"]) / math.sqrt(c["rx2"])
    if c["rx1"] == c["ry1"]:
        p1[:, :, 0] = np.eye(c["rx1"])
    if c["rx2"] == c["ry2"]:
        p2[:, 0, :] = np.eye(c["rx2"])
    return p1, p2


def _matvec_inputs(c, seed):
    rng = np.random.default_rng(seed)
    dt = DTYPES[c["dtype"]]
    p1, p2 = _interfaces(c, rng, dt)
    A = _normal(rng, dt, c["ra1"], c["n"], c["m"], c["ra2"])
    x = _normal(rng, dt, c["rx1"], c["m"], c["rx2"], c["nvec"])
    x /= np.linalg.norm(x) / math.sqrt(c["nvec"])
    return [np.asarray(a, dtype=dt) for a in (p1, A, p2, x)]


def _unfolding(c, seed):
    """An unfolding of a converged core: interface indices weighted by their
    (decaying) singular values on both sides, times mode and block indices."""
    rng = np.random.default_rng(seed)
    r, n, B = c["r"], c["n"], c["B"]
    w = 10.0 ** (-3.0 * np.arange(r) / max(r - 1, 1))
    A = np.repeat(w, n)[:, None] * rng.standard_normal((r * n, r * B)) * np.tile(w, B)[None, :]
    return A / np.linalg.norm(A)


def _grid_operator(c, seed):
    """Local operator L1 x I x I + I x D x I + I x I x L2 of a diffusion
    solve (D the 1-D Dirichlet Laplacian, L1 and L2 its projections onto the
    interface bases), as a separable operator of rank `ra`: ra / 2 copies of
    the rank-2 form with weights that add up to one."""
    rng = np.random.default_rng(seed)
    n, k = c["n"], c["ra"] // 2

    def proj(r):
        e = np.sort(10.0 ** rng.uniform(1.0, 3.0, r))
        s = rng.standard_normal((r, r))
        s = 0.15 * (s + s.T) / math.sqrt(2.0 * r)
        return np.sqrt(e)[:, None] * (np.eye(r) + s) * np.sqrt(e)[None, :]

    L1, L2 = proj(c["rx1"]), proj(c["rx2"])
    D = (n + 1) ** 2 * (2.0 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1))
    w = rng.uniform(0.5, 1.5, k)
    w /= w.sum()
    ra = 2 * k
    p1 = np.zeros((c["rx1"], c["rx1"], ra))
    p2 = np.zeros((c["rx2"], ra, c["rx2"]))
    A = np.zeros((ra, n, n, ra))
    for t in range(k):
        p1[:, :, 2 * t], p1[:, :, 2 * t + 1] = L1, np.eye(c["rx1"])
        p2[:, 2 * t, :], p2[:, 2 * t + 1, :] = np.eye(c["rx2"]), L2
        A[2 * t, :, :, 2 * t] = w[t] * np.eye(n)
        A[2 * t + 1, :, :, 2 * t] = w[t] * D
        A[2 * t + 1, :, :, 2 * t + 1] = w[t] * np.eye(n)
    rhs = rng.standard_normal((c["rx1"], n, c["rx2"]))
    return L1, D, L2, p1, A, p2, rhs / np.linalg.norm(rhs)


def _params():
    return np.load(os.path.join(PKG, "models", "mlp_precond_n64.npy"))


def _batch(M, seed):
    """Training pairs as the collection makes them: normalised tridiagonal
    blocks and residual slices, and the blocks' solutions."""
    rng = np.random.default_rng(seed)
    dg = 1.0 + 0.2 * rng.uniform(-1.0, 1.0, (64, M))
    dg /= dg.mean(axis=0)
    up = -0.47 * np.ones((64, M)) * (1.0 + 0.05 * rng.uniform(-1.0, 1.0, (64, M)))
    up[63] = 0.0
    lo = up.copy()
    rs = rng.standard_normal((64, M))
    rs /= np.linalg.norm(rs, axis=0)
    # Thomas algorithm over all blocks
    cp, dp = np.zeros((64, M)), np.zeros((64, M))
    cp[0], dp[0] = up[0] / dg[0], rs[0] / dg[0]
    for i in range(1, 64):
        den = dg[i] - lo[i - 1] * cp[i - 1]
        cp[i], dp[i] = up[i] / den, (rs[i] - lo[i - 1] * dp[i - 1]) / den
    t = np.zeros((64, M))
    t[63] = dp[63]
    for i in range(62, -1, -1):
        t[i] = dp[i] - cp[i] * t[i + 1]
    X = np.concatenate([dg, up, lo, rs]).astype(np.float32)
    return X, t.astype(np.float32)


def _tfim(d, g=1.0):
    """A = -i H of the transverse-field Ising chain as an MPO of rank 3."""
    I2, X, Z = np.eye(2), np.array([[0.0, 1.0], [1.0, 0.0]]), np.diag([1.0, -1.0])
    W = np.zeros((3, 3, 2, 2), dtype=np.complex128)
    W[0, 0], W[1, 0], W[2, 0], W[2, 1], W[2, 2] = I2, Z, -g * X, -Z, I2
    return _mpo([W] * d, 2, 0, first=-1j)


def _mpo(Ws, row, col, first=1.0):
    cores, ra = [], [1]
    for k, W in enumerate(Ws):
        Wk = W[row:row + 1] * first if k == 0 else W[:, col:col + 1] if k == len(Ws) - 1 else W
        cores.append(np.transpose(Wk, (0, 2, 3, 1)).reshape(-1, order="F"))
        ra.append(Wk.shape[1])
    return np.concatenate(cores), np.array(ra), np.full(len(Ws), 2)


SZ = np.diag([0.5, -0.5])
SP = np.array([[0.0, 1.0], [0.0, 0.0]])


def _fields(c, seed):
    rng = np.random.default_rng([c["seed"], seed])
    return rng.uniform(0.8, 1.2), rng.uniform(0.5, 1.5), rng.uniform(-1.0, 1.0, c["d"])


def _xxz(c, seed):
    """Open XXZ chain in random fields along z, an MPO of rank 5."""
    J, delta, h = _fields(c, seed)
    Ws = []
    for hk in h:
        W = np.zeros((5, 5, 2, 2))
        W[0, 0], W[1, 0], W[2, 0], W[3, 0] = np.eye(2), SP, SP.T, SZ
        W[4, 0], W[4, 1], W[4, 2], W[4, 3], W[4, 4] = hk * SZ, 0.5 * J * SP.T, 0.5 * J * SP, J * delta * SZ, np.eye(2)
        Ws.append(W)
    return _mpo(Ws, 4, 0)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).reshape(-1, order="F"))).cuda()


def _empty(count, dt):
    return torch.empty(int(count), dtype=torch.from_numpy(np.empty(0, dt)).dtype, device="cuda")


def prepare(case, seed):
    lib = ttfort.load()
    ttfort.check(lib.ttf_init(0), lib)
    c, kind = case, case["kind"]
    s = {"case": dict(case), "lib": lib}
    if kind == "matvec":
        s["in"] = [_dev(a) for a in _matvec_inputs(c, seed)]
        s["shape"] = tuple(c[k] for k in ("rx1", "m", "rx2", "ry1", "n", "ry2", "ra1", "ra2"))
        s["y"] = _empty(c["ry1"] * c["n"] * c["ry2"] * c["nvec"], DTYPES[c["dtype"]])
    elif kind == "truncation":
        A = _unfolding(c, seed)
        m, n = A.shape
        s["m"], s["n"], s["A"] = m, n, _dev(A)
        s["S"], s["O"] = _empty(min(m, n), np.float64), _empty((m if c["side"] == "L" else n) * min(m, n), np.float64)
    elif kind == "solve":
        _, _, _, p1, A, p2, rhs = _grid_operator(c, seed)
        s["p1"], s["A"], s["p2"], s["rhs"] = _dev(p1), _dev(A), _dev(p2), _dev(rhs)
        s["jacs"] = _empty(lib.ttf_djac_size(b"c", c["rx1"], c["n"], c["rx2"]), np.float64)
        s["z"], s["sol"] = _empty(rhs.size, np.float64), _empty(rhs.size, np.float64)
        s["it"], s["rr"] = np.zeros(2, dtype=np.int32), np.zeros(1)
    elif kind == "precond":
        _, _, _, p1, A, p2, rhs = _grid_operator(dict(c, n=64), seed)
        s["p1"], s["A"], s["p2"], s["v"] = _dev(p1), _dev(A), _dev(p2), _dev(rhs)
        s["z"] = _empty(rhs.size, np.float64)
        ttfort.mlp_set_params(_params())
    elif kind == "gradient":
        X, T = _batch(c["M"], seed)
        s["X"], s["T"] = _dev(X), _dev(T)
        s["loss"], s["g"] = np.zeros(1), np.empty(ttfort.mlp_param_count(), dtype=np.float32)
        ttfort.mlp_set_params(_params())
    elif kind == "ksl":
        rng = np.random.default_rng(seed)
        d = c["d"]
        ry = [min(c["r"], 2 ** min(k, d - k)) for k in range(d + 1)]
        Y = [_normal(rng, np.complex128, ry[k] * 2 * ry[k + 1]) / math.sqrt(2 * ry[k]) for k in range(d)]
        s["op"], s["Y"], s["ry"] = _tfim(d), np.concatenate(Y), np.array(ry)
    elif kind == "eigb":
        rng = np.random.default_rng(seed)
        d, B = c["d"], c["B"]
        ry = [1] + [4] * (d - 1) + [B]
        s["op"] = _xxz(c, seed)
        s["Y"], s["ry"] = np.concatenate([rng.standard_normal(ry[k] * 2 * ry[k + 1]) for k in range(d)]), ry
    return s


# -------------------------------------------------------------------- runs
def run(state):
    s, c, lib = state, state["case"], state["lib"]
    kind = c["kind"]
    if kind == "matvec":
        p1, A, p2, x = s["in"]
        y = s["y"]
        nx, ny = c["rx1"] * c["m"] * c["rx2"], c["ry1"] * c["n"] * c["ry2"]
        ttfort.check(getattr(lib, MATVEC[c["dtype"]])(*s["shape"], c["nvec"], p1.data_ptr(), A.data_ptr(),
                                                      p2.data_ptr(), x.data_ptr(), nx, y.data_ptr(), ny), lib)
        return y
    if kind == "truncation":
        S, O = s["S"], s["O"]
        rows = s["m"] if c["side"] == "L" else s["n"]
        ttfort.check(lib.ttf_dsvd_side(s["m"], s["n"], s["A"].data_ptr(), s["m"], c["side"].encode(), S.data_ptr(),
                                       O.data_ptr(), rows, None, None), lib)
        # singular vectors are defined up to sign: the largest entry of each
        # is made positive
        V = O.view(-1, rows)
        V *= torch.sign(V.gather(1, V.abs().argmax(dim=1, keepdim=True)))
        torch.cuda.current_stream().synchronize()   # the library works on a stream of its own
        return {"S": S, "vectors": V}
    if kind == "solve":
        dims = (c["rx1"], c["n"], c["rx2"])
        p1, A, p2 = s["p1"].data_ptr(), s["A"].data_ptr(), s["p2"].data_ptr()
        ttfort.check(lib.ttf_djac_gen(b"c", *dims, c["ra"], c["ra"], p1, A, p2, s["jacs"].data_ptr()), lib)
        ttfort.check(lib.ttf_dgmresr(p1, A, p2, s["rhs"].data_ptr(), *dims, c["ra"], c["ra"], 40, c["tol"], 2, b"c",
                                     s["jacs"].data_ptr(), s["z"].data_ptr(), ttfort._ip(s["it"]),
                                     ttfort._dp(s["rr"])), lib)
        ttfort.check(lib.ttf_djac_apply(b"c", *dims, s["jacs"].data_ptr(), s["z"].data_ptr(), s["sol"].data_ptr()),
                     lib)
        return s["sol"]
    if kind == "precond":
        ttfort.check(lib.ttf_mlp_precond(c["rx1"], 64, c["rx2"], c["ra"], c["ra"], s["p1"].data_ptr(),
                                         s["A"].data_ptr(), s["p2"].data_ptr(), s["v"].data_ptr(),
                                         s["z"].data_ptr()), lib)
        return s["z"]
    if kind == "gradient":
        ttfort.check(lib.ttf_mlp_loss_grad(c["M"], s["X"].data_ptr(), s["T"].data_ptr(), ttfort._dp(s["loss"]),
                                           s["g"].ctypes.data), lib)
        return {"loss": s["loss"], "grad": s["g"]}
    if kind == "ksl":
        crA, ra, n = s["op"]
        cr, ry, _ = ttfort.ztt_ksl(n, ra, crA, s["Y"], s["ry"], c["tau"], order=c["order"])
        return {"cores": cr, "ranks": ry}
    crA, ra, n = s["op"]
    lam, cr, ry, _ = ttfort.tt_eigb(n, ra, crA, s["Y"], s["ry"], c["eps"], c["rmax"], c["B"], nswp=12,
                                    max_full_size=200)
    # the states as full vectors (each up to sign: its largest entry positive)
    x, p = np.ones((1, 1)), 0
    for k in range(c["d"]):
        size = int(ry[k]) * 2 * int(ry[k + 1])
        x = x @ cr[p:p + size].reshape(int(ry[k]), -1, order="F")
        x = x.reshape(-1, int(ry[k + 1]), order="F")
        p += size
    x = x * np.sign(np.take_along_axis(x, np.abs(x).argmax(axis=0)[None, :], axis=0))
    return {"lam": lam, "states": x}


# -------------------------------------------------------------------- work
def _matvec_work(c, size, mult):
    rx1, m, rx2, ry1, n, ry2, ra1, ra2 = (c[k] for k in ("rx1", "m", "rx2", "ry1", "n", "ry2", "ra1", "ra2"))
    flops = 2.0 * rx1 * m * rx2 * ra2 * ry2 + 2.0 * ra1 * n * m * ra2 * ry2 * rx1 + 2.0 * ry1 * n * ry2 * rx1 * ra1
    count = ry1 * rx1 * ra1 + rx2 * ra2 * ry2 + ra1 * n * m * ra2 + c["nvec"] * (rx1 * m * rx2 + ry1 * n * ry2)
    return {"bytes": float(size * count), "flops": mult * c["nvec"] * flops}


def work(case):
    c, kind = case, case["kind"]
    if kind == "matvec":
        dt = np.dtype(DTYPES[c["dtype"]])
        return _matvec_work(c, dt.itemsize, 4.0 if dt.kind == "c" else 1.0)
    if kind == "truncation":
        m, n = c["r"] * c["n"], c["r"] * c["B"]
        k = min(m, n)
        rows = m if c["side"] == "L" else n
        # QR of the long side, then an SVD of the square factor
        return {"bytes": 8.0 * (m * n + rows * k + k), "flops": 2.0 * max(m, n) * k * k + 12.0 * k ** 3}
    if kind == "solve":
        rx1, n, rx2, ra = c["rx1"], c["n"], c["rx2"], c["ra"]
        w = _matvec_work({"rx1": rx1, "m": n, "rx2": rx2, "ry1": rx1, "n": n, "ry2": rx2, "ra1": ra, "ra2": ra,
                          "nvec": 1}, 8, 1.0)
        # about 16 products with the operator and the preconditioner, the
        # blocks' inverses, one read of the basis per step
        return {"bytes": w["bytes"] + 17 * 8.0 * rx1 * rx2 * n * n,
                "flops": 16.0 * w["flops"] + rx1 * rx2 * (2.0 * n ** 3 + 34.0 * n * n)}
    if kind == "precond":
        nb = c["rx1"] * c["rx2"]
        return {"bytes": 8.0 * (2 * nb * 64 + c["ra"] * (c["rx1"] ** 2 + c["rx2"] ** 2) + (64 * c["ra"]) ** 2)
                + 2.0 * 147456, "flops": 2.0 * nb * 147456}
    if kind == "gradient":
        return {"bytes": 4.0 * c["M"] * 320 + 3 * 4.0 * 148032, "flops": 2.0 * c["M"] * (3 * 147456 - 65536)}
    d, total, size = c["d"], 0.0, 0.0
    if kind == "ksl":
        ry = [min(c["r"], 2 ** min(k, d - k)) for k in range(d + 1)]
        for k in range(d):
            w = _matvec_work({"rx1": ry[k], "m": 2, "rx2": ry[k + 1], "ry1": ry[k], "n": 2, "ry2": ry[k + 1],
                              "ra1": 3, "ra2": 3, "nvec": 1}, 16, 4.0)
            total += 2 * 2 * c["order"] * w["flops"]   # forward and backward exponentials, two half steps
            size += 16.0 * 2 * ry[k] * ry[k + 1]
        return {"bytes": 2 * size, "flops": total}
    B = c["B"]
    ry = [min(c["rmax"], 2 ** k, B * 2 ** (d - k)) for k in range(d + 1)]
    for k in range(d):
        w = _matvec_work({"rx1": ry[k], "m": 2, "rx2": ry[k + 1], "ry1": ry[k], "n": 2, "ry2": ry[k + 1], "ra1": 5,
                          "ra2": 5, "nvec": B}, 8, 1.0)
        total += 4 * 20 * w["flops"]                   # about 20 block products per site, two sweeps back and forth
        size += 8.0 * 2 * ry[k] * ry[k + 1]
    return {"bytes": size + 8.0 * B * 2 ** d, "flops": total}


# ------------------------------------------------------------------- exact
def _wide(a):
    return a.astype(np.complex128 if a.dtype.kind == "c" else np.float64)


def _bf16(w):
    u = np.ascontiguousarray(w, dtype=np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32).astype(np.float64)


def _network():
    p = _params()
    out, o = [], 0
    for k, n in ((256, 256), (256, 256), (256, 64)):   # weights are held in bf16, biases in fp32
        out.append((_bf16(p[o:o + k * n]).reshape(k, n, order="F"), p[o + k * n:o + k * n + n].astype(np.float64)))
        o += k * n + n
    return out


def _forward(X):
    (W1, b1), (W2, b2), (W3, b3) = _network()
    H1 = np.maximum(W1.T @ X + b1[:, None], 0.0)
    H2 = np.maximum(W2.T @ H1 + b2[:, None], 0.0)
    return H1, H2, W3.T @ H2 + b3[:, None] + X[192:] / X[:64]


def _xxz_states(c, seed):
    """Lowest states by exact diagonalisation within the sectors of fixed
    total Sz (site 1 is the fastest index of a full vector)."""
    d, B = c["d"], c["B"]
    J, delta, h = _fields(c, seed)
    idx = np.arange(2 ** d)
    bits = (idx[:, None] >> np.arange(d)[None, :]) & 1
    sz = 0.5 - bits
    diag = sz @ h + J * delta * (sz[:, :-1] * sz[:, 1:]).sum(axis=1)
    ups, found = bits.sum(axis=1), []
    for q in range(d + 1):
        sec = idx[ups == q]
        pos = np.full(2 ** d, -1)
        pos[sec] = np.arange(sec.size)
        H = np.diag(diag[sec])
        for k in range(d - 1):
            one = np.nonzero(bits[sec, k] != bits[sec, k + 1])[0]
            to = pos[sec[one] ^ (3 << k)]
            H[to, one] += 0.5 * J
        w, v = np.linalg.eigh(H)
        for t in range(min(B, w.size)):
            x = np.zeros(2 ** d)
            x[sec] = v[:, t]
            found.append((w[t], x))
    found.sort(key=lambda e: e[0])
    X = np.stack([x for _, x in found[:B]], axis=1)
    X = X * np.sign(np.take_along_axis(X, np.abs(X).argmax(axis=0)[None, :], axis=0))
    return {"lam": np.array([w for w, _ in found[:B]]), "states": X}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "matvec":
        p1, A, p2, x = (_wide(a) for a in _matvec_inputs(c, seed))
        t = np.tensordot(x, p2, axes=([2], [0]))                       # b1 j v a2 c2
        t = np.tensordot(A, t, axes=([2, 3], [1, 3]))                  # a1 i b1 v c2
        y = np.tensordot(p1, t, axes=([1, 2], [2, 0]))                 # c1 i v c2
        return np.transpose(y, (0, 1, 3, 2)).reshape(-1, order="F")
    if kind == "truncation":
        A = _unfolding(c, seed)
        U, S, VT = np.linalg.svd(A, full_matrices=False)
        V = U.T if c["side"] == "L" else VT
        V = V * np.sign(np.take_along_axis(V, np.abs(V).argmax(axis=1)[:, None], axis=1))
        return {"S": S, "vectors": V}
    if kind == "solve":
        L1, D, L2, _, _, _, rhs = _grid_operator(c, seed)
        (e1, q1), (e, q), (e2, q2) = (np.linalg.eigh(a) for a in (L1, D, L2))

        def rotate(v, a, b, w):
            v = np.tensordot(a, v, axes=([1], [0]))
            v = np.einsum("ij,bjc->bic", b, v, optimize=True)
            return np.tensordot(v, w, axes=([2], [1]))

        t = rotate(rhs, q1.T, q.T, q2.T) / (e1[:, None, None] + e[None, :, None] + e2[None, None, :])
        return rotate(t, q1, q, q2).reshape(-1, order="F")
    if kind == "precond":
        L1, D, L2, _, _, _, v = _grid_operator(dict(c, n=64), seed)
        dg = np.diag(L1)[:, None] + np.diag(L2)[None, :]               # b1 b2
        diag = np.diag(D)[:, None, None] + dg[None]                    # i b1 b2
        s = np.abs(diag).mean(axis=0)
        r = np.transpose(v, (1, 0, 2))
        rn = np.sqrt((r * r).sum(axis=0))
        off = np.full((64,) + dg.shape, -(65.0 ** 2))
        off[63] = 0.0
        X = np.concatenate([diag / s, off / s, off / s, r / rn]).reshape(256, -1, order="F")
        y = _forward(X)[2].reshape((64,) + dg.shape, order="F") * (rn / s)
        return np.transpose(y, (1, 0, 2)).reshape(-1, order="F")
    if kind == "gradient":
        X, T = (a.astype(np.float64) for a in _batch(c["M"], seed))
        (_, _), (W2, _), (W3, _) = _network()
        H1, H2, Y = _forward(X)
        dY = 2.0 * (Y - T) / Y.size
        dH2 = (W3 @ dY) * (H2 > 0)
        dH1 = (W2 @ dH2) * (H1 > 0)
        g = [(X @ dH1.T).reshape(-1, order="F"), dH1.sum(axis=1), (H1 @ dH2.T).reshape(-1, order="F"), dH2.sum(axis=1),
             (H2 @ dY.T).reshape(-1, order="F"), dY.sum(axis=1)]
        return {"loss": np.array([((Y - T) ** 2).mean()]), "grad": np.concatenate(g)}
    if kind == "ksl":
        return None     # the fixed-rank step has no closed form
    return _xxz_states(c, seed)
