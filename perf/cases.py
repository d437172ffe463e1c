"""Timed cases of the framework's work: dense DMRG on one GPU.

A case is one operation that a DMRG, TEBD or preconditioner-training program
spends its time in, called through the package's public functions: the
two-site effective Hamiltonian and its Davidson solve, the factorisations of
a bond (density matrix, SVD, QR), general contractions, a training step of
the learned preconditioner, and one whole DMRG sweep. `listed()` are fixed
points of the ranges, `draw(rng)` gives others; sizes come from the
benchmark's chain (N = 100, chi = 2048, w = 5), the N = 20 chain (chi 10 to
200), the cylinder (w = 14) and the chi = 1024 microbench, with ragged ones
between.

Factorisations are unique only up to a gauge (signs, rotations inside
degenerate spaces), so those passes hand back what the program goes on with:
the spectrum and the product of the factors.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "itensorsgpu.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

F64, F32, C128 = torch.float64, torch.float32, torch.complex128


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a Heff product at the first bonds and in the first sweeps of the
        # N = 20 chain (chi = 20): launches, not arithmetic
        dict(name="heff_fp64_chi20", op="heff", dtype="float64", mode="native",
             chiL=20, chiR=20, w=5, d=2),
        # the effective-Hamiltonian microbench in FP32, chi = 1024
        dict(name="heff_fp32_chi1024", op="heff", dtype="float32", mode="native",
             chiL=1024, chiR=1024, w=5, d=2),
        # the benchmark chain's bulk product in split-BF16, chi = 2048
        dict(name="heff_bf16x3_chi2048", op="heff", dtype="float32", mode="bf16x3",
             chiL=2048, chiR=2048, w=5, d=2),
        # the eigensolve of one bond of the cylinder (w = 14) part way up its
        # ramp, unequal ragged links, three Krylov vectors
        dict(name="davidson_cylinder_chi300", op="davidson", chiL=300, chiR=277, w=14, d=2,
             maxiter=2),
        # factorize of a bond of the N = 20 chain: density matrix of 200,
        # truncated by the cutoff
        dict(name="factorize_eigen_chi100", op="factorize", chiL=100, chiR=100, d=2,
             decay=18.0, cutoff=1e-10, maxdim=200, ortho="left"),
        # factorize of a bulk bond of the benchmark chain: density matrix of
        # 4096, truncated to chi = 2048
        dict(name="factorize_eigen_chi2048", op="factorize", chiL=2048, chiR=2048, d=2,
             decay=5.0, cutoff=1e-12, maxdim=2048, ortho="left"),
        # the microbench's truncated SVD: a dense 2048 x 2048 matrix with no
        # decay to speak of, cutoff 1e-10, kept 1024
        dict(name="svd_2048", op="svd", chiL=1024, chiR=1024, d=2, cutoff=1e-10, maxdim=1024),
        # gauge move of one site tensor (orthogonalize, random MPS)
        dict(name="qr_chi1000", op="qr", chiL=1000, chiR=1000, d=2),
        # a general contraction whose indices come in no convenient order,
        # ragged extents
        dict(name="contract_fp64_ragged", op="contract", dtype="float64", a=61, b=37, c=53,
             e=41, k1=47, k2=39),
        # a two-site gate on complex tensors (time evolution)
        dict(name="gate_c128_chi500", op="gate", chiL=500, chiM=430, chiR=610, d=2),
        # a training step of the learned preconditioner on every bond pair of
        # a chi = 64 bond: forward, backward, Adam
        dict(name="mlp_train_4096", op="mlp_train", rows=4096, d=2),
        # a whole DMRG sweep on a converged state of a disordered cylinder
        # (4 x 6 sites), the kept states at most 128
        dict(name="dmrg_sweep_4x6", op="dmrg", lx=6, ly=4, maxdim=128, cutoff=1e-9),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["heff", "heff", "davidson", "factorize", "factorize", "svd", "qr",
                     "contract", "contract", "gate", "mlp_train", "dmrg"])
    if op == "heff":
        dtype, mode, top = rng.choice([("float64", "native", 1024), ("float32", "native", 1024),
                                       ("float32", "bf16x3", 2048)])
        w, d = rng.choice([(5, 2), (3, 2), (5, 3), (14, 2)])
        top = int(top / (1.0 if d == 2 and w <= 5 else 1.8))
        chiL = _logint(rng, 10, top)
        return dict(op="heff", dtype=dtype, mode=mode, chiL=chiL,
                    chiR=max(4, int(chiL * rng.uniform(0.6, 1.0))), w=w, d=d)
    if op == "davidson":
        chiL = _logint(rng, 10, 500)
        return dict(op="davidson", chiL=chiL, chiR=max(4, int(chiL * rng.uniform(0.6, 1.0))),
                    w=rng.choice([3, 5, 14]), d=2, maxiter=rng.choice([1, 2, 3]))
    if op == "factorize":
        chiL = _logint(rng, 10, 1500)
        chiR = max(8, int(chiL * rng.uniform(0.7, 1.0)))
        big = chiL > 400
        return dict(op="factorize", chiL=chiL, chiR=chiR, d=2,
                    decay=round(rng.uniform(4.0, 6.0) if big else rng.uniform(10.0, 18.0), 3),
                    cutoff=1e-12 if big else 1e-10, maxdim=max(8, int(chiL * rng.uniform(0.7, 1.0))),
                    ortho=rng.choice(["left", "right"]))
    if op == "svd":
        chiL = _logint(rng, 10, 1000)
        chiR = max(8, int(chiL * rng.uniform(0.6, 1.0)))
        return dict(op="svd", chiL=chiL, chiR=chiR, d=2, cutoff=1e-10,
                    maxdim=max(6, int(chiL * rng.uniform(0.5, 1.0))))
    if op == "qr":
        chiL = _logint(rng, 10, 1800)
        return dict(op="qr", chiL=chiL, chiR=max(4, int(chiL * rng.uniform(0.5, 1.0))), d=2)
    if op == "contract":
        s = _logint(rng, 5, 60)
        v = [max(2, int(s * rng.uniform(0.6, 1.1))) for _ in range(6)]
        return dict(op="contract", dtype=rng.choice(["float64", "float32"]), a=v[0], b=v[1],
                    c=v[2], e=v[3], k1=v[4], k2=v[5])
    if op == "gate":
        chi = _logint(rng, 16, 700)
        return dict(op="gate", chiL=chi, chiM=max(8, int(chi * rng.uniform(0.7, 1.2))),
                    chiR=max(8, int(chi * rng.uniform(0.7, 1.2))), d=rng.choice([2, 3]))
    if op == "mlp_train":
        return dict(op="mlp_train", rows=_logint(rng, 1000, 60000), d=rng.choice([2, 3]))
    return dict(op="dmrg", lx=rng.choice([4, 5]), ly=4, maxdim=rng.choice([40, 60, 80, 100]),
                cutoff=1e-9)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *dims, dtype=F64):
    return torch.randn(*dims, generator=g, device="cuda", dtype=dtype)


def _flat(x):
    """Column-major flat buffer of a tensor (first index fastest)."""
    return x.permute(*reversed(range(x.dim()))).contiguous().reshape(-1)


def _fields(n, seed):
    return np.random.RandomState(int(seed) % (2 ** 31)).uniform(-0.5, 0.5, n)


def _bond(case, g):
    """A two-site tensor phi(a, s1, s2, b) with a decaying Schmidt spectrum:
    Gaussian factors around exp(-decay i / r)."""
    m, n = case["chiL"] * case["d"], case["d"] * case["chiR"]
    r = min(m, n)
    s = torch.exp(-case["decay"] * torch.arange(r, device="cuda", dtype=F64) / r)
    phi = (_randn(g, m, r) * s) @ _randn(g, n, r).t().contiguous()
    phi /= phi.norm()
    return phi.reshape(case["d"], case["chiL"], n).permute(1, 0, 2) \
        .reshape(case["chiL"], case["d"], case["chiR"], case["d"]).permute(0, 1, 3, 2)


def _heff_inputs(case, g, dtype, hermitian):
    w, d, cl, cr = case["w"], case["d"], case["chiL"], case["chiR"]
    L, R = _randn(g, cl, w, cl, dtype=dtype), _randn(g, cr, w, cr, dtype=dtype)
    W1, W2 = _randn(g, w, w, d, d, dtype=dtype), _randn(g, w, w, d, d, dtype=dtype)
    psi = _randn(g, cl, d, d, cr, dtype=dtype)
    if hermitian:
        # environments of a Hermitian operator, scaled to a spectrum of O(1)
        L = (L + L.permute(2, 1, 0)) / math.sqrt(2.0 * cl)
        R = (R + R.permute(2, 1, 0)) / math.sqrt(2.0 * cr)
        W1 = (W1 + W1.permute(0, 1, 3, 2)) / (2.0 * w)
        W2 = (W2 + W2.permute(0, 1, 3, 2)) / (2.0 * w)
    return L, W1, W2, R, psi


def _mlp_dims(case):
    return 3 * case["d"] ** 2, 256, case["d"] ** 2


def _mlp_inputs(case, g):
    i, h, o = _mlp_dims(case)
    n = h * i + h + h * h + h + o * h + o
    P = _randn(g, n, dtype=F32)
    off = 0
    for size, scale in ((h * i, i ** -0.5), (h, 0.1), (h * h, h ** -0.5), (h, 0.1),
                        (o * h, h ** -0.5), (o, 0.1)):
        P[off:off + size] *= scale
        off += size
    rows = case["rows"]
    X, T = _randn(g, rows, i, dtype=F32), _randn(g, rows, o, dtype=F32)
    # Adam's moments part way through a training run
    m = 1e-3 * _randn(g, n, dtype=F32)
    v = 1e-6 * (0.5 + torch.rand(n, generator=g, device="cuda", dtype=F32))
    return P, X, T, m, v


def _dims6(case):
    w = case["w"]
    return (case["chiL"], w, w, w, case["d"], case["chiR"])


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    from itg import _lib, itensor, mps, ops
    _lib.ctx()      # the library's stream becomes torch's current one
    g = _gen(seed)
    op = case["op"]
    if op == "heff":
        L, W1, W2, R, psi = [_flat(x) for x in _heff_inputs(
            case, g, getattr(torch, case["dtype"]), False)]
        dims = _dims6(case)
        return dict(op=op, L=L, R=R, psi=psi, dims=dims, mode=case["mode"],
                    prep=ops.heff2_prepare(L, W1, W2, R, *dims, mode=case["mode"]),
                    work=ops.heff2_work(*dims))
    if op == "davidson":
        L, W1, W2, R, psi = [_flat(x) for x in _heff_inputs(case, g, F64, True)]
        dims = _dims6(case)
        return dict(op=op, L=L, R=R, psi=psi, dims=dims, maxiter=case["maxiter"],
                    prep=ops.heff2_prepare(L, W1, W2, R, *dims),
                    work=ops.heff2_work(*dims),
                    kwork=ops.davidson2_work(case["chiL"], case["d"], case["chiR"],
                                             case["maxiter"]))
    if op == "factorize" or op == "svd":
        ind = [itensor.Index(x) for x in (case["chiL"], case["d"], case["d"], case["chiR"])]
        if op == "svd":
            phi = _randn(g, *[i.dim for i in ind])
        else:
            phi = _bond(case, g)
        return dict(op=op, phi=itensor.ITensor(ind, _flat(phi)), left=ind[:2], case=case)
    if op == "qr":
        ind = [itensor.Index(x) for x in (case["chiL"], case["d"], case["chiR"])]
        A = _randn(g, *[i.dim for i in ind])
        return dict(op=op, A=itensor.ITensor(ind, _flat(A)), left=ind[:2])
    if op == "contract":
        a, b, c, e, k1, k2 = [itensor.Index(case[n]) for n in ("a", "b", "c", "e", "k1", "k2")]
        A, B = _contract_inputs(case, g)
        return dict(op=op, A=itensor.ITensor((a, k1, b, k2), _flat(A)),
                    B=itensor.ITensor((k2, c, k1, e), _flat(B)))
    if op == "gate":
        l, m, r = [itensor.Index(case[n]) for n in ("chiL", "chiM", "chiR")]
        s1, s2 = itensor.Index(case["d"]), itensor.Index(case["d"])
        A, B, G = _gate_inputs(case, g)
        return dict(op=op, A=itensor.ITensor((l, s1, m), _flat(A)),
                    B=itensor.ITensor((m, s2, r), _flat(B)),
                    G=itensor.ITensor((s1.prime(), s2.prime(), s1, s2), _flat(G)),
                    order=(l, s1.prime(), s2.prime(), r))
    if op == "mlp_train":
        i, h, o = _mlp_dims(case)
        P, X, T, m, v = _mlp_inputs(case, g)
        return dict(op=op, P=P, X=X, T=T, m=m, v=v, rows=case["rows"], dims=(i, h, o),
                    Y=ops.empty(case["rows"] * o, "float32"),
                    acts=ops.empty(4 * case["rows"] * h, "float32"),
                    G=ops.empty(P.numel(), "float32"))
    # dmrg: a state converged at the case's own truncation
    N = case["lx"] * case["ly"]
    terms = mps.heisenberg_opsum(mps.cylinder_bonds(case["lx"], case["ly"]))
    for j, f in enumerate(_fields(N, seed)):
        terms.add(float(f), "Sz", j)
        terms.add(0.3 * float(f) + 0.2, "Sx", j)
    H = mps.MPO.from_opsum(terms, N)
    psi = mps.random_mps(N, 2, 10, int(seed))
    md = case["maxdim"]
    mps.dmrg(H, psi, mps.Sweeps(6, maxdim=[16, 32, md, md, md, md], cutoff=[case["cutoff"]]))
    return dict(op=op, H=H, psi=psi, maxdim=md, cutoff=case["cutoff"])


def _contract_inputs(case, g):
    dt = getattr(torch, case["dtype"])
    return (_randn(g, case["a"], case["k1"], case["b"], case["k2"], dtype=dt),
            _randn(g, case["k2"], case["c"], case["k1"], case["e"], dtype=dt))


def _gate_inputs(case, g):
    d = case["d"]
    A = _randn(g, case["chiL"], d, case["chiM"], dtype=C128)
    B = _randn(g, case["chiM"], d, case["chiR"], dtype=C128)
    # a near-identity gate, as one Trotter step is
    G = torch.eye(d * d, device="cuda", dtype=C128) + 0.05 * _randn(g, d * d, d * d, dtype=C128)
    return A, B, G.reshape(d, d, d, d)


# ---------------------------------------------------------------------- run
def run(s):
    from itg import itensor, mps, ops
    op = s["op"]
    if op == "heff":
        return ops.heff2_apply_prepared(s["L"], s["R"], s["prep"], s["psi"], *s["dims"],
                                        mode=s["mode"], work=s["work"])
    if op == "davidson":
        phi = ops.copy(s["psi"])        # overwritten with the Ritz vector
        e, n = ops.davidson2(s["L"], s["R"], s["prep"], phi, *s["dims"], maxiter=s["maxiter"],
                             work=s["work"], kwork=s["kwork"])
        return {"energy": e, "matvecs": n, "phi": phi}
    if op == "factorize":
        c = s["case"]
        A, B, spec = itensor.factorize(s["phi"], s["left"], ortho=c["ortho"], maxdim=c["maxdim"],
                                       cutoff=c["cutoff"])
        T = A * B
        if list(T.inds) != list(s["phi"].inds):
            T = T.permute(*s["phi"].inds)
        return {"spectrum": np.asarray(spec.eigs), "theta": T.data}
    if op == "svd":
        c = s["case"]
        U, S, V, spec = itensor.svd(s["phi"], s["left"], maxdim=c["maxdim"], cutoff=c["cutoff"])
        return {"spectrum": np.asarray(spec.eigs), "theta": (U * S * V).data}
    if op == "qr":
        Q, R = itensor.qr(s["A"], s["left"])
        return {"Q": Q.data, "R": R.data}
    if op == "contract":
        return (s["A"] * s["B"]).data
    if op == "gate":
        return (s["G"] * (s["A"] * s["B"])).permute(*s["order"]).data
    if op == "mlp_train":
        i, h, o = s["dims"]
        Y, acts = ops.mlp_forward(s["P"], s["X"], s["rows"], i, h, o, Y=s["Y"], acts=s["acts"])
        G, loss = ops.mlp_backward(s["P"], s["X"], s["T"], acts, Y, s["rows"], i, h, o, G=s["G"])
        P = ops.copy(s["P"])
        m, v = ops.copy(s["m"]), ops.copy(s["v"])
        ops.mlp_adam(P, G, m, v, step=100, lr=3e-4)
        return {"Y": Y, "grad": G, "loss": loss, "params": P, "m": m, "v": v}
    psi = mps.MPS([ops.copy(t) for t in s["psi"].data], s["psi"].dims, s["psi"].llim,
                  s["psi"].rlim)
    energy = mps.dmrg(s["H"], psi, mps.Sweeps(1, maxdim=[s["maxdim"]], cutoff=[s["cutoff"]]))
    # the two-site reduced density matrix at the orthogonality centre
    th, td = ops.contract(psi.data[0], psi.dims[0], [1, 2, 3], psi.data[1], psi.dims[1],
                          [3, 4, 5], [1, 2, 4, 5])
    rho, _ = ops.contract(th, td, [1, 2, 4, 5], th, td, [1, 6, 7, 5], [2, 4, 6, 7])
    return {"energy": energy, "rho": rho}


# --------------------------------------------------------------------- work
def work(case):
    op = case["op"]
    if op in ("heff", "davidson"):
        w, d, cl, cr = case["w"], case["d"], case["chiL"], case["chiR"]
        es = 4 if case.get("dtype") == "float32" else 8
        applies = 1 if op == "heff" else case["maxiter"] + 1
        flops = applies * (2.0 * w * d * d * cl * cr * (cl + cr) + 2.0 * (w * d * d) ** 2 * cl * cr)
        return {"bytes": es * (w * (cl * cl + cr * cr) + 2.0 * d * d * cl * cr), "flops": flops}
    if op in ("factorize", "svd"):
        m, n = case["chiL"] * case["d"], case["d"] * case["chiR"]
        # the side that is diagonalised, its reduction and kept vectors
        q = min(m, n) if op == "svd" else (m if case["ortho"] == "left" else n)
        k = min(case["maxdim"], m, n)
        flops = 1.0 * m * n * q + 4.0 / 3.0 * q ** 3 + 2.0 * q * q * k + 2.0 * m * n * k * 2
        return {"bytes": 8.0 * 2 * m * n, "flops": flops}
    if op == "qr":
        m, n = case["chiL"] * case["d"], case["chiR"]
        r = min(m, n)
        return {"bytes": 8.0 * (m * n + m * r + r * n),
                "flops": 2.0 * (2.0 * m * n * r - (m + n) * r * r + 2.0 * r ** 3 / 3.0)}
    if op == "contract":
        es = 4 if case["dtype"] == "float32" else 8
        M, N, K = case["a"] * case["b"], case["c"] * case["e"], case["k1"] * case["k2"]
        return {"bytes": es * (M * K + K * N + M * N), "flops": 2.0 * M * N * K}
    if op == "gate":
        d, l, m, r = case["d"], case["chiL"], case["chiM"], case["chiR"]
        return {"bytes": 16.0 * (l * d * m + m * d * r + l * d * d * r),
                "flops": 8.0 * (l * d * d * r * m + d ** 4 * l * r)}
    if op == "mlp_train":
        i, h, o = _mlp_dims(case)
        n = h * i + h * h + h * o
        return {"bytes": 4.0 * (case["rows"] * (i + 2 * o) + 7 * n),
                "flops": 2.0 * case["rows"] * (3 * n - h * i)}
    # dmrg: two passes over the bonds, three Heff applies and one density
    # matrix each, on average at three quarters of the kept states
    n, chi, w = case["lx"] * case["ly"], 0.75 * case["maxdim"], 14
    bond = 3 * (16.0 * w * chi ** 3 + 32.0 * w * w * chi ** 2) + 8 * chi ** 3 * (2 + 4 / 3 + 2)
    return {"bytes": 2 * n * 8.0 * (2 * w * chi * chi + 8 * chi * chi), "flops": 2 * n * bond}


# -------------------------------------------------------------------- exact
def _heff_ref(L, W1, W2, R, x):
    cl, d, _, cr = x.shape
    w = L.shape[1]
    T = L.reshape(cl * w, cl) @ x.reshape(cl, d * d * cr)            # a' wl | s1 s2 b
    T = T.reshape(cl, w, d, d, cr)
    X = torch.tensordot(W1, W2, dims=([1], [0]))                     # wl s1' s1 wr s2' s2
    T = torch.tensordot(T, X, dims=([1, 2, 3], [0, 2, 5]))           # a' b s1' wr s2'
    T = T.permute(0, 2, 4, 3, 1).reshape(cl * d * d, -1)             # a' s1' s2' | wr b
    return (T @ R.permute(1, 2, 0).reshape(-1, cr)).reshape(cl, d, d, cr)


def _kept(w, maxdim, cutoff):
    """NDTensors' truncate: at most maxdim, then the smallest weights while
    their sum stays within cutoff of the total."""
    w = np.maximum(w, 0.0)
    total = w.sum()
    n = len(w)
    err = 0.0
    while n > maxdim:
        n -= 1
        err += w[n]
    while n > 1 and err + w[n - 1] <= cutoff * total:
        n -= 1
        err += w[n]
    return n


def exact(case, seed):
    g = _gen(seed)
    op = case["op"]
    if op == "heff":
        L, W1, W2, R, psi = [x.double() for x in _heff_inputs(
            case, g, getattr(torch, case["dtype"]), False)]
        return _flat(_heff_ref(L, W1, W2, R, psi))
    if op == "davidson":
        L, W1, W2, R, psi = _heff_inputs(case, g, F64, True)
        V = [psi / psi.norm()]
        AV = [_heff_ref(L, W1, W2, R, V[0])]
        lam = float((V[0] * AV[0]).sum())
        phi, q = V[0], AV[0] - lam * V[0]
        for _ in range(case["maxiter"]):
            t = q
            for _ in range(2):
                for v in V:
                    t = t - (v * t).sum() * v
            V.append(t / t.norm())
            AV.append(_heff_ref(L, W1, W2, R, V[-1]))
            M = np.array([[float((a * b).sum()) for b in AV] for a in V])
            ev, U = np.linalg.eigh(0.5 * (M + M.T))
            u = U[:, 0] if U[0, 0] >= 0 else -U[:, 0]
            lam = float(ev[0])
            phi = sum(float(c) * v for c, v in zip(u, V))
            q = sum(float(c) * v for c, v in zip(u, AV)) - lam * phi
        return {"energy": lam, "matvecs": None, "phi": _flat(phi / phi.norm())}
    if op in ("factorize", "svd"):
        cl, d, cr = case["chiL"], case["d"], case["chiR"]
        phi = _bond(case, g) if op == "factorize" else _randn(g, cl, d, d, cr)
        # (a s1) x (s2 b) in column-major order
        M = np.ascontiguousarray(_flat(phi).reshape(cr * d, d * cl).t().cpu().numpy())
        if op == "svd":
            U, s, Vt = np.linalg.svd(M, full_matrices=False)
            k = _kept(s ** 2, case["maxdim"], case["cutoff"])
            spec, T = s[:k] ** 2, (U[:, :k] * s[:k]) @ Vt[:k]
        else:
            rho = M @ M.T if case["ortho"] == "left" else M.T @ M
            w, U = np.linalg.eigh(rho)
            w, U = w[::-1], U[:, ::-1]
            k = _kept(w, case["maxdim"], case["cutoff"])
            U, spec = np.ascontiguousarray(U[:, :k]), w[:k]
            T = U @ (U.T @ M) if case["ortho"] == "left" else (M @ U) @ U.T
        return {"spectrum": np.ascontiguousarray(spec), "theta": np.ravel(T, order="F")}
    if op == "qr":
        cl, d, cr = case["chiL"], case["d"], case["chiR"]
        A = _flat(_randn(g, cl, d, cr)).reshape(cr, d * cl).t().cpu().numpy()
        Q, R = np.linalg.qr(A)
        return {"Q": np.ravel(Q, order="F"), "R": np.ravel(R, order="F")}
    if op == "contract":
        A, B = [x.double() for x in _contract_inputs(case, g)]
        M, N, K = case["a"] * case["b"], case["c"] * case["e"], case["k1"] * case["k2"]
        C = A.permute(0, 2, 1, 3).reshape(M, K) @ B.permute(2, 0, 1, 3).reshape(K, N)
        return _flat(C.reshape(case["a"], case["b"], case["c"], case["e"]))
    if op == "gate":
        A, B, G = _gate_inputs(case, g)
        l, d, m = A.shape
        T = (A.reshape(l * d, m) @ B.reshape(m, -1)).reshape(l, d, d, -1)
        return _flat(torch.tensordot(G, T, dims=([2, 3], [1, 2])).permute(2, 0, 1, 3))
    if op == "mlp_train":
        i, h, o = _mlp_dims(case)
        P, X, T, m, v = [x.double() for x in _mlp_inputs(case, g)]
        P.requires_grad_(True)
        W1, b1, W2, b2, W3, b3 = P.split([h * i, h, h * h, h, o * h, o])
        gelu = torch.nn.functional.gelu
        A = gelu(X @ W1.reshape(h, i).t() + b1)
        A = gelu(A @ W2.reshape(h, h).t() + b2)
        Y = A @ W3.reshape(o, h).t() + b3
        loss = ((Y - T) ** 2).mean()
        G, = torch.autograd.grad(loss, P)
        m, v = 0.9 * m + 0.1 * G, 0.999 * v + 0.001 * G * G
        Pn = P.detach() - 3e-4 * (m / (1 - 0.9 ** 100)) / ((v / (1 - 0.999 ** 100)).sqrt() + 1e-8)
        return {"Y": Y.detach().reshape(-1), "grad": G, "loss": float(loss), "params": Pn, "m": m,
                "v": v}
    return None
