"""Measured cases: what programs have this package do on one GPU.

A case is one call that a user's program repeats: a solver that it keeps
(built once per system) and a run of it over a time list with expectation
values (and, for the larger ones, the final state), or one product of the data
layer.  The listed cases stand for nine families; ``draw`` takes any of them
over its whole range of sizes.

* ``me_jc``      mesolve of a Jaynes-Cummings cavity (N levels and a qubit,
                 superoperator of (2 N)^2 rows): the small and ordinary
                 single solves, where latency and launches count.  N = 10 is
                 the textbook problem, N = 23 an odd one of ordinary size.
* ``me_ising``   mesolve of a dissipative spin chain (superoperator of 4^L
                 rows): the large sparse solve.
* ``se_ising``   sesolve of a closed chain (2^L rows), two-site quadratic
                 forms and the final state.
* ``me_driven``  the chain with a cosine drive (QuTiP's list form).
* ``me_kerr``    mesolve of a driven Kerr oscillator in matrix form with the
                 default precision (banded operators, FP64): stiff, many
                 steps between outputs.
* ``me_dense``   matrix form with dense collapse operators (a random sparse
                 H and random density matrices): the requests of a solve
                 server, complex64 products.
* ``mc_ising``   mcsolve of the chain, all trajectories of a seed list, in
                 complex128 and complex64.
* ``sde``        ssesolve / smesolve of a monitored, driven cavity.
* ``product``    one operator-block product of the data layer (the plain
                 drop-in's right-hand side): L of the chain times a block of
                 columns on the device.

Inputs depend on the seed: couplings, fields, initial states, random
operators and trajectory seeds.
"""
import math

import numpy as np
import torch

import qutip_amd as qa
from qutip_amd import data as qd

# options of the reference's accuracy (1e-8 / 1e-10), as the solve server's
TIGHT = {"rtol": 1e-8, "atol": 1e-10}
FINAL = {**TIGHT, "store_final_state": True}


def listed():
    return [
        # one small solve, alone: the launch and latency end
        {"name": "me_jc_n10", "kind": "me_jc", "N": 10, "tf": 25.0, "npts": 100},
        # an ordinary solve of an odd size (2116 rows)
        {"name": "me_jc_n23", "kind": "me_jc", "N": 23, "tf": 10.0, "npts": 50},
        # the large sparse master equation (65536 rows), dense output times
        {"name": "me_ising_8", "kind": "me_ising", "L": 8, "tf": 10.0, "npts": 200},
        # a closed chain of 14 spins
        {"name": "se_ising_14", "kind": "se_ising", "L": 14, "tf": 5.0, "npts": 51},
        # a driven open chain of 6 spins (4096 rows)
        {"name": "me_driven_6", "kind": "me_driven", "L": 6, "tf": 5.0, "npts": 51},
        # a stiff banded problem: many steps, few outputs
        {"name": "me_kerr_n256", "kind": "me_kerr", "N": 256, "tf": 2.0, "npts": 11},
        # the middle and the largest request of a solve server
        {"name": "me_dense_d128", "kind": "me_dense", "d": 128, "nc": 2, "tf": 10.0, "npts": 50},
        {"name": "me_dense_d512", "kind": "me_dense", "d": 512, "nc": 3, "tf": 1.0, "npts": 6},
        # a full ensemble of 10 spins, and a complex64 one of 8
        {"name": "mc_ising_10", "kind": "mc_ising", "L": 10, "ntraj": 2048, "tf": 20.0,
         "npts": 100, "fp32": False},
        {"name": "mc_ising_8_c64", "kind": "mc_ising", "L": 8, "ntraj": 500, "tf": 10.0,
         "npts": 50, "fp32": True},
        # a monitored cavity of 20 levels (400 rows), an ensemble of 256
        {"name": "sme_cavity_20", "kind": "sde", "open": True, "d": 20, "ntraj": 256,
         "steps": 500, "npts": 26},
        # one product with an odd block of columns
        {"name": "product_8x5", "kind": "product", "L": 8, "cols": 5},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any family, sizes spread over its range.  The products
    of sizes and times stay below the largest listed ones."""
    kind = rng.choice(["me_jc", "me_jc", "me_ising", "se_ising", "me_driven", "me_kerr",
                       "me_dense", "me_dense", "mc_ising", "sde", "product"])
    c = {"kind": kind}
    if kind == "me_jc":
        c.update(N=_logint(rng, 2, 44), tf=round(rng.uniform(3.0, 25.0), 2),
                 npts=_logint(rng, 11, 200))
    elif kind == "me_ising":
        c.update(L=rng.randint(4, 8), tf=round(rng.uniform(2.0, 10.0), 2),
                 npts=_logint(rng, 11, 200))
    elif kind == "se_ising":
        c.update(L=rng.randint(7, 17), tf=round(rng.uniform(1.0, 8.0), 2),
                 npts=_logint(rng, 6, 150))
    elif kind == "me_driven":
        c.update(L=rng.randint(3, 7), tf=round(rng.uniform(1.0, 8.0), 2),
                 npts=_logint(rng, 6, 120))
    elif kind == "me_kerr":
        c.update(N=_logint(rng, 16, 256), tf=round(rng.uniform(0.5, 2.0), 2),
                 npts=_logint(rng, 3, 60))
    elif kind == "me_dense":
        d = 16 * _logint(rng, 1, 32)
        c.update(d=d, nc=rng.randint(1, 4), npts=_logint(rng, 3, 50),
                 tf=round(rng.uniform(0.5, 10.0) * min(1.0, 128.0 / d), 2))
    elif kind == "mc_ising":
        c.update(L=rng.randint(3, 10), ntraj=_logint(rng, 32, 1024),
                 tf=round(rng.uniform(2.0, 12.0), 2), npts=_logint(rng, 6, 100),
                 fp32=rng.random() < 0.4)
    elif kind == "sde":
        op = rng.random() < 0.5
        c.update(open=op, d=_logint(rng, 2, 31) if op else _logint(rng, 2, 900),
                 ntraj=_logint(rng, 16, 256), steps=_logint(rng, 20, 400),
                 npts=_logint(rng, 2, 20))
    else:
        c.update(L=rng.randint(3, 9), cols=_logint(rng, 1, 16))
        if c["L"] == 9:
            c["cols"] = min(c["cols"], 4)
    return c


# ---- the systems, as numbers (shared by prepare and exact) -------------------
def _numbers(case, seed):
    """The random numbers of a case: couplings, fields, seeds."""
    rng = np.random.default_rng([seed, 20240229])
    k = case["kind"]
    if k == "me_jc":
        v = rng.normal(size=4)
        return {"g": 0.05 * 2 * np.pi * rng.uniform(0.8, 1.2), "det": rng.uniform(-0.3, 0.3),
                "psi": (v[:2] + 1j * v[2:]) / np.linalg.norm(v)}
    if k in ("me_ising", "se_ising", "me_driven", "mc_ising", "product"):
        out = {"h": rng.uniform(0.5, 1.5, case["L"]), "w": rng.uniform(0.8, 1.2),
               "tilt": rng.uniform(0.0, 0.3), "seed": int(rng.integers(2 ** 31))}
        if k == "product":
            n = 4 ** case["L"]
            v = rng.normal(size=(2, n, case["cols"]))
            out["x"] = v[0] + 1j * v[1]
        return out
    if k == "me_kerr":
        return {"delta": rng.uniform(0.4, 0.6), "F": rng.uniform(1.5, 2.5)}
    if k == "me_dense":
        d = case["d"]
        num = max(int(0.05 * d * d), 1)
        M = np.zeros((d, d), dtype=np.complex128)
        at = rng.choice(d * d, num, replace=False)
        M.ravel()[at] = rng.uniform(-1, 1, num) + 1j * rng.uniform(-1, 1, num)
        H = 0.5 * (M + M.conj().T)
        cs = []
        for _ in range(case["nc"]):
            g = rng.normal(size=(2, d, d))
            X = g[0] + 1j * g[1]
            r = X @ X.conj().T
            cs.append(np.sqrt(rng.uniform(0.01, 0.1)) * r / np.trace(r).real)
        v = rng.normal(size=(2, d))
        return {"H": H, "c": cs, "psi": (v[0] + 1j * v[1]) / np.linalg.norm(v)}
    # sde
    v = rng.normal(size=4)
    return {"F": rng.uniform(0.3, 0.6), "delta": rng.uniform(-0.3, 0.3),
            "seed": int(rng.integers(2 ** 31)),
            "psi": (v[:2] + 1j * v[2:]) / np.linalg.norm(v)}


JC_RATES = (0.005, 0.05)


def _ising_gamma(case):
    return 0.05 if case["kind"] == "mc_ising" else 0.1


def _tlist(case):
    if case["kind"] == "sde":
        return np.linspace(0.0, SDE_DT * case["steps"], case["npts"])
    return np.linspace(0.0, case["tf"], case["npts"])


SDE_DT = 0.002


# ---- prepare -----------------------------------------------------------------
def _site(op, i, L):
    return qa.tensor([op if j == i else qa.qeye(2) for j in range(L)])


def _ising(case, p):
    L = case["L"]
    sz = [_site(qa.sigmaz(), i, L) for i in range(L)]
    sx = [_site(qa.sigmax(), i, L) for i in range(L)]
    H, X, mz = 0, 0, 0
    for i in range(L - 1):
        H = H + sz[i] @ sz[i + 1]
    for i in range(L):
        X = X + p["h"][i] * sx[i]
        mz = mz + sz[i]
    cops = [np.sqrt(_ising_gamma(case)) * _site(qa.sigmam(), i, L) for i in range(L)]
    one = qa.Qobj(np.array([[math.cos(p["tilt"])], [math.sin(p["tilt"])]]))
    psi = qa.tensor([one] * L)
    herm = [qa.Qobj(O, isherm=True) for O in (mz * (1.0 / L), sz[0] @ sz[1])]
    return H, X, cops, psi, herm


class _View:
    """A device array of the package as torch sees it, without a copy."""

    def __init__(self, dense):
        self.dense = dense
        m, n = dense.shape
        self.__cuda_array_interface__ = {
            "shape": (n, m), "typestr": "<c16", "data": (dense.ptr, False), "version": 2}


def prepare(case, seed):
    p = _numbers(case, seed)
    k = case["kind"]
    if k == "product":
        _, X, cops, _, _ = _ising(case, p)
        H = X
        for i in range(case["L"] - 1):
            H = H + _site(qa.sigmaz(), i, case["L"]) @ _site(qa.sigmaz(), i + 1, case["L"])
        return {"kind": k, "A": qd.HipCSR(qa.liouvillian(H, cops).to_csr()),
                "x": qd.HipDense.from_array(p["x"])}
    st = {"kind": k, "tlist": _tlist(case)}
    if k == "me_jc":
        N = case["N"]
        a = qa.tensor(qa.destroy(N), qa.qeye(2))
        sm = qa.tensor(qa.qeye(N), qa.sigmam())
        sz = qa.tensor(qa.qeye(N), qa.sigmaz())
        wq = 2 * np.pi
        H = ((wq + p["det"]) * a.dag() @ a + wq * 0.5 * sz
             + p["g"] * (a @ sm.dag() + a.dag() @ sm))
        cops = [np.sqrt(JC_RATES[0]) * a, np.sqrt(JC_RATES[1]) * sm]
        st.update(solver=qa.MESolver(H, cops, options=TIGHT), e_ops=[a.dag() @ a, sz],
                  psi=qa.tensor(qa.basis(N, 0), qa.Qobj(p["psi"].reshape(2, 1))))
    elif k == "me_ising":
        H, X, cops, psi, e = _ising(case, p)
        st.update(solver=qa.MESolver(H + X, cops, options=FINAL), e_ops=e, psi=psi)
    elif k == "se_ising":
        H, X, _, psi, e = _ising(case, p)
        st.update(solver=qa.SESolver(H + X, options=FINAL), e_ops=e, psi=psi)
    elif k == "me_driven":
        H, X, cops, psi, e = _ising(case, p)
        Ht = qa.QobjEvo([H, [X, "cos(w * t)"]], args={"w": p["w"]})
        st.update(solver=qa.MESolver(Ht, cops, options=FINAL), e_ops=e, psi=psi)
    elif k == "me_kerr":
        a = qa.destroy(case["N"])
        H = (p["delta"] * a.dag() @ a + 0.05 * a.dag() @ a.dag() @ a @ a
             + p["F"] * (a + a.dag()))
        par = qa.Qobj(np.diag((-1.0) ** np.arange(case["N"])))
        st.update(solver=qa.MESolver(H, [a], options={**FINAL, "matrix_form": True,
                                                      "nsteps": 100000}),
                  e_ops=[a.dag() @ a, par], psi=qa.basis(case["N"], 0))
    elif k == "me_dense":
        d = case["d"]
        proj = qa.basis(d, 0) @ qa.basis(d, 0).dag()
        st.update(solver=qa.MESolver(qa.Qobj(p["H"]), [qa.Qobj(c) for c in p["c"]],
                                     options={**FINAL, "matrix_form": True, "nsteps": 100000}),
                  e_ops=[proj, qa.num(d) * (1.0 / d)], psi=qa.Qobj(p["psi"]))
    elif k == "mc_ising":
        H, X, cops, psi, e = _ising(case, p)
        st.update(solver=qa.MCSolver(H + X, cops, options={
            "precision": "fp32" if case["fp32"] else "fp64", "keep_runs_results": True}),
            e_ops=e, psi=psi, ntraj=case["ntraj"], seed=p["seed"])
    else:
        d = case["d"]
        a = qa.destroy(d)
        H = p["delta"] * a.dag() @ a + p["F"] * (a + a.dag())
        opts = {"dt": SDE_DT, "keep_runs_results": True}
        if case["open"]:
            solver = qa.SMESolver(H, [0.5 ** 0.5 * a], c_ops=[0.1 ** 0.5 * a], options=opts)
        else:
            solver = qa.SSESolver(H, [0.5 ** 0.5 * a], options=opts)
        psi = np.zeros(d, dtype=np.complex128)
        psi[:2] = p["psi"]
        st.update(solver=solver, e_ops=[a.dag() @ a, a + a.dag()], psi=qa.Qobj(psi),
                  ntraj=case["ntraj"], seed=p["seed"])
    return st


def run(st):
    k = st["kind"]
    if k == "product":
        out = qd.matmul(st["A"], st["x"])
        return torch.as_tensor(_View(out), device="cuda")
    if k in ("mc_ising", "sde"):
        res = st["solver"].run(st["psi"], st["tlist"], st["ntraj"], e_ops=st["e_ops"],
                               seeds=st["seed"])
        out = {"average": res.average_expect, "std": res.std_expect, "runs": res.runs_expect}
        if k == "mc_ising":
            out["jumps"] = np.asarray(res.num_jumps)
        return out
    res = st["solver"].run(st["psi"], st["tlist"], e_ops=st["e_ops"])
    out = {"expect": [np.asarray(v) for v in res.expect]}
    if res.final_state is not None:
        out["final"] = res.final_state.full()
    return out


# ---- work --------------------------------------------------------------------
# Right-hand sides per unit of time (vern7 at the cases' tolerances, from the
# solvers' own counts): 10 per attempt and 6 per dense output.
def _rhs_count(case):
    k = case["kind"]
    rate = {"me_jc": 156.0 * (case.get("N", 10) / 10.0) ** -0.05, "me_ising": 123.0,
            "se_ising": 426.0, "me_driven": 186.0,
            "me_kerr": 3900.0 * (case.get("N", 256) / 256.0) ** 2,
            "me_dense": 11.0 * case.get("d", 128) ** 0.5}[k]
    return rate * case["tf"] + 6.0 * case["npts"]


def work(case):
    """Operators, states and outputs once; the complex multiply-adds of the
    right-hand sides that the tolerances need (8 flops each)."""
    k = case["kind"]
    if k == "product":
        L, m = case["L"], case["cols"]
        n = 4 ** L
        nnz = n * (2 * L + 1) + L * 4 ** (L - 1)
        return {"bytes": nnz * 20 + 4 * n + 32 * n * m, "flops": 8 * nnz * m}
    if k == "mc_ising":
        L, b, s = case["L"], case["ntraj"], (8 if case["fp32"] else 16)
        d = 2 ** L
        nnz = d * (L + 1)
        attempts = 16.0 * case["tf"]
        rhs = 10 * attempts + 6 * case["npts"]
        return {"bytes": nnz * (s + 4) + 16 * d + 32 * b * case["npts"],
                "flops": 8.0 * nnz * rhs * b}
    if k == "sde":
        d = case["d"]
        n = d * d if case["open"] else d
        per = (2 * 8 + 2 * 2) * n if case["open"] else (2 * 4 + 4) * n
        return {"bytes": 20 * 8 * n + 8 * case["ntraj"] * (case["steps"] + 4 * case["npts"]),
                "flops": 8.0 * per * case["steps"] * case["ntraj"]}
    rhs = _rhs_count(case)
    if k == "me_dense":
        d, nc = case["d"], case["nc"]
        return {"bytes": 8 * d * d * (2 * nc + 2) + 32 * d * d + 32 * case["npts"],
                "flops": (1 + 1.5 * nc) * 8.0 * d ** 3 * rhs}
    if k == "me_kerr":
        n = case["N"] ** 2
        return {"bytes": 32 * n + 16 * 8 * case["N"] + 32 * case["npts"],
                "flops": 8.0 * 7 * n * rhs}
    if k == "me_jc":
        n = (2 * case["N"]) ** 2
        nnz = 7 * n
    elif k == "se_ising":
        n = 2 ** case["L"]
        nnz = n * (case["L"] + 1)
    else:
        n = 4 ** case["L"]
        nnz = n * (2 * case["L"] + 1) + case["L"] * 4 ** (case["L"] - 1)
    return {"bytes": 20 * nnz + 32 * n + 32 * case["npts"], "flops": 8.0 * nnz * rhs}


# ---- tolerance ---------------------------------------------------------------
def tolerance(case):
    """What another correct implementation shows: the integrators' truncation
    error at the stated tolerances (measured against 64-bit references), FP32
    products in me_dense, and in the ensembles a collapse time that the
    secant search may stop at elsewhere within its own tolerance (1e-4)."""
    k = case["kind"]
    if k == "product":
        return {"rel": 1e-15, "max": 1e-13}
    if k == "mc_ising":
        return ({"rel": 2e-4, "max": 0.05, "differ": 0.002} if case["fp32"]
                else {"rel": 1e-5, "max": 1e-2, "differ": 0.002})
    if k == "sde":
        return {"rel": 1e-10, "max": 1e-8}
    if k == "me_dense":
        return {"rel": 5e-6, "max": 5e-4}
    if k in ("me_ising", "me_driven"):
        return {"rel": 4e-7, "max": 2e-5}
    if k == "se_ising":
        return {"rel": 1e-7, "max": 1e-5}
    return {"rel": 2e-8, "max": 1e-6}


# ---- exact -------------------------------------------------------------------
DEV = "cuda" if torch.cuda.is_available() else "cpu"
C128 = torch.complex128


def _t(a):
    return torch.as_tensor(np.asarray(a, dtype=np.complex128), device=DEV)


def _lower(N):
    return np.diag(np.sqrt(np.arange(1, N)), 1).astype(np.complex128)


def _kron(ops):
    M = np.ones((1, 1), dtype=np.complex128)
    for o in ops:
        M = np.kron(M, o)
    return M


def _np_site(op, i, L):
    return np.kron(np.kron(np.eye(2 ** i), op), np.eye(2 ** (L - 1 - i)))


SZ = np.diag([1.0, -1.0]).astype(np.complex128)
SX = np.array([[0, 1], [1, 0]], dtype=np.complex128)
SM = np.array([[0, 0], [1, 0]], dtype=np.complex128)


def _ising_np(case, p):
    L = case["L"]
    d = 2 ** L
    bits = (np.arange(d)[:, None] >> np.arange(L - 1, -1, -1)) & 1
    z = 1.0 - 2.0 * bits  # [d, L]
    H = np.diag((z[:, :-1] * z[:, 1:]).sum(1)).astype(np.complex128)
    X = np.zeros((d, d), dtype=np.complex128)
    for i in range(L):
        X[np.arange(d), np.arange(d) ^ (1 << (L - 1 - i))] += p["h"][i]
    psi = _kron([np.array([[math.cos(p["tilt"])], [math.sin(p["tilt"])]])] * L).ravel()
    return H, X, psi, [np.diag(z.mean(1)), np.diag(z[:, 0] * z[:, 1])]


def _taylor(f, y, dt, norm, out):
    """y(k dt) for k = 1 .. out, dy/dt = f(y) linear with |f| <= norm."""
    sub = max(1, int(math.ceil(norm * dt / 6.0)))
    h = dt / sub
    order = int(30 + 2 * norm * h)
    ys = []
    for _ in range(out):
        for _ in range(sub):
            term = y
            acc = y.clone()
            for m in range(1, order):
                term = f(term) * (h / m)
                acc += term
            y = acc
        ys.append(y)
    return ys


def _gbs(f, y, t, dt, norm, out):
    """The same for dy/dt = f(t, y): Gragg's midpoint steps, extrapolated."""
    sub = max(1, int(math.ceil(norm * dt / 1.5)))
    h = dt / sub
    ns = [2, 4, 6, 8, 10, 12, 14]
    ys = []
    for _ in range(out):
        for _ in range(sub):
            T = []
            for j, n in enumerate(ns):
                g = h / n
                a, b = y, y + g * f(t, y)
                for m in range(1, n):
                    a, b = b, a + 2 * g * f(t + m * g, b)
                row = [0.5 * (a + b + g * f(t + h, b))]
                for q in range(j):
                    r = (n / ns[j - q - 1]) ** 2
                    row.append(row[q] + (row[q] - T[-1][q]) / (r - 1))
                T.append(row)
            y = T[-1][-1]
            t += h
        ys.append(y)
    return ys


def _span(H):
    e = np.linalg.eigvalsh(H)
    return float(e[-1] - e[0]), 0.5 * float(e[-1] + e[0])


def _expect(ys, ops, ket):
    out = []
    for O in ops:
        Ot = _t(O)
        v = []
        for y in ys:
            if ket:
                v.append((torch.vdot(y, Ot @ y) / torch.vdot(y, y)).real)
            else:
                v.append((torch.sum(Ot.T * y) / torch.trace(y)).real)
        out.append(torch.stack(v).cpu().numpy())
    return out


def _lindblad(H, cops, rho0, case, ops, X=None, w=0.0):
    """<O>(t) from dense matrices; X: driven by cos(w t)."""
    tl = _tlist(case)
    dt = tl[1] - tl[0]
    d = H.shape[0]
    nh = -0.5 * sum(c.conj().T @ c for c in cops)
    span, mid = _span(H if X is None else H + X)
    norm = span + 2 * np.linalg.norm(nh, 2) + sum(np.linalg.norm(c, 2) ** 2 for c in cops)
    M0 = _t(-1j * (H - (mid if X is None else 0.0) * np.eye(d)) + nh)
    Mx = None if X is None else _t(-1j * X)
    C = [_t(c) for c in cops]
    Cd = [c.conj().T.contiguous() for c in C]

    def f(r):
        a = M0 @ r
        k = a + a.conj().T
        for c, cd in zip(C, Cd):
            k = k + c @ (r @ cd)
        return k

    def ft(t, r):
        a = (M0 + math.cos(w * t) * Mx) @ r
        k = a + a.conj().T
        for c, cd in zip(C, Cd):
            k = k + c @ (r @ cd)
        return k

    y = _t(rho0)
    n = len(tl) - 1
    ys = _taylor(f, y, dt, norm, n) if X is None else _gbs(ft, y, 0.0, dt, norm, n)
    out = {"expect": _expect([y] + ys, ops, False)}
    if case["kind"] != "me_jc":
        out["final"] = (ys[-1] / torch.trace(ys[-1])).cpu().numpy()
    return out


def _sde_exact(case, p):
    """Platen's scheme for every trajectory at once, dense operators."""
    d, op, m = case["d"], case["open"], case["ntraj"]
    a = _lower(d)
    H = p["delta"] * a.conj().T @ a + p["F"] * (a + a.conj().T)
    sc = 0.5 ** 0.5 * a
    e_ops = [a.conj().T @ a, a + a.conj().T]
    tl = _tlist(case)
    t, counts = float(tl[0]), []
    for tk in tl[1:]:
        n, rest = divmod(tk - t, SDE_DT)
        n = 0 if tk - t < 0.5 * SDE_DT else int(n) + (1 if rest > 0.5 * SDE_DT else 0)
        counts.append(n)
        t += SDE_DT * n
    total = sum(counts)
    dW = np.stack([np.random.default_rng(s).normal(0, np.sqrt(SDE_DT), size=(total, 1, 1))[:, 0, 0]
                   for s in np.random.SeedSequence(p["seed"]).spawn(m)])
    dW = torch.as_tensor(dW, device=DEV)
    psi = np.zeros(d, dtype=np.complex128)
    psi[:2] = p["psi"]
    dt, sq = SDE_DT, math.sqrt(SDE_DT)
    if op:
        ex = 0.1 ** 0.5 * a
        M0 = _t(-1j * H - 0.5 * (sc.conj().T @ sc + ex.conj().T @ ex))
        S, E = _t(sc), _t(ex)
        Sd, Ed, Md = S.conj().T.contiguous(), E.conj().T.contiguous(), M0.conj().T.contiguous()
        x = _t(np.outer(psi, psi.conj())).repeat(m, 1, 1)

        def drift(r):
            return (torch.matmul(M0, r) + torch.matmul(r, Md)
                    + torch.matmul(torch.matmul(S, r), Sd)
                    + torch.matmul(torch.matmul(E, r), Ed))

        def diff(r):
            y = torch.matmul(S, r) + torch.matmul(r, Sd)
            return y - torch.diagonal(y, dim1=1, dim2=2).sum(1)[:, None, None] * r

        def col(w):
            return w[:, None, None]

        def ev(r):
            return [torch.sum(_t(O).T * r, dim=(1, 2)).real for O in e_ops]
    else:
        M0, S = _t((-1j * H - 0.5 * sc.conj().T @ sc).T), _t(sc.T)
        x = _t(psi).repeat(m, 1)

        def e_of(r, y):
            return 2 * torch.sum(r.conj() * y, dim=1).real[:, None]

        def drift(r):
            y = r @ S
            e = e_of(r, y)
            return r @ M0 + 0.5 * e * y - 0.125 * e * e * r

        def diff(r):
            y = r @ S
            return y - 0.5 * e_of(r, y) * r

        def col(w):
            return w[:, None]

        def ev(r):
            return [torch.sum(r.conj() * (r @ _t(O.T)), dim=1).real for O in e_ops]
    outs = [ev(x)]
    k = 0
    for n in counts:
        for _ in range(n):
            w = col(dW[:, k])
            k += 1
            d1 = x + dt * drift(x)
            b = diff(x)
            out = 0.5 * (d1 + x) + 0.5 * w * b + 0.5 * dt * drift(d1 + w * b)
            c2 = 0.25 / sq * (w * w - dt)
            x = (out + (0.25 * w + c2) * diff(d1 + sq * b) + (0.25 * w - c2) * diff(d1 - sq * b))
        outs.append(ev(x))
    runs = [torch.stack([o[j] for o in outs], dim=1).cpu().numpy() for j in range(2)]
    av = [v.sum(0) / m for v in runs]
    sd = [np.sqrt(np.abs((v ** 2).sum(0) / m - (v.sum(0) / m) ** 2)) for v in runs]
    return {"average": av, "std": sd, "runs": runs}


def exact(case, seed):
    k = case["kind"]
    p = _numbers(case, seed)
    if k == "mc_ising":
        return None  # the collapse times depend on where the search stops
    if k == "sde":
        return _sde_exact(case, p)
    if k == "me_jc":
        N = case["N"]
        a, sm, sz = np.kron(_lower(N), np.eye(2)), np.kron(np.eye(N), SM), np.kron(np.eye(N), SZ)
        wq = 2 * np.pi
        n = a.conj().T @ a
        H = (wq + p["det"]) * n + wq * 0.5 * sz + p["g"] * (a @ sm.conj().T + a.conj().T @ sm)
        psi = np.kron(np.eye(N)[0], p["psi"])
        return _lindblad(H, [np.sqrt(JC_RATES[0]) * a, np.sqrt(JC_RATES[1]) * sm],
                         np.outer(psi, psi.conj()), case, [n, sz])
    if k == "me_kerr":
        a = _lower(case["N"])
        ad = a.conj().T
        H = p["delta"] * ad @ a + 0.05 * ad @ ad @ a @ a + p["F"] * (a + ad)
        rho = np.zeros_like(H)
        rho[0, 0] = 1
        return _lindblad(H, [a], rho, case, [ad @ a, np.diag((-1.0) ** np.arange(case["N"]))])
    if k == "me_dense":
        d = case["d"]
        proj = np.zeros((d, d), dtype=np.complex128)
        proj[0, 0] = 1
        return _lindblad(p["H"], p["c"], np.outer(p["psi"], p["psi"].conj()), case,
                         [proj, np.diag(np.arange(d) / d)])
    if k == "se_ising":
        L = case["L"]
        dd = 2 ** L
        idx = torch.arange(dd, device=DEV)
        z = torch.stack([1.0 - 2.0 * ((idx >> (L - 1 - i)) & 1) for i in range(L)]).double()
        diag = (z[:-1] * z[1:]).sum(0)
        flips = [idx ^ (1 << (L - 1 - i)) for i in range(L)]

        def f(y):
            r = diag * y
            for i in range(L):
                r = r + float(p["h"][i]) * y[flips[i]]
            return -1j * r
        y = _t(_kron([np.array([[math.cos(p["tilt"])], [math.sin(p["tilt"])]])] * L).ravel())
        tl = _tlist(case)
        ys = [y] + _taylor(f, y, tl[1] - tl[0], L - 1 + p["h"].sum(), len(tl) - 1)
        e = [torch.stack([((o * v.abs() ** 2).sum() / (v.abs() ** 2).sum()).real
                          for v in ys]).cpu().numpy() for o in (z.mean(0), z[0] * z[1])]
        fin = ys[-1] / torch.linalg.vector_norm(ys[-1])
        return {"expect": e, "final": fin.cpu().numpy().reshape(-1, 1)}
    H, X, psi, ops = _ising_np(case, p)
    L = case["L"]
    cops = [np.sqrt(_ising_gamma(case)) * _np_site(SM, i, L) for i in range(L)]
    if k == "product":
        M0 = _t(-1j * (H + X) - 0.5 * sum(c.conj().T @ c for c in cops))
        C = [_t(c) for c in cops]
        out = []
        for q in range(case["cols"]):
            r = _t(p["x"][:, q].reshape(2 ** L, 2 ** L).T)  # vec stacks columns
            v = M0 @ r + r @ M0.conj().T
            for c in C:
                v = v + c @ r @ c.conj().T
            out.append(v.T.reshape(-1))
        return torch.stack(out)
    rho = np.outer(psi, psi.conj())
    if k == "me_driven":
        return _lindblad(H, cops, rho, case, ops, X=X, w=p["w"])
    return _lindblad(H + X, cops, rho, case, ops)
