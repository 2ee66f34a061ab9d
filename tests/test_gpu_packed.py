"""The packed operator form of the trajectory and whole-solve kernels against
the ELL form of the same kernels.

Same stages, same step control; only the order of the sums of a row's
products differs (the diagonal first, then by distance).  A right-hand side
of at most 17 products differs by 34 eps times the row's absolute sum, here
at most 6; times a step below 4 / 6 and 16 stages of a method whose weights
sum to at most 4 in absolute value, that is below 10^4 eps an attempt, and
the flow does not amplify it: tol = 10^4 eps attempts.  Sizes at the edges of
waves and of the two kernel forms (at most 512 rows and at most 256 systems,
or else), widths 0 to 16, imaginary and complex values.  In complex64 the
order is the same, so the bits are: there rounding alone could send a
trajectory to another jump."""
import numpy as np
import pytest
import scipy.sparse as sp

import qutip_amd as qa
from qutip_amd.solver import mcsolve as _mc  # noqa: F401  (the function shadows the module)
from qutip_amd.solver.small import SmallSolve
from qutip_amd.solver.tableaus import TABLEAUS
import sys

M = sys.modules["qutip_amd.solver.mcsolve"]


def _op(n, width, imag, seed=0):
    """Diagonal in the left half plane; `width` off-diagonal entries a row
    (fewer at the edges) with few distinct values, absolute row sum <= 6."""
    rng = np.random.default_rng(seed)
    vals = rng.uniform(-1, 1, 7) * 4.0 / max(width, 1)
    z = 1j * vals if imag else vals * np.exp(1j * rng.uniform(0, 2 * np.pi, 7))
    A = sp.diags(-1.0 - rng.uniform(0, 1, n) + 0j, 0).tolil()
    offs = rng.permutation(np.arange(1, 40))[:(width + 1) // 2]
    offs = np.concatenate([offs, -offs])[:width]
    A = sp.csr_matrix(A)
    for o in offs:
        m = n - abs(int(o))
        if m > 0:
            A = A + sp.diags(z[rng.integers(0, 7, m)] / 1.0, int(o), shape=(n, n))
    return sp.csr_matrix(A, dtype=np.complex128)


@pytest.mark.parametrize("n,width,imag", [(1, 0, True), (2, 1, False), (65, 16, True),
                                          (1024, 16, False), (300, 7, False)])
def test_packed_host_holds_the_operator(n, width, imag):
    A = _op(n, width, imag)
    codes, diag, table, w, cbits, im = M._packed_host(A, n, False)
    B = np.diag(diag).astype(complex)
    val = 1j * table if im else table
    assert table[0] == 0 and w % 2 == 0 and codes.shape[0] == max(w, 1)
    for u in range(w):
        col, idx = codes[u] & ((1 << cbits) - 1), codes[u].astype(int) >> cbits
        assert (col < n).all() and (idx < len(table)).all()
        np.add.at(B, (np.arange(n), col), val[idx])
    assert (B == A.toarray()).all()


def test_packed_host_refuses(monkeypatch):
    tab = TABLEAUS["vern7"]
    assert M._packed_host(_op(200, 17, True), 200, False) is None  # too many entries a row
    A = sp.csr_matrix(np.diag(np.arange(1.0, 300), 1) * 1j)  # 299 distinct values
    assert M._packed_host(A, 300, False) is None
    A = _op(1024, 4, True) + sp.diags(1j * (np.arange(1.0, 1024) % 70), 1)
    assert M._packed_host(A, 1024, False) is None  # more than 6 bits of values
    # stored zeros do not count
    B = _op(200, 16, True).tocoo()
    z = np.arange(30)
    B = sp.csr_matrix((np.concatenate([B.data, 0.0 * z]),
                       (np.concatenate([B.row, 0 * z + 7]),
                        np.concatenate([B.col, 100 + z]))), shape=(200, 200))
    assert np.diff(B.indptr).max() > 17 and M._packed_host(B, 200, False) is not None
    assert M._packed_host(sp.csr_matrix((3, 3), dtype=complex), 3, False) is not None
    dense = sp.csr_matrix(np.random.default_rng(0).normal(size=(512, 512)) + 0j)
    monkeypatch.setattr(sp.csr_matrix, "copy", None)  # refused before any work on the whole
    assert M._packed_host(dense, 512, False) is None
    monkeypatch.undo()
    ok = _op(20, 4, True)
    assert M.packed_op(ok, 20, False, TABLEAUS["tsit5"], True) is None
    assert M.packed_op(ok, 20, False, tab, False) is None


def test_packed_host_complex64_keeps_the_order():
    A = _op(300, 8, False)
    codes, diag, table, w, cbits, im = M._packed_host(A, 300, True)
    E = sp.csr_matrix(A, dtype=np.complex64)
    E.sort_indices()
    assert codes.shape == (w + 1, 300)
    for r in range(300):
        row = [(codes[u, r] & 511, table[codes[u, r] >> cbits]) for u in range(w)
               if codes[u, r] >> cbits]
        row.insert(int(codes[w, r]), (r, diag[r]))
        assert [c for c, _ in row] == list(E.indices[E.indptr[r]:E.indptr[r + 1]])
        assert [v for _, v in row] == list(E.data[E.indptr[r]:E.indptr[r + 1]])


@pytest.mark.gpu
@pytest.mark.parametrize("n,width,imag,nsys", [
    (1, 0, True, 1), (2, 1, False, 1), (63, 2, True, 3), (64, 3, False, 1), (65, 16, True, 300),
    (512, 16, False, 1), (512, 6, True, 257), (513, 10, True, 2), (1000, 4, False, 1),
    (1024, 16, True, 2), (1024, 15, False, 1)])
@pytest.mark.parametrize("fp32", [False, True])
def test_small_packed_against_ell(n, width, imag, nsys, fp32):
    A = _op(n, width, imag, seed=n + width)
    rng = np.random.default_rng(1)
    y0 = rng.normal(size=(nsys, n)) + 1j * rng.normal(size=(nsys, n))
    y0 /= np.linalg.norm(y0, axis=1)[:, None]
    rtol, atol = (1e-4, 1e-5) if fp32 else (1e-6, 1e-8)
    S = SmallSolve(A, rtol=rtol, atol=atol, fp32=fp32)
    k = np.arange(n, dtype=np.int32)
    S.set_functionals(np.array([0, 1], np.int32), np.array([0, n, 2 * n], np.int32),
                      np.concatenate([k, k]), np.concatenate([k, k[::-1]]),
                      np.ones(2 * n, np.complex128))
    times = np.linspace(0.3, 1.0, 7)
    assert S._packed is not None
    got, yg, ig = S.run(0.0, y0, times)
    S._packed = None
    ref, yr, ir = S.run(0.0, y0, times)
    assert (ig[:, 0] == ir[:, 0]).all() and (ig[:, 0] >= 0).all()
    assert (ig[:, 3] == ir[:, 3]).all()  # attempts
    eps = np.finfo(np.float32 if fp32 else np.float64).eps
    tol = 0.0 if fp32 else 1e4 * eps * ir[:, 3].max()
    a, b = (np.empty((nsys, n), np.complex128) for _ in range(2))
    yg.download(a)
    yr.download(b)
    assert np.linalg.norm(a - b, axis=1).max() <= tol
    assert np.abs(got - ref).max() <= 2 * np.sqrt(n) * tol
    if fp32:
        assert np.array_equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("N,fp32", [(2, False), (32, False), (128, False), (300, False),
                                    (128, True), (500, True)])
def test_trajectories_packed_against_ell(N, fp32):
    """A damped two-level system times an N-level ring with equal couplings
    (few values, width 3): the same jumps, times and expectation values."""
    ring = sp.diags([np.ones(N - 1), np.ones(N - 1)], [1, -1]) if N > 1 else sp.csr_matrix((1, 1))
    sx, sm = sp.csr_matrix([[0, 1], [1, 0]]), sp.csr_matrix([[0, 1], [0, 0]])
    H = qa.Qobj(sp.csr_matrix(sp.kron(sp.identity(2), ring) + 0.5 * sp.kron(sx, sp.identity(N)),
                              dtype=np.complex128))
    c = qa.Qobj(sp.csr_matrix(sp.kron(sm, sp.identity(N)), dtype=np.complex128))
    e = qa.Qobj(sp.csr_matrix(sp.kron(sm.T @ sm, sp.identity(N)), dtype=np.complex128))
    S = qa.MCSolver(H, [c], options={"precision": "fp32" if fp32 else "fp64"})
    psi = np.zeros(2 * N, dtype=complex)
    psi[N] = 1.0
    tl = np.linspace(0, 4.0, 9)
    draws = M.draws_for(np.random.SeedSequence(3).spawn(40), 64)
    dev = S._device_ops(fp32)
    assert dev[4] is not None
    got, ig, tg, wg = S.run_batch(psi, tl, [e], draws)
    S._dev = dev[:4] + (None,)
    ref, ir, tr, wr = S.run_batch(psi, tl, [e], draws)
    assert (ig[:, :3] == ir[:, :3]).all() and (ig[:, 0] == 0).all()
    eps = np.finfo(np.float32 if fp32 else np.float64).eps
    # a jump's time is found to norm_tol, its state to 1e4 eps attempts
    tol = 1e4 * eps * ir[:, 3].max()
    assert np.abs(got - ref).max() <= 4 * tol
    hit = np.arange(tr.shape[1])[None, :] < ir[:, 1:2]
    assert (wg[hit] == wr[hit]).all()
    assert np.abs(tg[hit] - tr[hit]).max(initial=0.0) <= 4 * tol + (1e-6 if fp32 else 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("d,fit", [(20, 2048), (64, 2048), (65, 1024), (129, 512), (300, 256),
                                   (512, 256)])
def test_ell_trajectories_of_both_forms(d, fit):
    """An operator that does not pack: `fit` trajectories are the most that
    take the kernel with 256 registers (eight entries a load), one more takes
    the other (four).  Same sums in the same order: the same bits."""
    print(f"ELL trajectories d={d} fit={fit}", flush=True)
    H = qa.rand_herm(d, density=min(1.0, 30.0 / d), seed=d)
    S = qa.MCSolver(H, [0.3 * qa.destroy(d)])
    psi = np.ones(d, dtype=complex) / np.sqrt(d)
    tl = np.linspace(0, 0.5, 4)
    one = M.draws_for(np.random.SeedSequence(5).spawn(7), 64)
    assert S._device_ops(False)[4] is None
    out = []
    for nt in (fit, fit + 1):
        e, info, _, _ = S.run_batch(psi, tl, [qa.num(d)], np.resize(one, (nt, 64)))
        assert (info[:, 0] == 0).all()
        # every seventh trajectory is the same one
        assert (info == np.resize(info[:7], info.shape)).all()
        assert np.array_equal(e, np.resize(e[:7], e.shape))
        out.append((e[:7], info[:7]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
