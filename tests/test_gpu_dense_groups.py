"""The Hermitian dense stages with the products of a tile shared: by groups
of waves of one workgroup (16 x 16 tiles, at most 256 of them) and by several
workgroups, the last of which adds the sums (32 x 32 tiles, fewer than 512).

Against the full-RHS kernels on the same solve.  Every element of a stage is
np sums of N products in FP32, in other orders: a difference of at most
np N eps32 of the sums' absolute values, here below 2 per unit time, over a
time of 0.1.  The sums are added in a fixed order: a second run gives the
same bits.  Shapes: every split of K, two to ten products, tile counts
around both limits (351 -> 352 rows and 1024), a single tile column."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from qutip_amd.solver.hip_rk import RKEngine  # noqa: E402
from tests.test_gpu_dense_herm import _system, _trace_functionals  # noqa: E402


def _solve(Hnh, cs, rho0, tl, prec, herm, ops, shape, shared=False):
    eng = RKEngine(None, "vern7", 1e-6, 1e-8, dense=(Hnh, cs), dense_precision=prec,
                   shared=shared)
    eng.set_hermitian(herm)
    if shape is not None:
        eng.dense_shape = (shape[0], eng.dense_shape[1], shape[1])
    eng.set_functionals(*_trace_functionals(ops, Hnh.shape[0]))
    out = []
    for _ in range(2):
        eng.set_state(tl[0], rho0.ravel(order="F"))
        vals, _, _ = eng.run(tl[1:])
        _, y = eng.get_state()
        out.append((vals, y.to_array().reshape(Hnh.shape, order="F")))
    return out


@pytest.mark.parametrize("N,nc,tiled,hsplit", [
    (32, 6, 0, 1), (64, 0, 0, 2), (64, 3, 0, 1), (128, 1, 0, 4), (128, 6, 0, 2), (128, 8, 0, 4),
    (256, 2, 0, 8), (352, 3, 0, 1), (384, 1, 0, 4), (64, 3, 1, 2), (192, 0, 1, 1),
    (512, 3, 1, 8), (960, 1, 1, 1), (1024, 1, 1, 8)])
@pytest.mark.parametrize("prec", ["fp32", "bf16x6"])
def test_shared_products_match_full_rhs(N, nc, tiled, hsplit, prec):
    print(f"dense groups N={N} nc={nc} tiled={tiled} hsplit={hsplit} {prec}", flush=True)
    _check(N, nc, tiled, hsplit, prec, False)


@pytest.mark.parametrize("N,nc,hsplit", [(32, 6, 1), (64, 3, 2), (128, 2, 4), (256, 1, 8),
                                         (352, 3, 1)])
@pytest.mark.parametrize("prec", ["fp32", "bf16x6"])
def test_one_group_of_a_shared_engine_matches_full_rhs(N, nc, hsplit, prec):
    print(f"dense, shared engine N={N} nc={nc} hsplit={hsplit} {prec}", flush=True)
    _check(N, nc, 0, hsplit, prec, True)


def _check(N, nc, tiled, hsplit, prec, shared):
    H, cs, Hnh, rho0 = _system(N, 3 + N + nc, nc)
    tl = np.linspace(0, 0.1, 3)
    ops = [H, np.diag(np.arange(N) / N).astype(complex)]
    (vh, yh), (v2, y2) = _solve(Hnh, cs, rho0, tl, prec, True, ops, (tiled, hsplit), shared)
    (vf, yf), _ = _solve(Hnh, cs, rho0, tl, prec, False, ops, None)
    assert np.array_equal(vh, v2) and np.array_equal(yh, y2)
    assert np.array_equal(yh, yh.conj().T)
    eps = np.finfo(np.float32).eps
    tol = 2 * 0.1 * (2 + nc) * N * eps * max(1.0, np.abs(vf).max())
    assert np.abs(vh - vf).max() <= tol
    assert np.abs(yh - yf).max() <= tol * np.abs(yf).max()
