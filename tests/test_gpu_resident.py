"""The resident step loop (one launch for many attempts) against the
launched loop.

Both take the same products, combines, sums and step control in the same
order, so everything must be the same bits: functionals, stored states, the
final state, the counts.  QUTIP_AMD_RESIDENT=0 (read when an engine is
created) keeps the launched loop; the counts of committed resident launches
say which of the two ran.  Sizes at the edges of the resident shapes:
one workgroup, a part of one, a ring that wraps, one XCD full, one row more
(every XCD), two rows of workgroups.  Bar: bit-identical."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

import qutip_amd as qa  # noqa: E402
from qutip_amd import _lib, autotune  # noqa: E402
from qutip_amd.solver.hip_rk import RKEngine, time_dependent_operator  # noqa: E402
from qutip_amd.solver.tableaus import TABLEAUS  # noqa: E402
from tests import systems  # noqa: E402

STATS = ("attempts", "accepted", "dense_preps", "rhs_evals", "status", "out_idx")


def _banded(n, seed=0, offs=(0, 1, -1, 7, -7), few=True):
    """A generator with eigenvalues in the left half plane: few distinct
    values (a coded form) or all distinct (plain SELL)."""
    rng = np.random.default_rng(seed)
    vals = rng.uniform(0.2, 1.0, 9)
    rows = []
    for o in offs:
        m = n - abs(o)
        if m <= 0:
            continue
        v = vals[rng.integers(0, 9, m)] if few else rng.uniform(0.2, 1.0, m)
        rows.append(sp.diags(v * (1j if o else -1.0), o, shape=(n, n)))
    return sp.csr_matrix(sum(rows), dtype=np.complex128)


def _run(eng, y0, tl, fun, store):
    eng.set_functionals(*fun)
    eng.set_state(tl[0], y0)
    buf = qa.HipDense((eng.npad, len(tl))) if store else None
    vals, st, t = eng.run(tl, states_out=buf.ptr if store else None)
    _, y = eng.get_state()
    more, _, _ = eng.run([tl[-1] + 0.05])  # goes on from the state at hand
    stats = eng.stats()
    return (vals, t, y.to_array(), more, buf.to_array() if store else None,
            {k: stats[k] for k in STATS}, _launches(stats))


def _launches(stats):
    return stats["resident_launches"], stats["resident_giveups"], stats["graph_launches"]


def _compare(monkeypatch, make, y0, tl, fun, store=False):
    monkeypatch.setenv("QUTIP_AMD_RESIDENT", "0")
    a = _run(make(), y0, tl, fun, store)
    monkeypatch.delenv("QUTIP_AMD_RESIDENT")
    assert a[6][:2] == (0, 0) and a[6][2] > 0
    eng = make()
    for rep in range(2):
        b = _run(eng, y0, tl, fun, store)
        assert b[6][0] >= 2 and b[6][1:] == (0, 0)  # both runs, no launched iteration
        assert a[5] == b[5]
        assert a[1] == b[1]
        for x, y in ((a[0], b[0]), (a[2], b[2]), (a[3], b[3])):
            assert np.array_equal(x, y)
        if store:
            assert np.array_equal(a[4], b[4])


def _fun(n, rng):
    """A linear functional of scattered rows, a quadratic one and the norm."""
    c = rng.choice(n, min(n, 37), replace=False)
    r = rng.choice(n, min(n, 21), replace=False)
    q = rng.choice(n, len(r), replace=False)
    kinds = [0, 1, 1]
    fptr = np.cumsum([0, len(c), len(r), n])
    w = rng.standard_normal(fptr[-1]) + 1j * rng.standard_normal(fptr[-1])
    return (kinds, fptr, np.concatenate([c * 0, r, np.arange(n)]),
            np.concatenate([c, q, np.arange(n)]), w)


def _state(n, rng):
    y = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return y / np.linalg.norm(y)


# (n, lanes): lanes 1 takes 256 rows a workgroup; 8192 rows fill one XCD's 32
# workgroups, 16384 with two rows of them, 16385 goes to every XCD
@pytest.mark.parametrize("n,lanes", [(64, 1), (300, 4), (1025, 8), (8192, 1), (8193, 1),
                                     (16384, 1), (16385, 1), (5000, 2), (20000, 4), (65536, 1),
                                     (70001, 1)])
@pytest.mark.parametrize("form", ["uniform", "coded", "sell", "sell_c64"])
def test_resident_sparse(monkeypatch, n, lanes, form):
    print(f"resident {form}: n={n} lanes={lanes}", flush=True)
    if n > 20000 and form in ("coded", "sell_c64"):
        pytest.skip("the size is covered by the other forms")
    rng = np.random.default_rng(n)
    A = _banded(n, n, few=form in ("uniform", "coded"))
    coded = form in ("uniform", "coded")
    kw = dict(lanes=lanes, coded=coded, fp32=form == "sell_c64")
    if coded:
        kw["uniform"] = form == "uniform"
    tl = np.array([0.0, 0.3, 0.31, 0.315, 0.32, 0.325, 0.33, 1.0, 3.0])
    _compare(monkeypatch, lambda: RKEngine(A, "vern7", 1e-8, 1e-10, **kw), _state(n, rng), tl,
             _fun(n, rng), store=n <= 20000)


@pytest.mark.parametrize("tableau", ["vern7", "tsit5"])
@pytest.mark.parametrize("interpolate", [True, False])
def test_resident_tableaus(monkeypatch, tableau, interpolate):
    """No dense-output stages (tsit5), and steps that end at the outputs."""
    print(f"resident {tableau} interpolate={interpolate}", flush=True)
    n = 700
    rng = np.random.default_rng(5)
    A = _banded(n)
    tl = np.linspace(0.0, 2.0, 6)

    def make():
        return RKEngine(A, tableau, 1e-7, 1e-9, lanes=2, interpolate=interpolate)

    if not interpolate:  # a step cannot stop at an output in between: an error either way
        for env in ("0", "1"):
            monkeypatch.setenv("QUTIP_AMD_RESIDENT", env)
            eng = make()
            eng.set_functionals(*_fun(n, np.random.default_rng(6)))
            eng.set_state(0.0, _state(n, np.random.default_rng(7)))
            if env == "0":
                try:
                    ref = eng.run(tl[1:])[0]
                except qa.IntegratorException as e:
                    ref = str(e)
            else:
                try:
                    got = eng.run(tl[1:])[0]
                except qa.IntegratorException as e:
                    got = str(e)
                assert _launches(eng.stats())[0] >= 1
        assert np.array_equal(ref, got)
        return
    _compare(monkeypatch, make, _state(n, rng), tl, _fun(n, rng), store=True)


def test_resident_rejections_and_limits(monkeypatch):
    """Rejected attempts (a first step far too long), and a run that spends
    its step budget: the same error at the same count."""
    n = 1500
    rng = np.random.default_rng(3)
    A = _banded(n) * 20.0
    y0 = _state(n, rng)
    tl = np.array([0.2, 0.9, 1.0])
    _compare(monkeypatch, lambda: RKEngine(A, "vern7", 1e-8, 1e-10, lanes=1, first_step=0.5),
             y0, tl, _fun(n, rng))
    seen = []
    for env in ("0", "1"):
        monkeypatch.setenv("QUTIP_AMD_RESIDENT", env)
        eng = RKEngine(A, "vern7", 1e-8, 1e-10, lanes=1, nsteps=5)
        eng.set_state(0.0, y0)
        with pytest.raises(qa.IntegratorException) as e:
            eng.run([50.0])
        seen.append((str(e.value), eng.stats()["attempts"]))
        assert (_launches(eng.stats())[0] > 0) == (env == "1")
    assert seen[0] == seen[1]


def test_resident_output_batches(monkeypatch):
    """More outputs than one launch keeps states for (a 64 MB buffer)."""
    n = 16384
    rng = np.random.default_rng(9)
    A = _banded(n)
    tl = np.linspace(0.0, 1.0, 400)
    _compare(monkeypatch, lambda: RKEngine(A, "vern7", 1e-6, 1e-8, lanes=1), _state(n, rng), tl,
             _fun(n, rng))


@pytest.mark.parametrize("N", [5, 37, 91, 128, 200])
def test_resident_banded_matrix_form(monkeypatch, N):
    print(f"resident banded matrix form N={N}", flush=True)
    s = systems.kerr(N)
    tl = np.linspace(0.0, 0.3, 5)
    out = []
    for env in ("0", "1"):
        monkeypatch.setenv("QUTIP_AMD_RESIDENT", env)
        solver = qa.MESolver(s["H"], s["c_ops"], options={
            "matrix_form": True, "dense_precision": "fp64_banded", "rtol": 1e-8, "atol": 1e-10,
            "store_final_state": True, "nsteps": 100000})
        res = solver.run(s["psi0"], tl, e_ops=s["e_ops"])
        st = solver._integrator.stats()
        assert (_launches(st)[0] > 0) == (env == "1")
        out.append((np.array(res.expect), res.final_state.full(), {k: st[k] for k in STATS}))
    assert out[0][2] == out[1][2]
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("L", [3, 5, 6])
def test_resident_time_dependent(monkeypatch, L):
    print(f"resident time-dependent chain L={L}", flush=True)
    s = systems.ising(L, 0.1)
    X = 0
    for i in range(L):
        X = X + systems.site(qa.sigmax(), i, L)
    H = qa.QobjEvo([s["H"], [X, "cos(w * t)"], [s["e_ops"][0], "exp(-t) * sin(t)"]],
                   args={"w": 1.3})
    td = time_dependent_operator(qa.MESolver(H, s["c_ops"]).rhs.matmul_data)
    n, rng = 4 ** L, np.random.default_rng(L)
    for lanes in (1, 4):
        _compare(monkeypatch, lambda: RKEngine(None, "vern7", 1e-8, 1e-10, td=td, lanes=lanes),
                 _state(n, rng), np.linspace(0.0, 2.0, 9), _fun(n, rng))


def test_resident_switched_off_and_on(monkeypatch):
    """qa_rk_set_resident between runs, in every order with the functionals:
    the loop that is asked for runs, with the same results; no memory is
    taken by switching; the environment's choice stands."""
    print("resident switched off and on", flush=True)
    n = 40000  # a ring of 20 MB
    rng = np.random.default_rng(11)
    A = _banded(n)
    y0, fun, other = _state(n, rng), _fun(n, rng), _fun(n, rng)
    tl = np.array([0.0, 0.4, 0.6])

    def run(eng, f):
        eng.set_functionals(*f)
        eng.set_state(0.0, y0)
        vals = eng.run(tl[1:])[0]
        return vals, eng.get_state()[1].to_array(), _launches(eng.stats())

    monkeypatch.setenv("QUTIP_AMD_RESIDENT", "0")
    eng = RKEngine(A, "vern7", 1e-8, 1e-10, lanes=1)
    eng.set_resident(True)
    ref = {0: run(eng, fun), 1: run(eng, other)}
    assert ref[0][2][0] == ref[1][2][0] == 0
    monkeypatch.delenv("QUTIP_AMD_RESIDENT")
    eng = RKEngine(A, "vern7", 1e-8, 1e-10, lanes=1)
    for on, which in ((False, 0), (True, 0), (True, 1), (False, 1), (False, 0), (True, 0),
                      (True, 1), (False, 0), (True, 1)):
        eng.set_resident(on)
        vals, y, launches = run(eng, (fun, other)[which])
        assert (launches[0] > 0) == on and launches[1] == 0
        assert np.array_equal(vals, ref[which][0]) and np.array_equal(y, ref[which][1])

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        _lib.call("qa_mem_info", C.byref(free), C.byref(total))
        return free.value

    free = free_bytes()
    for _ in range(10):  # a plan each would take 200 MB
        eng.set_resident(False)
        eng.set_resident(True)
        assert run(eng, other)[2][0] > 0
    assert free_bytes() > free - (50 << 20)


@pytest.mark.parametrize("n,lanes,form", [
    (64, 1, "uniform"), (2116, 4, "uniform"), (8192, 1, "sell"),  # one XCD
    (8193, 1, "uniform"), (16385, 2, "sell"), (65536, 1, "uniform")])  # every XCD
@pytest.mark.parametrize("polls", [-1, 0, 1, 4, 16, 64])
def test_resident_gives_up(n, lanes, form, polls):
    """Waits that end before the grid has come together (no polls at all, or
    so few that some workgroups pass a barrier and others do not): the kernels
    end, nothing is written back, and the launched loop goes on from the
    state as it was, as it does where the launch is refused (-1); asked again, the engine's next launch goes through."""
    print(f"resident give-up: n={n} lanes={lanes} {form} polls={polls}", flush=True)
    rng = np.random.default_rng(n + 1)
    A = _banded(n, n, few=form == "uniform")
    kw = dict(lanes=lanes, coded=form == "uniform")
    y0, fun = _state(n, rng), _fun(n, rng)
    tl = np.array([0.0, 0.3, 0.31, 1.0, 3.0])
    eng = RKEngine(A, "vern7", 1e-8, 1e-10, **kw)
    eng.set_functionals(*fun)

    def run(times):
        vals, _, t = eng.run(times)
        st = eng.stats()
        return vals, t, eng.get_state()[1].to_array(), {k: st[k] for k in STATS}, _launches(st)

    def same(a, b):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2])
        assert a[1] == b[1] and a[3] == b[3]

    eng.set_resident(False)
    eng.set_state(0.0, y0)
    ref = [run(tl[1:]), run([3.5, 4.0])]
    assert ref[1][4][0] == 0
    # from the state that was set, and from a resident launch's
    for first in (polls, 1 << 20):
        eng.set_resident(True)
        _lib.call("qa_rk_set_resident_polls", eng.handle, first)
        eng.set_state(0.0, y0)
        got = run(tl[1:])
        same(got, ref[0])
        if first == 1 << 20:
            assert got[4][0] >= 1 and got[4][1] == 0
        _lib.call("qa_rk_set_resident_polls", eng.handle, polls)
        eng.set_resident(True)
        got = run([3.5, 4.0])
        same(got, ref[1])
        if polls <= 0:
            gave_up = (0 if polls < 0 else 1) * (2 if first == polls else 1)
            assert got[4][:2] == (0 if first == polls else 1, gave_up)


def test_resident_lanes_only_for_its_engines(monkeypatch):
    """The resident loop's lane count goes to engines that take that loop: not
    to one of many that run at once, nor to a tableau it refuses (here one
    whose first stage is not at the step's start)."""
    print("resident lanes", flush=True)
    monkeypatch.setenv("QUTIP_AMD_NO_TUNE", "1")
    A = _banded(5000, offs=(0, 1, -1, 3, -3, 7, -7, 9, -9, 20, -20, 30, -30), few=False)
    launched, ruled = autotune.lanes_for(A), autotune.resident_lanes(A)
    assert launched != ruled
    off = dict(TABLEAUS["tsit5"], c=np.asarray(TABLEAUS["tsit5"]["c"]) + 0.01)
    for kw, lanes in (({}, ruled), ({"shared": True}, launched), ({"tableau": off}, launched),
                      ({"lanes": 8}, 8)):
        eng = RKEngine(A, rtol=1e-6, atol=1e-8, coded=False, **kw)
        assert eng.lanes == eng.sell.lanes == lanes
        if "tableau" not in kw:
            eng.set_state(0.0, _state(5000, np.random.default_rng(2)))
            eng.run([0.01])
            assert (eng.stats()["resident_launches"] > 0) == (kw != {"shared": True})
    m = systems.ising(3, 0.1)
    H = qa.QobjEvo([m["H"], [m["e_ops"][0], "cos(t)"]])
    td = time_dependent_operator(qa.MESolver(H, m["c_ops"]).rhs.matmul_data)
    for kw in ({}, {"shared": True}):
        eng = RKEngine(None, rtol=1e-6, atol=1e-8, td=td, **kw)
        eng.set_state(0.0, _state(64, np.random.default_rng(2)))
        eng.run([0.01])
        assert (eng.stats()["resident_launches"] > 0) == (not kw)


def test_served_requests_keep_the_launched_loop():
    print("served sesolve of 1200 rows", flush=True)
    from qutip_amd.serve import SolveRequest, _Running
    d = 1200
    rng = np.random.default_rng(8)
    H = qa.Qobj(sp.csr_matrix(sp.diags([rng.uniform(size=d - 1), rng.uniform(size=d),
                                        np.zeros(d - 1)], [-1, 0, 1]), dtype=complex))
    H = H + H.dag()
    req = SolveRequest("se", H, qa.basis(d, 0), np.linspace(0, 0.5, 3), e_ops=[qa.num(d)])
    run = _Running(req)
    while not run.poll():
        pass
    st = run.eng.stats()
    assert req.error is None and st["resident_launches"] == 0 and st["graph_launches"] > 0
