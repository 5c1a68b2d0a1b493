"""Reading trajectories back member by member: the transposition on the device
(clode_members_f64 / _f32, tiles of 64 members x 32 rows) and the staged copy
(from 8 MiB on) against the rows as the integrator stores them."""

import os
import threading

import numpy as np
import pytest

import clode_amd as clode
from clode_amd.cpp import clode_cpp_wrapper as w

MODELS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "clode_amd", "models")


def test_member_rows():
    """Each member's first rows as an array with the type of a row, copied, in blocks of at most 64 KiB."""
    a = np.random.default_rng(0).random((4, 5, 2))
    dt = np.dtype({"names": ["u", "v"], "formats": [np.float64] * 2})
    rows = w.member_rows(a, [5, 0, 3, 1], dt)
    assert [r.shape for r in rows] == [(5,), (0,), (3,), (1,)] and all(r.dtype == dt for r in rows)
    for i, r in enumerate(rows):
        assert np.array_equal(r["u"], a[i, :len(r), 0]) and np.array_equal(r["v"], a[i, :len(r), 1])
        assert r.flags.writeable and r.flags.c_contiguous and not np.shares_memory(r, a)
    assert not any(np.shares_memory(r, q) for r in rows for q in rows if r is not q and len(r) and len(q))
    flat = w.member_rows(a[:, :, 0].copy(), [1, 2, 3, 4], np.dtype(np.float64))
    assert [r.tolist() for r in flat] == [a[i, :i + 1, 0].tolist() for i in range(4)]
    many = np.arange(700 * 40.0).reshape(700, 40)
    counts = [(7 * i) % 41 for i in range(700)]
    rows = w.member_rows(many, counts, np.dtype(np.float64))
    assert all(np.array_equal(r, many[i, :counts[i]]) and r.base.nbytes <= 65536 for i, r in enumerate(rows))
    assert len({id(r.base) for r in rows if r.size}) == -(-sum(counts) * 8 // 65536)
    large = w.member_rows(np.ones((3, 9000)), [9000, 1, 8999], np.dtype(np.float64))
    assert [r.size for r in large] == [9000, 1, 8999] and [r.base.size for r in large] == [9000, 1, 8999]
    for bad in (([6, 0, 0, 0], dt), ([-1, 0, 0, 0], dt), ([1, 1, 1], dt), ([1, 1, 1, 1], np.dtype(np.float64))):
        with pytest.raises(ValueError):
            w.member_rows(a, *bad)


@pytest.mark.gpu
def test_outputs_own_their_samples(gpu_available):
    """An output of an ensemble has a copy of its samples, in a block of at most 64 KiB: writing into one changes neither the others nor what the
    simulator holds."""
    sim = clode.TrajectorySimulator(src_file=os.path.join(MODELS, "van_der_pol.cl"), variables={"x": 1.0, "y": 0.0},
                                    parameters={"mu": 1.0}, dt=0.01, stepper=clode.Stepper.rk4, t_span=(0.0, 0.2),
                                    max_store=50, single_precision=False)
    sim.set_ensemble(variables={"x": np.linspace(0.5, 2.0, 5)})
    out = sim.trajectory()
    held = {k: getattr(sim, "_device_" + k).copy() for k in ("t", "x", "dx")}
    other = out[3].to_ndarray("x").copy()
    for slot in ("t", "x", "dx"):
        a = getattr(out[2], slot)
        assert a.base.nbytes <= 65536 and len(a) < 50
        a[:] = 0
    assert all(np.array_equal(getattr(sim, "_device_" + k), held[k], equal_nan=True) for k in held)
    assert np.array_equal(out[3].to_ndarray("x"), other)


def test_getters_before_any_data():
    """Empty results before problem data are set, also where there is no device."""
    pi = w.ProblemInfo(os.path.join(MODELS, "van_der_pol.cl"), ["x", "y"], ["mu"], [], 0)
    sim = w.TrajectorySimulatorBase(pi, "rk4", False, w.OpenCLResource(), "")
    for name in ("x0", "xf", "dt", "tf", "t_members", "x_members", "dx_members", "aux_members"):
        assert np.size(getattr(sim, "get_" + name)()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("members", [0, 1, 5, 70, 200])
def test_members_block_by_block(gpu_available, monkeypatch, members, single):
    """Read-back in blocks of a few members (the last one smaller; 0: not even one member fits, and the host takes the
    rows apart), blocks that differ from kind to kind, and one that stays for the next read."""
    n, store = 257, 67
    monkeypatch.setenv("CLODE_MEMBERS_BYTES", str(members * store * 2 * 8))
    test_members_are_the_stored_rows(None, n, store, single)


@pytest.mark.gpu
def test_reading_compiles_nothing(gpu_available, capfd):
    """Trajectories are read after the simulator was configured for another program, which is not compiled for it."""
    sim = _native("van_der_pol.cl", ["x", "y"], ["mu"], [], np.ones((3, 2)), np.ones((3, 1)), 7)
    x = sim.get_x_members()
    sim.set_stepper("heun")
    level = clode.get_log_level()
    clode.set_log_level(clode.LogLevel.debug)
    try:
        again = sim.get_x_members()
    finally:
        clode.set_log_level(level)
    assert np.array_equal(x, again)
    assert "compiled" not in "".join(capfd.readouterr())


@pytest.mark.gpu
@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("n, store", [(1, 5), (63, 32), (64, 33), (65, 31), (257, 1), (5001, 130)])
def test_members_are_the_stored_rows(gpu_available, n, store, single):
    rng = np.random.default_rng(n)
    sim = clode.TrajectorySimulator(src_file=os.path.join(MODELS, "linear_drag.cl"),
                                    variables={"y1": 0.0, "y2": 0.0},
                                    parameters={"m": 0.25, "w": 8.0, "k": 2.0, "H": 10.0}, aux=["g1"], num_noise=0,
                                    dt=0.01, stepper=clode.Stepper.rk4, t_span=(0.0, 0.6), max_store=store,
                                    max_steps=1000, single_precision=single)
    sim.set_ensemble(variables={"y1": rng.random(n), "y2": rng.random(n)})
    out = sim.trajectory()
    out = [out] if n == 1 else out
    native = sim._integrator
    count = np.minimum(np.array(native.get_n_stored()) + 1, store)
    rows = {}
    for name, width in (("t", 1), ("x", 2), ("dx", 2), ("aux", 1)):
        flat = np.array(getattr(native, "get_" + name)())
        rows[name] = flat[: n * width * store].reshape((n, width, store), order="F")
    assert len(out) == n
    for i, tr in enumerate(out):
        k = count[i]
        assert np.array_equal(tr.t, rows["t"][i, 0, :k])
        for j, v in enumerate(("y1", "y2")):
            assert np.array_equal(tr.x[v], rows["x"][i, j, :k])
            assert np.array_equal(tr.dx[v], rows["dx"][i, j, :k])
        assert np.array_equal(tr.aux["g1"], rows["aux"][i, 0, :k])
        assert np.array_equal(tr.to_ndarray("x"), rows["x"][i, :, :k].T)


def _native(model, variables, parameters, aux, x0, pars, store):
    pi = w.ProblemInfo(os.path.join(MODELS, model), variables, parameters, aux, 0)
    sim = w.TrajectorySimulatorBase(pi, "rk4", False, w.OpenCLResource(), "")
    sim.set_solver_params(w.SolverParams(0.01, 1.0, 1e-6, 1e-4, 1000, store, 1))  # the step of data set after it
    sim.set_problem_data(x0.ravel(order="F"), pars.ravel(order="F"))
    sim.set_tspan([0.0, 0.5])
    sim.trajectory()
    return sim


@pytest.mark.gpu
def test_data_of_another_problem_are_not_read(gpu_available):
    """A problem with more variables and aux outputs: what is on the device is refused until it is set or integrated
    again, by getters and launches alike, and then has the new sizes."""
    n, store = 65, 33
    rng = np.random.default_rng(5)
    vdp = ("van_der_pol.cl", ["x", "y"], ["mu"], [], rng.random((n, 2)), rng.random((n, 1)), store)
    drag = ("linear_drag.cl", ["y1", "y2"], ["m", "w", "k", "H"], ["g1"], rng.random((n, 2)), 1 + rng.random((n, 4)), store)
    lorenz = ("lorenz.cl", ["x", "y", "z"], ["r", "s", "b"], [], rng.random((n, 3)), 1 + rng.random((n, 3)), store)
    for second in (drag, lorenz):
        sim = _native(*vdp)
        sim.set_problem_info(w.ProblemInfo(os.path.join(MODELS, second[0]), second[1], second[2], second[3], 0))
        for name in ("aux_members",) if second is drag else ("x_members", "dx_members"):
            with pytest.raises(ValueError):
                getattr(sim, "get_" + name)()
        if len(second[1]) > 2:
            with pytest.raises(ValueError):
                sim.get_x0()
            with pytest.raises(ValueError):
                sim.set_x0(second[4].ravel(order="F"))
        for call in (sim.transient, sim.trajectory, sim.shift_x0):
            with pytest.raises(ValueError):
                call()
        sim.set_problem_data(second[4].ravel(order="F"), second[5].ravel(order="F"))
        sim.trajectory()
        fresh = _native(*second)
        for name in ("t_members", "x_members", "dx_members", "aux_members", "n_stored", "xf"):
            assert np.array_equal(getattr(sim, "get_" + name)(), getattr(fresh, "get_" + name)())


@pytest.mark.gpu
def test_two_threads_read_one_simulator(gpu_available):
    """Threads that read one simulator at the same time get what each gets alone: trajectories, and the feature matrix,
    whose getter gives up the interpreter lock."""
    n, store = 4099, 67
    rng = np.random.default_rng(6)
    sim = _native("lorenz.cl", ["x", "y", "z"], ["r", "s", "b"], [], rng.random((n, 3)), 1 + rng.random((n, 3)), store)
    pi = w.ProblemInfo(os.path.join(MODELS, "lorenz.cl"), ["x", "y", "z"], ["r", "s", "b"], [], 0)
    feat = w.FeatureSimulatorBase(pi, "rk4", "basicall", w.ObserverParams(), True, w.OpenCLResource(), "")
    feat.set_problem_data(rng.random(3 * n), 1 + rng.random(3 * n))
    feat.set_tspan([0.0, 0.5])
    feat.features()
    calls = [sim.get_t_members, sim.get_x_members, sim.get_dx_members, sim.get_xf] + 4 * [feat.get_f_members]
    alone = [np.array(call()) for call in calls]
    wrong = []

    def read(k):
        for _ in range(12):
            if not np.array_equal(calls[k](), alone[k], equal_nan=True):
                wrong.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []


def test_to_ndarray_of_replaced_samples():
    """A slot that was given an array of other field types is converted, not reinterpreted."""
    x = np.arange(10.0).reshape(5, 2)
    out = clode.TrajectoryOutput(t=np.arange(5.0), x=x, dx=-x, aux=np.empty((5, 0)), variable_names=["u", "v"], aux_names=[])
    assert np.array_equal(out.to_ndarray("x"), x) and out.to_ndarray("x").dtype == np.float64
    out.x = out.x.astype([("u", np.float32), ("v", np.float32)])
    assert np.array_equal(out.to_ndarray("x"), x)
    out.dx = out.dx.astype([("u", np.int64), ("v", np.float64)])
    assert np.array_equal(out.to_ndarray("dx"), -x)
