"""The work that users have this framework do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which public entry points a pass goes through:

  transient   Simulator.transient with the final state read back
  trajectory  TrajectorySimulator.trajectory with every stored sample read back
  features    FeatureSimulator: set_ensemble, transient, features (warm-up pass where the observer has one) and the
              feature matrix read back, one after the other as a parameter study does it
  batch       BatchSimulator: transient and features of four different systems in shared launches
  train       MLPSurrogate: a new network trained on a labelled set, its weights and its losses read back
  screen      MLPSurrogate.screen_grid over a parameter grid, with a trained-size network
  forward     MLPSurrogate.forward, the raw head outputs of given points
  grad        MLPSurrogate.loss_grad, loss and gradient over given rows

`exact` integrates the same ensemble with the published steppers and the same controller rule in 64-bit torch, and
evaluates the network in 64-bit torch; it uses none of the framework's code.
"""
import math
import os

import numpy as np
import torch

import clode_amd as clode
from clode_amd.surrogate import MLPSurrogate

MODELS = os.path.join(os.path.dirname(os.path.abspath(clode.__file__)), "models")

STEPPERS = {"euler": clode.Stepper.euler, "heun": clode.Stepper.heun, "rk4": clode.Stepper.rk4,
            "bs23": clode.Stepper.bs23, "dopri5": clode.Stepper.dormand_prince,
            "seuler": clode.Stepper.stochastic_euler}
OBSERVERS = {"basic": clode.Observer.basic, "basicall": clode.Observer.basic_all_variables,
             "localmax": clode.Observer.local_max, "nhood2": clode.Observer.neighbourhood_2,
             "thresh2": clode.Observer.threshold_2}

# Systems: variables, parameters, aux outputs, noise terms; rk4 step; first and largest adaptive step; steps per unit
# of time that the adaptive steppers take at rtol 1e-6; operations of one right-hand side (exp counted as 10)
SYSTEMS = {
    "lactotroph": dict(vars={"v": -60.0, "n": 0.0, "f": 0.0, "c": 0.1},
                       pars={"gcal": 1.5, "gsk": 3.0, "gbk": 1.0, "gk": 2.0}, aux=["ica"], noise=0, dt=0.1,
                       dt0=0.1, dtmax=1.0, rate={"dopri5": 1.0, "bs23": 5.0}, rhs=75),
    "lactotroph_noise": dict(vars={"v": -60.0, "n": 0.0, "f": 0.0, "c": 0.1},
                             pars={"gcal": 1.5, "gsk": 3.0, "gbk": 1.0, "sigma": 2.0}, aux=["ica"], noise=1, dt=0.05,
                             dt0=0.05, dtmax=0.05, rate={}, rhs=90),
    "lorenz": dict(vars={"x": 1.0, "y": 1.0, "z": 1.0}, pars={"sigma": 10.0, "rho": 28.0, "beta": 8.0 / 3.0},
                   aux=[], noise=0, dt=0.01, dt0=0.01, dtmax=1.0, rate={"dopri5": 50.0, "bs23": 250.0}, rhs=9),
    "van_der_pol": dict(vars={"x": 2.0, "y": 0.0}, pars={"mu": 1.0}, aux=[], noise=0, dt=0.01, dt0=0.01, dtmax=1.0,
                        rate={"dopri5": 16.0, "bs23": 80.0}, rhs=6),
    "chay_keizer": dict(vars={"v": -50.0, "n": 0.01, "c": 0.12}, pars={"gca": 1200.0, "gkca": 750.0, "kpmca": 0.1},
                        aux=[], noise=0, dt=0.1, dt0=0.1, dtmax=1.0, rate={"dopri5": 1.2, "bs23": 6.0}, rhs=55),
    "ornstein_uhlenbeck": dict(vars={"x": 0.0}, pars={"theta": 1.0, "mu": 0.0, "sigma": 0.5}, aux=[], noise=1,
                               dt=0.05, dt0=0.05, dtmax=0.05, rate={}, rhs=20),
}
STAGES = {"euler": 1, "seuler": 1, "heun": 2, "rk4": 4, "bs23": 3, "dopri5": 6}
TWO_PASS = ("thresh2", "nhood2")
RTOL, ATOL = 1e-6, 1e-8
NPARAM = 32 * 256 + 256 + 3 * (256 * 256 + 256) + 256 * 128 + 128  # the surrogate's weights and biases
NMAC = 32 * 256 + 3 * 256 * 256 + 256 * 72                          # its products for one point


def listed():
    return [
        # a first try of a model: one member, the API's default stepper and precision; the call's own latency
        dict(name="transient 1 vdp", kind="transient", system="van_der_pol", precision="single", stepper="rk4", members=1,
             span=2.005),
        # a few cells looked at closely: every step of ten members kept and read back
        dict(name="trajectory 10 lactotroph", kind="trajectory", system="lactotroph", precision="double",
             stepper="dopri5", members=10, store=1000, span=4000.0),
        # many short stored trajectories; the read-back is most of what it moves
        dict(name="trajectory 8191 lorenz", kind="trajectory", system="lorenz", precision="double", stepper="dopri5",
             members=8191, store=64, span=1000.0),
        # the API's default precision and stepper on an odd-sized ensemble, observer of all variables
        dict(name="basicall 1000 lactotroph", kind="features", system="lactotroph", precision="single", stepper="rk4",
             observer="basicall", members=1000, transient=100.05, span=300.05),
        # the fixed-step parameter line of the relaxation oscillator, too few members to fill the chip
        dict(name="thresh2 4096 vdp", kind="features", system="van_der_pol", precision="double", stepper="rk4",
             observer="thresh2", members=4096, transient=40.005, span=100.005),
        # the 256 x 256 two-parameter feature map of the bursting cell, one wave of members for each SIMD
        dict(name="thresh2 65536 lactotroph", kind="features", system="lactotroph", precision="double",
             stepper="dopri5", observer="thresh2", members=65536, transient=5000.0, span=20000.0),
        # a larger map in the fast precision, several waves for each SIMD
        dict(name="thresh2 262144 fp32c", kind="features", system="lactotroph", precision="fp32c", stepper="dopri5",
             observer="thresh2", members=262144, transient=5000.0, span=10000.0),
        # a very large ensemble of a small system: integration and a read-back of 193 MB
        dict(name="localmax 1048576 lorenz", kind="features", system="lorenz", precision="double", stepper="dopri5",
             observer="localmax", members=1048576, transient=0.0, span=10.0),
        # the low-order adaptive stepper in the fast precision
        dict(name="localmax 300000 bs23", kind="features", system="van_der_pol", precision="fp32c", stepper="bs23",
             observer="localmax", members=300000, transient=20.0, span=60.0),
        # noise realisations of one cell
        dict(name="thresh2 16384 noise", kind="features", system="lactotroph_noise", precision="double",
             stepper="seuler", observer="thresh2", members=16384, transient=500.0, span=2000.0),
        # the surrogate of a feature map: training on integrated samples
        dict(name="train 65536", kind="train", rows=65536, epochs=2, batch=2048),
        # the surrogate of a feature map: the grid it screens
        dict(name="screen 2048x2048", kind="screen", nx=2048, ny=2048, dilate=5),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _between_steps(system, span):
    """An end time half a fixed step away from any step's end, so that a rounding of the time adds or drops none."""
    dt = SYSTEMS[system]["dt"]
    return round((math.floor(span / dt) + 0.5) * dt, 6)


def draw(rng):
    kind = rng.choice(["transient", "trajectory", "features", "features", "features", "batch", "train", "screen",
                       "forward", "grad"])
    if kind == "transient":
        system, stepper = rng.choice([("van_der_pol", "rk4"), ("lorenz", "dopri5"), ("lactotroph", "rk4"),
                                      ("lactotroph", "dopri5"), ("chay_keizer", "heun"), ("van_der_pol", "euler")])
        unit = 10.0 if system in ("lactotroph", "chay_keizer") else 0.5
        return dict(kind=kind, system=system, precision=rng.choice(["single", "double", "fp32c"]), stepper=stepper,
                    members=int(_log_uniform(rng, 1, 50000)),
                    span=_between_steps(system, unit * _log_uniform(rng, 2, 12)))
    if kind == "trajectory":
        system, stepper = rng.choice([("lactotroph", "dopri5"), ("lorenz", "dopri5"), ("van_der_pol", "bs23")])
        store = int(_log_uniform(rng, 20, 100 if system == "lorenz" else 500))
        return dict(kind=kind, system=system, precision=rng.choice(["double", "fp32c"]), stepper=stepper,
                    members=int(_log_uniform(rng, 1, 300000 / store)), store=store, span=100000.0)
    if kind == "features":
        system, stepper, observer, tr, span, most = rng.choice([
            ("lactotroph", "dopri5", "thresh2", (500, 5000), (1000, 20000), 65536),
            ("lactotroph", "rk4", "basicall", (50, 200), (100, 400), 65536),
            ("lactotroph", "bs23", "nhood2", (200, 1000), (500, 2000), 40000),
            ("chay_keizer", "dopri5", "thresh2", (200, 2000), (1000, 10000), 65536),
            ("van_der_pol", "rk4", "thresh2", (5, 40), (20, 100), 30000),
            ("van_der_pol", "dopri5", "localmax", (20, 100), (50, 500), 65536),
            ("van_der_pol", "bs23", "localmax", (5, 30), (20, 80), 300000),
            ("lorenz", "dopri5", "localmax", (0, 0), (2, 8), 1 << 20),
            ("lorenz", "bs23", "basic", (0, 0), (2, 6), 1 << 19),
            ("lactotroph_noise", "seuler", "thresh2", (50, 500), (200, 2000), 16384),
        ])
        # localmax of a Lorenz member on its fixed point counts rounding noise in FP32: the means and extrema instead
        precision = rng.choice(["single", "double", "fp32c"])
        if system == "lorenz" and precision != "double":
            observer = "basicall"
        return dict(kind=kind, system=system, precision=precision, stepper=stepper, observer=observer,
                    members=int(_log_uniform(rng, 50, most)),
                    transient=_between_steps(system, _log_uniform(rng, *tr)) if tr[1] else 0.0,
                    span=_between_steps(system, _log_uniform(rng, *span)))
    if kind == "batch":
        return dict(kind=kind, members=int(_log_uniform(rng, 300, 16000)), span=round(_log_uniform(rng, 10, 40), 1))
    if kind == "train":
        return dict(kind=kind, rows=int(_log_uniform(rng, 3000, 60000)), epochs=rng.randint(1, 2),
                    batch=int(_log_uniform(rng, 256, 4096)))
    if kind == "screen":
        return dict(kind=kind, nx=int(_log_uniform(rng, 20, 2048)), ny=int(_log_uniform(rng, 20, 2048)),
                    dilate=rng.randint(0, 6))
    if kind == "forward":
        return dict(kind=kind, rows=int(_log_uniform(rng, 1, 200000)))
    return dict(kind=kind, rows=int(_log_uniform(rng, 64, 65536)))


# ------------------------------------------------------------------ inputs
def _ensemble(system, n, seed):
    """Initial states [n][nVar] and parameters {name: [n]} of a parameter study: a two-parameter grid in member order
    where the system has one, single parameters spread over their range elsewhere, both placed by the seed."""
    r = np.random.default_rng(seed)
    s = SYSTEMS[system]
    x0 = np.tile(np.array(list(s["vars"].values())), (n, 1))
    line = (np.arange(n) + r.random()) / n
    if system in ("lactotroph", "chay_keizer"):
        n1 = max(1, math.isqrt(n))
        n2 = -(-n // n1)
        a, b = (np.arange(n) // n2 + r.random()) / n1, (np.arange(n) % n2 + r.random()) / n2
        if system == "lactotroph":
            return x0, {"gk": 10.0 * a, "gbk": 2.0 * b}
        return x0, {"gca": 550.0 + 500.0 * a, "kpmca": 0.095 + 0.06 * b}
    if system == "lactotroph_noise":  # repeats of one cell
        return x0, {"gbk": np.full(n, 1.0 + 0.2 * r.random())}
    if system == "lorenz":  # spiralling onto a fixed point: no chaotic member, so that results can be compared
        return x0 + 0.1 * r.standard_normal((n, 3)), {"rho": 5.0 + 8.0 * line}
    if system == "van_der_pol":
        return x0, {"mu": 0.1 + 4.9 * line}
    return x0, {"theta": np.ones(n) + 0.1 * r.random()}


def _arguments(system, precision, stepper):
    s = SYSTEMS[system]
    adaptive = stepper in ("bs23", "dopri5")
    return dict(src_file=os.path.join(MODELS, system + ".cl"), variables=s["vars"], parameters=s["pars"],
                aux=s["aux"], num_noise=s["noise"], stepper=STEPPERS[stepper], single_precision=precision,
                dt=s["dt0"] if adaptive else s["dt"], dtmax=s["dtmax"], abstol=ATOL, reltol=RTOL,
                max_steps=100000000)


def _state_compares(case):
    """Whether a pass also reads the final state back: not where members spike for so long that their phase at the end
    depends on rounding (a Lorenz member here spirals onto its fixed point)."""
    return case["system"] == "lorenz" or (case["stepper"] not in ("bs23", "dopri5") and case["system"] != "lactotroph_noise")


def _tolerances(precision):
    """FP32 runs ask for what FP32 can give."""
    return dict(abstol=1e-6, reltol=1e-4) if precision == "single" else {}


def _training_set(n, seed):
    """Points of the unit square with a smooth period, amplitude and class, as a feature map gives them."""
    r = np.random.default_rng(seed)
    X = r.random((n, 2))
    u = X[:, 0] + 0.3 * np.sin(5 * X[:, 1])
    T = np.stack([np.tanh(3 * (u - 0.5)), np.sin(4 * X[:, 0]) * X[:, 1]], axis=1)
    return X, T, np.clip((6 * u).astype(np.int64), 0, 15).astype(np.int32)


def _network(seed):
    """A network with weights of a trained network's size, on the GPU."""
    net = MLPSurrogate(seed=seed)
    r = np.random.default_rng(seed)
    net.set_params(net.get_params() * (1.0 + 0.1 * r.standard_normal(net.n_params)))
    net.set_target_scaling([5.0, 20.0], [0.5, 10.0])
    return net


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("transient", "trajectory", "features"):
        args = {**_arguments(case["system"], case["precision"], case["stepper"]), **_tolerances(case["precision"])}
        x0, pars = _ensemble(case["system"], case["members"], seed)
        if kind == "transient":
            sim = clode.Simulator(t_span=(0.0, case["span"]), **args)
        elif kind == "trajectory":
            sim = clode.TrajectorySimulator(t_span=(0.0, case["span"]), max_store=case["store"], **args)
        else:
            sim = clode.FeatureSimulator(observer=OBSERVERS[case["observer"]], observer_x_up_thresh=0.3,
                                         observer_x_down_thresh=0.2, **args)
        sim.set_ensemble(variables=x0, parameters=pars)
        if SYSTEMS[case["system"]]["noise"]:
            sim.seed_rng(seed)
        return dict(case=case, sim=sim, x0=x0, pars=pars)
    if kind == "batch":
        sims, r = [], np.random.default_rng(seed)
        for k, (system, stepper, observer) in enumerate((("van_der_pol", "dopri5", "thresh2"),
                                                         ("lactotroph", "rk4", "basicall"),
                                                         ("chay_keizer", "dopri5", "localmax"),
                                                         ("ornstein_uhlenbeck", "seuler", "basicall"))):
            sim = clode.FeatureSimulator(observer=OBSERVERS[observer], observer_x_up_thresh=0.3,
                                         observer_x_down_thresh=0.2, **_arguments(system, "fp32c", stepper))
            x0, pars = _ensemble(system, case["members"], seed + k)
            sim.set_ensemble(variables=x0, parameters=pars)
            sim.set_member_tspan(0.0, case["span"] * np.exp(r.standard_normal(case["members"])))
            sim.seed_rng(seed + k)
            sims.append(sim)
        return dict(case=case, batch=clode.BatchSimulator(sims), sims=sims)
    if kind == "train":
        return dict(case=case, seed=seed, data=_training_set(case["rows"], seed))
    net = _network(seed)
    if kind == "screen":
        return dict(case=case, net=net)
    X, T, cls = _training_set(case["rows"], seed)
    return dict(case=case, net=net, X=X.astype(np.float32), T=T.astype(np.float32), cls=cls)


# -------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "transient":
        return state["sim"].transient(update_x0=False, fetch_results=True)
    if kind == "trajectory":
        out = state["sim"].trajectory(update_x0=False, fetch_results=True)
        out = out if isinstance(out, list) else [out]
        return {"t": np.stack([o.t for o in out]), "x": np.stack([o.to_ndarray("x") for o in out]),
                "dx": np.stack([o.to_ndarray("dx") for o in out])}
    if kind == "features":
        sim = state["sim"]
        sim.set_ensemble(variables=state["x0"], parameters=state["pars"])
        if case["transient"] > 0:
            sim.transient(t_span=(0.0, case["transient"]))
        out = sim.features(t_span=(0.0, case["span"]), initialize_observer=True)
        if not _state_compares(case):
            return {"features": out.to_ndarray()}
        return {"features": out.to_ndarray(), "state": sim.get_final_state()}
    if kind == "batch":
        state["batch"].transient()
        state["batch"].features(initialize_observer=True)
        return [s.get_observer_results().to_ndarray() for s in state["sims"]]
    if kind == "train":
        net = MLPSurrogate(seed=state["seed"])
        X, T, cls = state["data"]
        loss = net.train(X, T, cls, epochs=case["epochs"], batch=case["batch"], lr=3e-3, seed=state["seed"])
        return {"weights": net.get_params(), "loss": loss}
    if kind == "screen":
        P, A, C, F = state["net"].screen_grid(case["nx"], case["ny"], dilate=case["dilate"])
        return {"period": P, "amplitude": A, "class": C, "flags": F}
    if kind == "forward":
        return state["net"].forward(state["X"])
    loss, grad = state["net"].loss_grad(state["X"], state["T"], state["cls"])
    return {"loss": loss, "grad": grad}


# -------------------------------------------------------------------- work
def _steps(case, system, stepper, span):
    s = SYSTEMS[system]
    return span * s["rate"][stepper] if stepper in s["rate"] else span / s["dt"]


def _step_flops(system, stepper):
    n = len(SYSTEMS[system]["vars"])
    return STAGES[stepper] * (SYSTEMS[system]["rhs"] + 2 * n * (STAGES[stepper] + 1) / 2)


def work(case):
    kind = case["kind"]
    if kind in ("transient", "trajectory", "features"):
        s, n = SYSTEMS[case["system"]], case["members"]
        size = 8 if case["precision"] == "double" else 4
        nv, na = len(s["vars"]), len(s["aux"])
        moved = n * size * (2 * nv + len(s["pars"]) + 2) + 16 * n
        if kind == "trajectory":
            steps = case["store"]
            moved += n * case["store"] * size * (1 + 2 * nv + na)
        elif kind == "features":
            passes = 2 if case["observer"] in TWO_PASS else 1
            steps = (_steps(case, case["system"], case["stepper"], case["transient"])
                     + passes * _steps(case, case["system"], case["stepper"], case["span"]))
            moved += n * 8 * (25 + 5 * nv + 3 * na if case["observer"] == "thresh2" else 8 + 5 * nv + 3 * na)
        else:
            steps = _steps(case, case["system"], case["stepper"], case["span"])
        return {"bytes": moved, "flops": n * max(1.0, steps) * _step_flops(case["system"], case["stepper"])}
    if kind == "batch":
        n, span = case["members"], 1.65 * case["span"]  # the mean of exp(z), z ~ N(0, 1)
        flops = sum(p * n * _steps(case, s, st, span) * _step_flops(s, st) for s, st, p in
                    (("van_der_pol", "dopri5", 3), ("lactotroph", "rk4", 2), ("chay_keizer", "dopri5", 2),
                     ("ornstein_uhlenbeck", "seuler", 2)))
        return {"bytes": n * 1500, "flops": flops}
    if kind == "train":
        steps = case["epochs"] * -(-case["rows"] // case["batch"])
        return {"bytes": 20 * case["rows"] * case["epochs"] + 28 * NPARAM * steps,
                "flops": 6 * NMAC * case["rows"] * case["epochs"]}
    if kind == "screen":
        n = case["nx"] * case["ny"]
        return {"bytes": 13 * n + 2 * NPARAM, "flops": 2 * NMAC * n}
    if kind == "forward":
        return {"bytes": (8 + 288) * case["rows"] + 2 * NPARAM, "flops": 2 * NMAC * case["rows"]}
    return {"bytes": 20 * case["rows"] + 6 * NPARAM, "flops": 6 * NMAC * case["rows"]}


def tolerance(case):
    """About four times what the same code shows when its products and sums are rounded apart instead of fused (the
    integrators), when the inputs move by 1e-7 (training) or against 64 bits (the BF16 layers).  Adaptive steps near a
    bifurcation of a spiking cell decide on the last bits: the largest difference of a single member is allowed there."""
    kind = case["kind"]
    if kind == "screen":
        return {"rel": 2e-3, "max": 0.1, "differ": 5e-3}
    if kind in ("forward", "grad"):
        return {"rel": 1.6e-2, "max": 0.5}
    if kind == "train":
        return {"rel": 6e-3, "max": 0.25}
    if kind == "batch":
        return {"rel": 2e-2, "max": 0.99}
    spiking = case["system"] in ("lactotroph", "chay_keizer") and case["stepper"] in TABLEAUS
    if case["precision"] == "single":
        return {"rel": 2e-2, "max": 0.99} if case["stepper"] in TABLEAUS else {"rel": 1e-4, "max": 1e-2}
    if case["precision"] == "fp32c":
        if kind == "trajectory":  # the samples are at the steps, which FP32 rounding moves
            return {"rel": 3e-2, "max": 0.99}
        if case["stepper"] in TABLEAUS:
            return {"rel": 1e-2, "max": 0.99}
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-3, "max": 0.8} if spiking else {"rel": 1e-8, "max": 1e-5}


# ------------------------------------------------------------------- exact
def _rhs(system, p):
    """dx/dt of rows x [nVar][n] in the working type of x."""
    if system == "van_der_pol":
        return lambda x: torch.stack([x[1], p["mu"] * (1 - x[0] * x[0]) * x[1] - x[0]])
    if system == "lorenz":
        return lambda x: torch.stack([p["sigma"] * (x[1] - x[0]), p["rho"] * x[0] - x[1] - x[0] * x[2],
                                      x[0] * x[1] - p["beta"] * x[2]])
    if system == "lactotroph":
        def f(x):
            v, n, g, c = x
            boltzmann = lambda mid, slope: 1 / (1 + torch.exp((mid - v) / slope))  # noqa: E731
            ica = p["gcal"] * boltzmann(-20.0, 12.0) * (v - 60.0)
            drive = v + 75.0
            total = (ica + p["gsk"] * c * c / (c * c + 0.16) * drive + p["gbk"] * g * drive + p["gk"] * n * drive
                     + 0.05 * (v + 50.0))
            return torch.stack([-total / 10.0, (boltzmann(-5.0, 10.0) - n) / 30.0, (boltzmann(-20.0, 2.0) - g) / 8.0,
                                -0.01 * (0.0015 * ica + 0.2 * c)])
        return f
    if system == "chay_keizer":
        def f(x):
            v, n, c = x
            ica = p["gca"] / (1 + torch.exp((-20.0 - v) / 12.0)) * (v - 25.0)
            hill = c * c / (c * c + 0.4 * 0.4)
            total = ica + 3000.0 * n * (v + 75.0) + p["gkca"] * hill * (v + 75.0)
            return torch.stack([-total / 5300.0, (1 / (1 + torch.exp((-16.0 - v) / 5.0)) - n) / 20.0,
                                0.01 * (-4.5e-6 * ica - p["kpmca"] * c)])
        return f
    return None


# Bogacki & Shampine 3(2) and Dormand & Prince 5(4): stage rows, solution weights, error weights, error order
TABLEAUS = {
    "bs23": (((1 / 2,), (0, 3 / 4)), (2 / 9, 1 / 3, 4 / 9), (-5 / 72, 1 / 12, 1 / 9, -1 / 8), 3, 0.5),
    "dopri5": (((1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
                (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
                (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656)),
               (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84),
               (71 / 57600, 0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40), 5, 0.1),
}


def _weighted(k, w):
    return sum(c * a for c, a in zip(w, k) if c)


def _integrate(f, x, dt, span, stepper, dtmax, atol, rtol, store=0):
    """From t = 0 past t = span; with `store`, the first `store` samples (t, x, dx) of every member, else the final
    state.  x [nVar][n], dt [n]; returns what was asked for and the step sizes."""
    n = x.shape[1]
    t, k1 = torch.zeros(n, dtype=x.dtype, device=x.device), f(x)
    kept, fill = [], torch.zeros(n, dtype=torch.long, device=x.device)
    if store:
        kept = [torch.zeros((n, store) + s, dtype=x.dtype, device=x.device) for s in ((), x.shape[:1], x.shape[:1])]
        kept[1][:, 0], kept[2][:, 0] = x.T, k1.T
    trial, failed = dt.clone(), torch.zeros(n, dtype=torch.bool, device=x.device)
    count = 0
    while True:
        live = (t <= span) if not store else (t <= span) & (fill < store - 1)
        if count % 16 == 0 and not bool(live.any()):
            break
        count += 1
        if stepper not in TABLEAUS:
            if stepper == "euler":
                new = x + dt * k1
            elif stepper == "heun":
                new = x + dt * 0.5 * (k1 + f(x + dt * k1))
            else:
                k2 = f(x + dt * 0.5 * k1)
                k3 = f(x + dt * 0.5 * k2)
                k4 = f(x + dt * k3)
                new = x + dt * (k1 + 2 * k2 + 2 * k3 + k4) / 6
            x, t = torch.where(live, new, x), torch.where(live, t + dt, t)
            k1 = f(x)
            done = live
        else:
            rows, sol, err, order, shrink = TABLEAUS[stepper]
            hmin = 16 * (torch.nextafter(t, torch.full_like(t, 1.1 * span)) - t).abs()
            h = torch.minimum(torch.maximum(trial, hmin), torch.full_like(t, dtmax))
            k = [k1]
            for row in rows:
                k.append(f(x + h * _weighted(k, row)))
            new = x + h * _weighted(k, sol)
            k.append(f(new))
            e = h * _weighted(k, err) / torch.maximum(torch.maximum(x.abs(), new.abs()),
                                                     torch.full_like(x, atol / rtol))
            norm = e.abs().amax(0)
            factor = 0.8 * (rtol / norm) ** (1.0 / order)
            good = norm <= rtol
            done = live & (good | (h <= hmin))
            grown = torch.where(failed, h, h * factor.clamp(max=5.0))
            grown = torch.minimum(grown, span - (t + h))
            grown = torch.minimum(torch.maximum(grown, hmin), torch.full_like(t, dtmax))
            next_dt = torch.where(good, grown, hmin)
            shrunk = torch.where(failed, 0.5 * h, h * factor.clamp(min=shrink))
            trial = torch.where(live, torch.where(done, next_dt, shrunk), trial)
            dt = torch.where(done, next_dt, dt)
            failed = torch.where(live, ~done, failed)
            move = done & good
            x, k1, t = torch.where(move, new, x), torch.where(move, k[-1], k1), torch.where(move, t + h, t)
        if store:
            fill = fill + done
            at = fill[done]
            kept[0][done, at], kept[1][done, at], kept[2][done, at] = t[done], x.T[done], k1.T[done]
    return (kept if store else x), dt


def _exact_ensemble(case, seed):
    s, device = SYSTEMS[case["system"]], "cuda" if torch.cuda.is_available() else "cpu"
    steps = case.get("store") or (_steps(case, case["system"], case["stepper"], case["span"])
                                  + _steps(case, case["system"], case["stepper"], case.get("transient", 0.0)))
    ops = steps * (STAGES[case["stepper"]] * (s["rhs"] / 2 + 8) + 30)  # torch calls, about 10 us each
    if s["noise"] or ops > 1.2e6 or (case["kind"] == "features" and not _state_compares(case)):
        return None
    x0, pars = _ensemble(case["system"], case["members"], seed)
    p = {k: torch.as_tensor(np.broadcast_to(pars.get(k, v), case["members"]).copy(), dtype=torch.float64,
                            device=device) for k, v in s["pars"].items()}
    x = torch.as_tensor(x0.T.copy(), dtype=torch.float64, device=device)
    tol = _tolerances(case["precision"]) or dict(abstol=ATOL, reltol=RTOL)
    adaptive = case["stepper"] in TABLEAUS
    dt = torch.full((case["members"],), s["dt0"] if adaptive else s["dt"], dtype=torch.float64, device=device)
    f = _rhs(case["system"], p)
    if case["kind"] == "trajectory":
        kept, _ = _integrate(f, x, dt, case["span"], case["stepper"], s["dtmax"], tol["abstol"], tol["reltol"],
                             case["store"])
        # the fast precisions take other steps: the samples' times are then not the same ones
        if case["precision"] != "double":
            return None
        return dict(zip(("t", "x", "dx"), (v.cpu().numpy() for v in kept)))
    for span in ([case["transient"]] if case.get("transient") else []) + [case["span"]]:
        x, dt = _integrate(f, x, dt, span, case["stepper"], s["dtmax"], tol["abstol"], tol["reltol"])
    x = x.T.cpu().numpy()
    if case["kind"] != "features":
        return x
    return {"features": None, "state": x}


def _exact_layers(net, X):
    """Head outputs [n][72] of points X in 64 bits from the network's own weights, differentiable in them."""
    p = torch.as_tensor(net.get_params(), dtype=torch.float64, device=X.device).requires_grad_()
    B = torch.as_tensor(net.fourier(), dtype=torch.float64, device=X.device)
    phase = 2 * math.pi * (X @ B)
    a, off = torch.stack([torch.sin(phase), torch.cos(phase)], dim=2).reshape(X.shape[0], 32), 0
    for layer, (i, o) in enumerate([(32, 256), (256, 256), (256, 256), (256, 256), (256, 128)]):
        z = a @ p[off:off + i * o].reshape(o, i).T + p[off + i * o:off + i * o + o]
        off += i * o + o
        a = z * torch.sigmoid(z) if layer < 4 else z
    return a[:, :72], p


def _keeps(n):
    """Which head sees which row: the bootstrap hash of (row, head), 0 mod 4 left out."""
    with np.errstate(over="ignore"):
        z = (np.arange(n, dtype=np.uint64)[:, None] * np.uint64(4) + np.arange(4, dtype=np.uint64)
             + np.uint64(0x9e3779b97f4a7c15))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
        return ((z ^ (z >> np.uint64(31))) & np.uint64(3)) != 0


def exact(case, seed):
    kind = case["kind"]
    if kind in ("transient", "trajectory", "features"):
        return _exact_ensemble(case, seed)
    if kind in ("train", "batch"):
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    net = _network(seed)
    if kind == "screen":
        nx, ny = case["nx"], case["ny"]
        c = torch.arange(nx * ny, device=device)
        X = torch.stack([(c // ny).double() / max(nx - 1, 1), (c % ny).double() / max(ny - 1, 1)], dim=1)
        P, A = [], []
        with torch.no_grad():
            for part in X.split(1 << 18):
                z = _exact_layers(net, part)[0].reshape(-1, 4, 18)
                P.append(torch.exp(z[:, :, 0] * 0.5 + 5.0).mean(1))
                A.append((z[:, :, 1] * 10.0 + 20.0).mean(1))
        return {"period": torch.cat(P).reshape(nx, ny).cpu().numpy(),
                "amplitude": torch.cat(A).reshape(nx, ny).cpu().numpy(), "class": None, "flags": None}
    X, T, cls = _training_set(case["rows"], seed)
    X, T = (torch.as_tensor(v.astype(np.float32), device=device).double() for v in (X, T))
    if kind == "forward":
        with torch.no_grad():
            return _exact_layers(net, X)[0].cpu().numpy()
    z, p = _exact_layers(net, X)
    z = z.reshape(-1, 4, 18)
    y = torch.as_tensor(cls.astype(np.int64), device=device)[:, None].expand(-1, 4)
    each = ((z[:, :, :2] - T[:, None, :]) ** 2).sum(2) - torch.log_softmax(z[:, :, 2:], 2).gather(2, y[..., None])[..., 0]
    loss = (each * torch.as_tensor(_keeps(case["rows"]), device=device)).sum() / case["rows"]
    loss.backward()
    return {"loss": float(loss), "grad": p.grad.cpu().numpy()}
