"""The work whose speed is measured: networks as users of this framework simulate them.

A case is a network that has been built, prepared and simulated through its start-up transient,
and a pass is the next Run of it (batch_simulate for a sweep of several networks), after which
the program reads the state of every neuron. Every pass goes through the package's public calls.

kinds:
- "random": one recurrent network with fixed in-degree (80 % excitatory), a seeded Poisson
  background per neuron and one neuron model; "arrays" connects it with ConnectArrays from
  arrays drawn here, else by the fixed_indegree rule;
- "circuit": the 8-population layered circuit of bench.py at a scale, one-step min_delay,
  optionally with stdp_synapse between the excitatory populations;
- "sweep": instances of uneven size and two models, advanced together by batch_simulate.
"""

import math
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "nest-simulator_amd"))

import nestgpu  # noqa: E402

H = 0.1  # ms, resolution of every case
DELTA = {"C_m": 1.0, "tau_m": 20.0, "V_th": 20.0, "V_reset": 10.0, "E_L": 0.0, "t_ref": 2.0}
EXP = {"tau_m": 10.0, "tau_syn_ex": 0.5, "tau_syn_in": 0.5, "C_m": 250.0, "V_th": -55.0, "V_reset": -70.0,
       "t_ref": 2.0, "E_L": -70.0}
ALPHA = dict(EXP, V_min=-80.0)
AEIF = {"a": 4.0, "b": 80.5, "tau_w": 144.0, "Delta_T": 2.0, "g_L": 30.0, "gsl_error_tol": 1e-3}
IAF_FIELDS = ("V_m", "I_syn_ex", "I_syn_in")
# per model: parameters, initial V_m, excitatory weight, inhibitory factor, standard deviation
# of the weights, drive weight, drive rate (Hz), fields read after a pass, and the mean rate
# (Hz) at which such networks fire, for work()
MODELS = {
    "iaf_psc_delta": (DELTA, (0.0, 20.0), 0.1, -5.0, 0.0, 0.1, 20000.0, ("V_m",), 80.0),
    "iaf_psc_exp": (EXP, (-70.0, -55.0), 87.8, -4.0, 0.1, 87.8, 8000.0, IAF_FIELDS, 30.0),
    "iaf_psc_alpha": (ALPHA, (-70.0, -55.0), 40.0, -4.0, 0.1, 40.0, 8000.0, IAF_FIELDS, 50.0),
    "aeif_cond_exp": (AEIF, (-70.6, -55.0), None, -5.0, 0.0, 6.0, 15000.0, ("V_m", "g_ex", "g_in", "w"), 17.0),
}
PRESIM_MS = 100.0  # the start-up transient, simulated before the measured passes
CIRCUIT_PRESIM_MS = 20.0
POPS = [20683, 5834, 21915, 5479, 4850, 1065, 14395, 2948]  # E/I alternating
STDP = {"tau_plus": 20.0, "lambda": 0.01, "alpha": 1.0, "mu_plus": 1.0, "mu_minus": 1.0, "Wmax": 175.6}


def _random_case(name, model, n, k, d_lo, d_hi, t_ms, n_vp=1, arrays=False, record=False):
    return {"name": name, "kind": "random", "model": model, "n": n, "k": k, "d_lo": d_lo, "d_hi": d_hi, "t_ms": t_ms,
            "n_vp": n_vp, "arrays": arrays, "record": record}


def _circuit_case(name, scale, t_ms, stdp=False):
    return {"name": name, "kind": "circuit", "scale": scale, "t_ms": t_ms, "stdp": stdp}


def _sweep_case(name, instances, n_min, n_max, t_ms):
    return {"name": name, "kind": "sweep", "instances": instances, "n_min": n_min, "n_max": n_max, "t_ms": t_ms}


def listed():
    return [
        # a program in a closed loop: one min_delay slice per call on a small network
        _random_case("step_delta", "iaf_psc_delta", 500, 50, 15, 15, 1.5, arrays=True),
        # an interactive small network of odd size on several virtual processes
        _random_case("small_exp", "iaf_psc_exp", 1777, 125, 10, 30, 20.0, n_vp=3, arrays=False),
        # the balanced random network of the tutorials (5,000 neurons, in-degree 500)
        _random_case("brunel_delta", "iaf_psc_delta", 5000, 500, 15, 15, 60.0, arrays=True),
        # alpha-shaped currents, a prime number of neurons
        _random_case("alpha", "iaf_psc_alpha", 10007, 400, 10, 30, 30.0, arrays=True),
        # a run that is recorded: spikes and sampled potentials, in calls that end inside slices
        _random_case("recorded_exp", "iaf_psc_exp", 4001, 200, 8, 25, 100.0, n_vp=2, record=True),
        # the exponential-synapse network of bench.py: 1e5 neurons, 1.25e8 synapses
        _random_case("large_exp", "iaf_psc_exp", 100000, 1250, 10, 30, 200.0, n_vp=8),
        # conductance-based neurons with adaptive integration
        _random_case("aeif", "aeif_cond_exp", 6000, 600, 15, 15, 30.0, n_vp=4),
        # many neurons with few synapses each: beyond the sizes an LDS window serves
        _random_case("sparse_delta", "iaf_psc_delta", 300000, 100, 12, 24, 60.0, n_vp=8),
        # the layered circuit: a desk-sized one, the full one, and a plastic one
        _circuit_case("circuit_small", 0.1, 40.0),
        _circuit_case("circuit_full", 1.0, 100.0),
        _circuit_case("circuit_stdp", 0.25, 40.0, stdp=True),
        # a parameter sweep: uneven instances of two models advanced together
        _sweep_case("sweep", 48, 1000, 8000, 15.0),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["random"] * 6 + ["circuit"] * 3 + ["sweep"])
    if kind == "circuit":
        stdp = rng.random() < 0.35
        scale = round(_log_uniform(rng, 0.05, 0.25 if stdp else 0.6), 3)
        return dict(_circuit_case("", scale, float(rng.randint(20, 60)), stdp))
    if kind == "sweep":
        n_max = rng.randint(2000, 10000)
        return _sweep_case("", rng.randint(8, 48), rng.randint(400, 1500), n_max, float(rng.randint(10, 30)))
    model = rng.choice(list(MODELS) + ["iaf_psc_exp"])
    n = int(_log_uniform(rng, 300, 8000 if model == "aeif_cond_exp" else 80000)) | 1
    k = max(20, min(n // 10, int(_log_uniform(rng, 50, 1000))))
    d_lo = rng.randint(3, 20)
    d_hi = d_lo + rng.choice([0, rng.randint(1, 30)])
    t = float(rng.randint(10, 60)) if n > 3000 else round(rng.randint(3, 300) * H, 1)
    return _random_case("", model, n, k, d_lo, d_hi, t, n_vp=rng.randint(1, 8),
                        arrays=model != "aeif_cond_exp" and n * k < 3000000 and rng.random() < 0.5,
                        record=n < 20000 and rng.random() < 0.25)


# ------------------------------------------------------------------ networks
def _weights(model, k):
    """Excitatory and inhibitory mean weight at in-degree k."""
    w = MODELS[model][2]
    if model == "aeif_cond_exp":
        w = 6.0 * math.sqrt(0.8 / k)
    elif model == "iaf_psc_delta":
        w = 0.1 * min(1.0, 500.0 / k)
    else:
        w = w * min(1.0, math.sqrt(1250.0 / k))
    return w, w * MODELS[model][3]


def _arrays(case, seed):
    """Connections (source, target, weight, delay in steps), initial V_m: drawn from the seed."""
    rng = np.random.default_rng([seed, 11])
    n, k = case["n"], case["k"]
    ke = int(0.8 * k)
    ne = int(0.8 * n)
    src = np.concatenate([rng.integers(0, ne, size=(n, ke)), rng.integers(ne, n, size=(n, k - ke))], axis=1)
    we, wi = _weights(case["model"], k)
    w = np.where(np.arange(k) < ke, we, wi) * (1.0 + MODELS[case["model"]][4] * rng.standard_normal((n, k)))
    d = rng.integers(case["d_lo"], case["d_hi"] + 1, size=(n, k))
    tgt = np.repeat(np.arange(n), k)
    v0 = rng.uniform(*MODELS[case["model"]][1], n)
    return src.ravel(), tgt, w.ravel(), d.ravel(), v0


def _prepare_random(case, seed):
    model, n, k = case["model"], case["n"], case["k"]
    params, v_range, _, _, sd, w_drive, rate, _, _ = MODELS[model]
    kern = nestgpu.Kernel(0)
    kern.SetKernelStatus({"total_num_virtual_procs": case["n_vp"], "rng_seed": seed % 2000000011 + 1})
    pop = kern.Create(model, n, params)
    if case["arrays"]:
        src, tgt, w, d, v0 = _arrays(case, seed)
        pop.set(V_m=v0)
        ids = pop.global_id
        kern.ConnectArrays(ids[src], ids[tgt], w, d * H)
    else:
        pop.set(V_m=np.random.default_rng([seed, 12]).uniform(*v_range, n))
        ke = int(0.8 * k)
        ne = int(0.8 * n)
        delay = case["d_lo"] * H
        if case["d_hi"] > case["d_lo"]:
            delay = delay + H * nestgpu.random.uniform_int(case["d_hi"] - case["d_lo"] + 1)
        for pre, deg, w in ((pop[:ne], ke, _weights(model, k)[0]), (pop[ne:], k - ke, _weights(model, k)[1])):
            kern.Connect(pre, pop, {"rule": "fixed_indegree", "indegree": deg},
                         {"weight": nestgpu.random.normal(w, sd * abs(w)) if sd else w, "delay": delay})
    gen = kern.Create("spike_generator", n, {"poisson_rate": rate, "poisson_seed": seed})
    kern.Connect(gen, pop, "one_to_one", {"weight": w_drive, "delay": case["d_lo"] * H})
    state = {"case": case, "kernels": [kern], "pops": [pop], "fields": MODELS[model][7]}
    if case["record"]:
        # the usual recording: the spikes of 50 neurons and the potentials of a few
        state["spikes"] = kern.Create("spike_recorder")
        kern.Connect(pop[:min(50, n)], state["spikes"])
        state["meter"] = kern.Create("multimeter", 1, {"interval": 5.0, "record_from": ["V_m"]})
        kern.Connect(state["meter"], pop[:5])
        state["now"] = int(round(PRESIM_MS / H))  # steps simulated so far
    kern.Prepare()
    kern.Run(PRESIM_MS)
    return state


def _prepare_circuit(case, seed):
    rng = np.random.default_rng([seed, 13])
    sizes = [max(1, int(round(p * case["scale"]))) for p in POPS]
    # bench.py's probability matrix and background (drawn after its initial potentials), the
    # same for every seed, so that passes on different inputs do the same work
    bench = np.random.default_rng(777)
    bench.uniform(size=sum(POPS))
    prob = bench.uniform(0.0, 0.14, size=(8, 8))
    k_ext = bench.integers(1500, 2501, size=8)
    kern = nestgpu.Kernel(0)
    kern.SetKernelStatus({"total_num_virtual_procs": 8, "rng_seed": seed % 2000000011 + 1})
    pops = [kern.Create("iaf_psc_exp", m, EXP) for m in sizes]
    for p in pops:
        p.set(V_m=rng.uniform(-70.0, -55.0, len(p)))
    for j, pre in enumerate(pops):
        exc = j % 2 == 0
        w = nestgpu.random.normal(87.8, 8.78) * (1.0 if exc else -4.0)
        d = nestgpu.math.max(nestgpu.random.normal(*((1.5, 0.75) if exc else (0.75, 0.375))), H)
        for i, post in enumerate(pops):
            syn = {"weight": w, "delay": d}
            if case["stdp"] and exc and i % 2 == 0:
                syn.update(STDP, synapse_model="stdp_synapse")
            kern.Connect(pre, post, {"rule": "pairwise_bernoulli", "p": float(prob[i, j])}, syn)
    for i, post in enumerate(pops):
        gen = kern.Create("spike_generator", len(post), {"poisson_rate": 8.0 * float(k_ext[i]), "poisson_seed": seed + i})
        kern.Connect(gen, post, "one_to_one", {"weight": 87.8, "delay": H})
    kern.Prepare()
    kern.Run(CIRCUIT_PRESIM_MS)
    return {"case": case, "kernels": [kern], "pops": pops, "fields": IAF_FIELDS}


def _sweep_specs(case):
    """Model and size of every instance, the same for every seed."""
    rng = np.random.default_rng(4242)
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
    return [("aeif_cond_exp" if i % 2 else "iaf_psc_exp", int(round(math.exp(rng.uniform(lo, hi)))))
            for i in range(case["instances"])]


def _prepare_sweep(case, seed):
    def build(arg):
        i, (model, n) = arg
        params, v_range, _, _, _, w_drive, rate, _, _ = MODELS[model]
        k = n // 10
        kern = nestgpu.Kernel(0)
        # the layout that batch_autotune picks for such instances
        kern.SetKernelStatus({"total_num_virtual_procs": 4, "rng_seed": (seed + 7919 * i) % 2000000011 + 1,
                              "keep_host_connections": False, "targets_per_block": 512, "window_slots": 4})
        pop = kern.Create(model, n, params)
        pop.set(V_m=np.random.default_rng([seed, i]).uniform(*v_range, n))
        ne, ke = int(0.8 * n), int(0.8 * k)
        we, wi = _weights(model, k)
        kern.Connect(pop[:ne], pop, {"rule": "fixed_indegree", "indegree": ke}, {"weight": we, "delay": 1.5})
        kern.Connect(pop[ne:], pop, {"rule": "fixed_indegree", "indegree": k - ke}, {"weight": wi, "delay": 1.5})
        gen = kern.Create("spike_generator", n, {"poisson_rate": rate, "poisson_seed": seed + i})
        kern.Connect(gen, pop, "one_to_one", {"weight": w_drive, "delay": 1.5})
        kern.Prepare()
        return kern, pop

    with ThreadPoolExecutor(8) as ex:
        built = list(ex.map(build, enumerate(_sweep_specs(case))))
    state = {"case": case, "kernels": [b[0] for b in built], "pops": [b[1] for b in built], "fields": ("V_m",)}
    nestgpu.batch_simulate(state["kernels"], 30.0)
    return state


def prepare(case, seed):
    build = {"random": _prepare_random, "circuit": _prepare_circuit, "sweep": _prepare_sweep}[case["kind"]]
    return build(case, int(seed))


def run(state):
    case = state["case"]
    if case["kind"] == "sweep":
        nestgpu.batch_simulate(state["kernels"], case["t_ms"])
        # every instance's potentials, as one table of the sweep
        return {"V_m": np.concatenate([np.atleast_1d(p.get("V_m")) for p in state["pops"]])}
    kern = state["kernels"][0]
    if case.get("record"):
        # three calls, the first two ending inside a slice
        steps = int(round(case["t_ms"] / H))
        parts = [steps // 3, steps // 3, steps - 2 * (steps // 3)]
        for part in parts:
            kern.Run(round(part * H, 1))
    else:
        kern.Run(case["t_ms"])
    out = {f: np.concatenate([np.atleast_1d(p.get(f)) for p in state["pops"]]) for f in state["fields"]}
    if case.get("record"):
        # this pass's spikes as a raster [recorded neuron, step], and its sampled potentials
        ev, mm = state["spikes"].get("events"), state["meter"].get("events")
        first = state["pops"][0].global_id[0]
        at = np.rint(ev["times"] / H).astype(np.int64) - 1 - state["now"]
        raster = np.zeros((min(50, case["n"]), steps), np.uint8)
        raster[ev["senders"][at >= 0] - first, at[at >= 0]] = 1
        out["raster"] = raster
        out["sampled"] = mm["V_m"][np.rint(mm["times"] / H).astype(np.int64) > state["now"]]
        state["now"] += steps
    return out


# ------------------------------------------------------------------ necessary work
def _iaf_work(n, k, steps, rate, fields):
    """Per delivered event: its 12-byte synapse record read once and one addition; per neuron:
    its state read and written once; per neuron and step: about ten operations."""
    events = n * k * rate * steps * H * 1e-3
    return events * 12 + n * (fields * 8 + 4) * 2, events + 10 * n * steps


def work(case):
    steps = int(round(case["t_ms"] / H))
    if case["kind"] == "circuit":
        sizes = [max(1, int(round(p * case["scale"]))) for p in POPS]
        n = sum(sizes)
        # out-degree about 0.056 N; 23 Hz at scale 0.1, 52 Hz at full scale
        b, f = _iaf_work(n, 0.056 * n, steps, 20.0 + 32.0 * case["scale"], 3)
    elif case["kind"] == "random":
        m = case["model"]
        b, f = _iaf_work(case["n"], case["k"], steps, MODELS[m][8], len(MODELS[m][7]))
        if m == "aeif_cond_exp":
            f += 600 * case["n"] * steps  # two accepted RKF45 steps per time step
    else:
        b = f = 0.0
        for m, n in _sweep_specs(case):
            x, y = _iaf_work(n, n // 10, steps, MODELS[m][8], 4)
            b += x
            f += y + (600 * n * steps if m == "aeif_cond_exp" else 0)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ plain numpy, 64 bits
def _poisson(lam, seed, streams, step):
    """Counts of the seeded Poisson drive: splitmix64 of (seed, stream, step), inverse CDF."""
    cdf, p, c = [], math.exp(-lam), 0.0
    for q in range(64):
        c += p
        cdf.append(c)
        if 1.0 - c < 1e-17:
            break
        p *= lam / (q + 1)
    with np.errstate(over="ignore"):
        z = (np.uint64(seed) + streams.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
             + np.uint64(step) * np.uint64(0xD1B54A32D192ED03))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = (z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0
    return np.minimum(np.searchsorted(np.array(cdf), u, side="right"), len(cdf) - 1)


def exact(case, seed):
    """Exact integration in 64 bits where the connections are arrays drawn here."""
    if case["kind"] != "random" or not case["arrays"] or case["record"]:
        return None
    n, k, model = case["n"], case["k"], case["model"]
    steps = int(round((PRESIM_MS + case["t_ms"]) / H))
    params, _, _, _, _, w_drive, rate, fields, hz = MODELS[model]
    if steps * (3e-4 + 6e-8 * n + 4e-8 * n * k * hz * H * 1e-3) > 18.0:
        return None
    src, tgt, w, d, v0 = _arrays(case, int(seed))
    order = np.argsort(src, kind="stable")
    tgt, w, d = tgt[order], w[order], d[order]
    row = np.searchsorted(src[order], np.arange(n + 1))
    del src
    slots = case["d_hi"] + 1
    exc, inh = np.zeros((slots, n)), np.zeros((slots, n))
    e_l = params["E_L"]
    v = v0 - e_l
    theta, reset = params["V_th"] - e_l, params["V_reset"] - e_l
    ref = int(round(params["t_ref"] / H))
    r = np.zeros(n, np.int64)
    tau, c_m = params["tau_m"], params["C_m"]
    p_m = math.exp(-H / tau)
    if model != "iaf_psc_delta":
        ts = params["tau_syn_ex"]
        p_s = math.exp(-H / ts)
        beta = ts * tau / (tau - ts)
        em = math.expm1(H * (tau - ts) / (ts * tau))
        p_21 = beta / c_m * p_s * em
        p_31 = beta / c_m * p_s * (beta * em - H)
    ie, ii, de, di = (np.zeros(n) for _ in range(4))
    streams = np.arange(n + 1, 2 * n + 1)  # the generators' node ids
    for t in range(steps):
        s = t % slots
        we, wi = exc[s].copy(), inh[s].copy()
        exc[s] = 0.0
        inh[s] = 0.0
        active = r == 0
        if model == "iaf_psc_delta":
            v = np.where(active, p_m * v + (we + wi), v)
        elif model == "iaf_psc_exp":
            v = np.where(active, v * p_m + ie * p_21 + ii * p_21, v)
            ie, ii = ie * p_s + we, ii * p_s + wi
        else:
            new = p_31 * de + p_21 * ie + p_31 * di + p_21 * ii + p_m * v
            v = np.where(active, np.maximum(new, params["V_min"] - e_l), v)
            ie, ii = H * p_s * de + p_s * ie, H * p_s * di + p_s * ii
            de, di = de * p_s + math.e / ts * we, di * p_s + math.e / ts * wi
        r = np.where(active, r, r - 1)
        spk = np.flatnonzero(v >= theta)
        r[spk] = ref
        v[spk] = reset
        if len(spk):
            idx = np.concatenate([np.arange(row[q], row[q + 1]) for q in spk])
            at = (t + d[idx]) % slots * n + tgt[idx]
            pos = w[idx] > 0
            np.add.at(exc.reshape(-1), at[pos], w[idx][pos])
            np.add.at(inh.reshape(-1), at[~pos], w[idx][~pos])
        exc[(t + case["d_lo"]) % slots] += w_drive * _poisson(rate * H * 1e-3, int(seed), streams, t)
    out = {"V_m": v + e_l}
    if "I_syn_ex" in fields:
        out["I_syn_ex"], out["I_syn_in"] = ie, ii
    return out
