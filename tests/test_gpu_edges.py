"""The slice kernel at the sizes where its branches change, against the oracle.

- aeif_cond_exp blocks below, at and above the number of lane quads (a block's neurons are then
  taken from a pool, likely long updates first), several parameter sets in one block, slices of
  more than 64 steps, divisors that rule out the reciprocal division, Delta_T = 0;
- spike lists of more entries than are loaded with the counts, slices of more than one chunk of
  spikes, more blocks than threads (global delivery), blocks of one to 512 targets (the split of
  a target's bucket, the drive's thread groups);
- updates whose lags lie inside and outside the LDS window, and across a 64-lag word;
- results read between runs: two recorders and every state variable of a mixed network.

iaf models: identical spikes and bit-identical state. aeif_cond_exp: identical senders, times
within one step, states within 1e-6 relative (the repository's bar for that model).
"""

import numpy as np
import pytest

import nestgpu
import netbuild as nb

pytestmark = pytest.mark.gpu


def _spikes_equal(sr, o, exact=True):
    ev = sr.get("events")
    og, os_ = nb.sorted_spikes_oracle(o)
    print("spikes gpu=%d oracle=%d" % (len(ev["senders"]), len(og)), flush=True)
    assert len(og) > 0
    assert np.array_equal(ev["senders"], og)
    assert np.max(np.abs(ev["times"] - os_ * 0.1)) <= (1e-9 if exact else 0.1 + 1e-9)


def _run(desc, layout, fields, parts=None, exact=True):
    k, pops, sr = nb.build_gpu(desc, layout=layout)
    o, opops = nb.build_oracle(desc, portable_math=True)
    for t in parts or [desc["T"]]:
        k.Simulate(t)
        o.simulate(t)
    _spikes_equal(sr, o, exact)
    for p, op in zip(pops, opops):
        for f in fields:
            a, b = np.atleast_1d(p.get(f)), o.get(op, f)
            if exact:
                assert np.array_equal(a, b), "%s: max abs diff %g" % (f, np.max(np.abs(a - b)))
            else:
                assert np.max(np.abs(a - b) / np.maximum(np.abs(b), 1e-12)) <= 1e-6, f
    return k


AEIF_FIELDS = ("V_m", "g_ex", "g_in", "w")


@pytest.mark.parametrize("n, tb, delay", [(1, 0, 1.5), (127, 127, 1.5), (128, 128, 1.5), (129, 129, 1.5), (700, 512, 1.5),
                                          (300, 300, 7.0)])
def test_aeif_blocks(n, tb, delay):
    # delay 7.0: slices of 70 steps, two words of spike bits per neuron
    rng = np.random.default_rng(n)
    T = 60.0
    k = max(1, min(40, n // 4))
    desc = dict(n_vp=2, seed=17 + n, pops=[("aeif_cond_exp", n, dict(nb.AEIF_C4))], v0={0: rng.uniform(-70.6, -48.0, n)},
                conns=[((0, 0, n), (0, 0, n), "fixed_indegree", k, 1.5, delay)],
                drive=[(0, rng.poisson(2.0, size=(600, n)).astype(np.uint8), 6.0, delay)], T=T)
    _run(desc, {"targets_per_block": tb} if tb else {}, AEIF_FIELDS, exact=False)


@pytest.mark.parametrize("change", [{"tau_w": 1e201}, {"Delta_T": 0.0}, {"C_m": 120.0, "g_L": 12.0, "E_ex": 3.0}])
def test_aeif_parameter_sets_in_one_block(change):
    # two populations of one block with different parameters: the first pair of values changes
    # the division of the whole network, the second one's neurons have no spike current
    rng = np.random.default_rng(3)
    second = dict(nb.AEIF_C4, **change)
    if second.get("Delta_T") == 0.0:
        second["V_peak"] = -40.0
    desc = dict(n_vp=1, seed=5, pops=[("aeif_cond_exp", 90, dict(nb.AEIF_C4)), ("aeif_cond_exp", 70, second)],
                v0={0: rng.uniform(-70.6, -50.0, 90), 1: rng.uniform(-70.6, -52.0, 70)},
                conns=[((0, 0, 90), (1, 0, 70), "fixed_indegree", 10, 2.0, 1.5),
                       ((1, 0, 70), (0, 0, 90), "fixed_indegree", 10, -2.0, 1.5)],
                drive=[(0, rng.poisson(2.0, size=(600, 90)).astype(np.uint8), 6.0, 1.5),
                       (1, rng.poisson(2.0, size=(600, 70)).astype(np.uint8), 6.0, 1.5)], T=60.0)
    _run(desc, {"targets_per_block": 160}, AEIF_FIELDS, exact=False)


@pytest.mark.parametrize("change, quiet", [
    ({}, [(95, 1), (1, 170)]),  # conductances: denormal from 142 ms (0.2) and 248 ms (0.35) after the last input
    # w too (1 ms, driven by spikes only), and no spike current; V_m in a network that settles at 0
    ({"tau_w": 1.0, "a": 0.0}, [(95, 1), (1, 170), (380, 1), (1, 120)]),
    ({"Delta_T": 0.0, "E_L": 0.0, "V_reset": -10.0, "V_th": 12.0, "V_peak": 20.0, "E_ex": 60.0, "E_in": -20.0, "C_m": 30.0,
      "tau_w": 1.0, "a": 0.0}, [(95, 1), (1, 170), (380, 1), (1, 120)]),
])
def test_aeif_division_by_reciprocals_equals_plain_division(change, quiet):
    # a neuron without connections whose tau_w rules out the reciprocals makes the whole network
    # divide plainly: the other neurons' states keep every bit, down to denormal values
    rng = np.random.default_rng(12)
    n, T = 450, 40.0
    prm = dict(nb.AEIF_C4, tau_syn_ex=0.2, tau_syn_in=0.35, **change)
    lo, hi = prm.get("V_reset", -70.6), prm.get("V_th", -52.0)
    v0, counts = rng.uniform(lo, hi, n), rng.poisson(2.0, size=(int(T / 0.1), n)).astype(np.uint8)
    sims = []
    for tau_w in (144.0, 1e201):
        desc = dict(n_vp=1, seed=3, pops=[("aeif_cond_exp", n, prm), ("aeif_cond_exp", 1, dict(nb.AEIF_C4, tau_w=tau_w))],
                    v0={0: v0}, conns=[((0, 0, 360), (0, 0, n), "fixed_indegree", 10, 2.0, 1.5),
                                       ((0, 360, n), (0, 0, n), "fixed_indegree", 10, -2.0, 1.5)],
                    drive=[(0, counts, 6.0, 1.5)], T=T)
        sims.append(nb.build_gpu(desc, layout={"targets_per_block": n + 1}))
    smallest = 1.0
    at = 0.0
    for t in [T] + [float(t) for step, count in quiet for t in [step] * count]:
        at += t
        state = []
        for k, pops, sr in sims:
            k.Simulate(t)
            state.append({f: pops[0].get(f) for f in AEIF_FIELDS})
        for f in AEIF_FIELDS:
            a, b = state[0][f], state[1][f]
            bad = np.flatnonzero(a.view(np.uint64) != b.view(np.uint64))
            assert len(bad) == 0, "%g ms, %s: %d of %d differ, first %r, plain %r" % (at, f, len(bad), n, a[bad[0]], b[bad[0]])
            if np.any(a != 0.0):
                smallest = min(smallest, np.min(np.abs(a[a != 0.0])))
    ev = [sr.get("events") for _, _, sr in sims]
    assert np.array_equal(ev[0]["senders"], ev[1]["senders"]) and np.array_equal(ev[0]["times"], ev[1]["times"])
    print("spikes %d, smallest state value %g" % (len(ev[0]["senders"]), smallest), flush=True)
    assert len(ev[0]["senders"]) > 100 and smallest < 2.0 ** -1022


@pytest.mark.parametrize("layout", [{"targets_per_block": 1, "delivery_mode": "global"}, {"targets_per_block": 5},
                                    {"targets_per_block": 64}, {"targets_per_block": 65}, {"targets_per_block": 257},
                                    {"targets_per_block": 512}, {"targets_per_block": 2, "delivery_mode": "global"}],
                         ids=lambda x: "%s%d" % (x.get("delivery_mode", "auto"), x["targets_per_block"]))
def test_block_sizes(layout):
    # 1 and 2 targets per block: more blocks than threads; 257 and 512: no room for a drive group
    n = 1100 if layout["targets_per_block"] > 2 else 1030
    _run(nb.exp_random(N=n, KE=40, KI=10, T=40.0, seed=layout["targets_per_block"]), layout,
         ("V_m", "I_syn_ex", "I_syn_in"))


@pytest.mark.parametrize("layout", [{"targets_per_block": 512}, {"targets_per_block": 160, "delivery_mode": "global"}, {}],
                         ids=["win512", "global160", "auto"])
def test_many_spikes_per_slice(layout):
    # every neuron spikes every few steps: lists of hundreds of entries and several chunks of
    # spikes in a slice of 20 steps
    n, T = 1500, 30.0
    rng = np.random.default_rng(8)
    params = {"C_m": 1.0, "tau_m": 20.0, "V_th": 20.0, "V_reset": 10.0, "E_L": 0.0, "t_ref": 0.2}
    desc = dict(n_vp=3, seed=4, pops=[("iaf_psc_delta", n, params)], v0={0: rng.uniform(0, 20, n)},
                conns=[((0, 0, n), (0, 0, n), "fixed_indegree", 20, ("normal", 0.05, 0.2), ("uniform", 2.0, 3.0))],
                drive=[(0, rng.poisson(8.0, size=(300, n)).astype(np.uint8), 0.8, 2.0)], T=T)
    _run(desc, layout, ("V_m",))


def _volleys(n, of, T):
    # every slice (15 steps) the first `of` neurons of each half spike
    params = {"C_m": 1.0, "tau_m": 20.0, "V_th": 20.0, "V_reset": 10.0, "E_L": 0.0, "t_ref": 1.0}
    counts = np.zeros((int(round(T / 0.1)), n), np.uint8)
    for first in (0, n // 2):
        counts[::15, first:first + of] = 1
    return dict(n_vp=1, seed=6, pops=[("iaf_psc_delta", n, params)], v0={0: np.random.default_rng(n).uniform(0, 10, n)},
                conns=[((0, 0, n), (0, 0, n), "fixed_indegree", 20, ("normal", 0.001, 0.1), 1.5)],
                drive=[(0, counts, 40.0, 1.5)], T=T)


@pytest.mark.parametrize("of", [3, 4, 5, 16, 17, 100, 511, 512])
def test_spike_lists_of_one_length(of):
    # lists that come with the counts, that one thread copies and that are looked up
    _run(_volleys(1024, of, 15.0), {"targets_per_block": 512}, ("V_m",))


def test_long_spike_lists_cost_what_many_spikes_cost():
    # 1,000 spikes per slice in two lists, and 1,030 (in three), which are more than a chunk: a thread that
    # copied a list of 500 entries made the smaller number the slower one (60 %)
    import time

    sims = [nb.build_gpu(_volleys(n, n // 2, 600.0), layout={"targets_per_block": 512}) for n in (1000, 1030)]
    took = [[], []]
    for i in range(10):
        for (k, _, _), t in zip(sims, took):
            if i == 0:
                k.Prepare()
            at = time.perf_counter()
            k.Run(60.0)
            t.append(time.perf_counter() - at)
    us = [sorted(t[2:])[4] / 40 * 1e6 for t in took]
    print("us per slice: %.1f (1,000 spikes), %.1f (1,030)" % tuple(us), flush=True)
    assert us[0] < 1.15 * us[1]


@pytest.mark.parametrize("model, fields", [("iaf_psc_exp", ("V_m", "I_syn_ex", "I_syn_in")),
                                           ("iaf_psc_alpha", ("V_m", "I_syn_ex", "I_syn_in")), ("iaf_psc_delta", ("V_m",))])
@pytest.mark.parametrize("delay, slots", [(7.0, 0), (7.0, 20), (0.1, 0)])
def test_update_inside_and_outside_the_window(model, fields, delay, slots):
    # delay 7.0: slices of 70 steps (two words of lags), all or 20 of their slots in LDS; parts
    # that end inside a slice
    n = 260
    rng = np.random.default_rng(6)
    params = {"tau_m": 10.0, "C_m": 250.0, "V_th": -55.0, "V_reset": -70.0, "t_ref": 2.0, "E_L": -70.0}
    w = 90.0
    if model == "iaf_psc_delta":
        params, w = {"C_m": 1.0, "tau_m": 20.0, "V_th": 20.0, "V_reset": 10.0, "E_L": 0.0, "t_ref": 2.0}, 0.3
    else:
        params.update(tau_syn_ex=0.5, tau_syn_in=0.5)
    lo, hi = (params["V_reset"], params["V_th"])
    desc = dict(n_vp=2, seed=31, pops=[(model, n, params)], v0={0: rng.uniform(lo, hi, n)},
                conns=[((0, 0, n), (0, 0, n), "fixed_indegree", 20, ("normal", w, 0.1 * w), ("uniform", delay, delay + 2.0))],
                drive=[(0, rng.poisson(1.5, size=(420, n)).astype(np.uint8), w, delay)], T=42.0)
    _run(desc, {"window_slots": slots} if slots else {}, fields, parts=[10.3, 7.0, 24.7])


@pytest.mark.parametrize("model", ["iaf_psc_exp", "iaf_psc_alpha", "iaf_psc_delta"])
@pytest.mark.parametrize("layout", [{"delivery_mode": "global"}, {"window_slots": 20}, {}])
def test_update_of_four_words_of_lags(model, layout):
    # slices of 250 steps in parts that start at odd lags: groups of lags cross all three words
    n = 200
    rng = np.random.default_rng(9)
    params = {"tau_m": 10.0, "C_m": 250.0, "V_th": -55.0, "V_reset": -70.0, "t_ref": 0.2, "E_L": -70.0}
    w = 200.0
    if model == "iaf_psc_delta":
        params, w = {"C_m": 1.0, "tau_m": 20.0, "V_th": 20.0, "V_reset": 10.0, "E_L": 0.0, "t_ref": 0.2}, 1.5
    else:
        params.update(tau_syn_ex=0.5, tau_syn_in=0.5)
    desc = dict(n_vp=2, seed=37, pops=[(model, n, params)], v0={0: rng.uniform(params["V_reset"], params["V_th"], n)},
                conns=[((0, 0, n), (0, 0, n), "fixed_indegree", 10, ("normal", w, 0.1 * w), ("uniform", 25.0, 27.0))],
                drive=[(0, rng.poisson(2.0, size=(900, n)).astype(np.uint8), w, 25.0)], T=90.0)
    fields = ("V_m",) if model == "iaf_psc_delta" else ("V_m", "I_syn_ex", "I_syn_in")
    _run(desc, layout, fields, parts=[5.9, 24.1, 60.0])


def test_results_read_between_runs():
    # two recorders on parts of a mixed network, read after every run, and all state variables
    desc = nb.mixed_models(T=60.0)
    k, pops, sr = nb.build_gpu(desc)
    few = k.Create("spike_recorder")
    k.Connect(pops[1][10:60], few)
    o, opops = nb.build_oracle(desc, portable_math=True)
    ids = set(pops[1][10:60].tolist())
    for t in (7.3, 20.0, 0.4, 32.3):
        k.Simulate(t)
        o.simulate(t)
        og, os_ = nb.sorted_spikes_oracle(o)
        keep = np.isin(og, list(ids))
        for rec, g, s in ((sr, og, os_), (few, og[keep], os_[keep])):
            ev = rec.get("events")
            assert rec.get("n_events") == len(g) == len(ev["senders"])
            assert np.array_equal(ev["senders"], g)
        for p, op in zip(pops[:2], opops[:2]):
            assert np.array_equal(np.atleast_1d(p.get("V_m")), o.get(op, "V_m"))
        assert np.array_equal(pops[1].get("I_syn_in"), o.get(opops[1], "I_syn_in"))
        everyone = (pops[2] + pops[0]).get("V_m")
        assert np.array_equal(everyone[len(pops[2]):], np.atleast_1d(pops[0].get("V_m")))
        w = o.get(opops[2], "w")
        assert np.max(np.abs(pops[2].get("w") - w) / np.maximum(np.abs(w), 1e-12)) <= 1e-6
