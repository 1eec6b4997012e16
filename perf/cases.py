"""Workloads of the sparse FFT, through the package's public entry points.

A case is one call as a program makes it with a plan in hand: ``version`` 1,
2 or 3, the signal length ``n``, the sparsity ``k``, ``signals`` per call, the
``precision`` form and the ``call``:

  host    sfft.execute: one numpy signal in, the dense spectrum out as numpy
  dense   sfft.execute_device: one device signal, dense device spectrum
  sparse  sfft.execute_many_sparse: a batch of device signals, sparse results
  mix     ManyPlansCall: signals of several plans in one call (v3: n fixed,
          k, 5/2 k and 5 k in turn; v1/v2: the keys of ``MIX``)

``snr_db`` None is a noiseless signal; ``graphs`` replays captured HIP graphs.
Signals are k tones of unit amplitude at random frequencies and phases, plus
complex white noise of per-sample variance k * 10^(-snr_db / 10).
"""
import random

import numpy as np
import torch

import sfft_amd
from sfft_amd.sfft import ManyPlansCall, derive_params

# v1/v2 plans of uneven (n, k) served together (version, n, k)
MIX = [(2, 1 << 18, 10), (2, 1 << 18, 50), (2, 1 << 20, 20), (2, 1 << 20, 100),
       (2, 1 << 20, 300), (2, 1 << 22, 10), (2, 1 << 22, 64), (2, 1 << 22, 200),
       (1, 1 << 18, 20), (1, 1 << 20, 10), (1, 1 << 20, 50), (1, 1 << 22, 30)]


def _case(name, call, version, n, k, signals=1, precision="fp64", snr_db=None, graphs=False):
    c = {"call": call, "version": version, "n": n, "k": k, "signals": signals,
         "precision": precision, "snr_db": snr_db, "graphs": graphs}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the Python class as constructed by default, on a host array: the
        # smallest call a script makes
        _case("host_v1_n14", "host", 1, 1 << 14, 50),
        # one plain-v1 transform into a dense device spectrum
        _case("dense_v1_n20_k50", "dense", 1, 1 << 20, 50),
        # one noisy v2 transform in the reference's calling convention; k > 50
        # uses the default parameters, whose located set is large
        _case("dense_v2_n22_k100", "dense", 2, 1 << 22, 100, snr_db=30.0),
        # latency of one request in a serving loop: a replayed graph
        _case("one_v2_n22_k64", "sparse", 2, 1 << 22, 64, 1, "fp32_refine", 40.0, True),
        # the headline batch: throughput in the fast form
        _case("batch256_v2_n22_k64", "sparse", 2, 1 << 22, 64, 256, "fp32_refine", 40.0, True),
        # the same transform in batches where every bit has to be the reference's
        _case("batch64_v2_n22_fp64", "sparse", 2, 1 << 22, 64, 64, "fp64", 40.0),
        # long signals of few tones: small located sets, wide comb prefilter
        _case("batch4_v2_n24_k50", "sparse", 2, 1 << 24, 50, 4, "fp32_refine", 30.0),
        # the densest spectrum v2 accepts at this length: largest buckets and results
        _case("batch8_v2_n24_k1000", "sparse", 2, 1 << 24, 1000, 8, "fp32_refine", 40.0),
        # serving step of many small groups: 12 plans, 4 signals each
        _case("mix48_v12", "mix", 0, 1 << 22, 300, 48, "fp32_refine", 30.0),
        # one exactly sparse transform: the shortest v3 call
        _case("dense_v3_n20_k50", "dense", 3, 1 << 20, 50),
        # exactly sparse batch of uneven k, faithful and refined forms
        _case("mix64_v3_n24", "mix", 3, 1 << 24, 200, 64),
        _case("mix64_v3_n24_refine", "mix", 3, 1 << 24, 200, 64, "fp32_refine"),
    ]


def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    while True:
        call = rng.choice(["host", "dense", "sparse", "sparse", "sparse", "mix"])
        version = 3 if call == "mix" else rng.choice([1, 2, 2, 3])
        log_n = rng.randint(14, 20 if call == "host" else 24)
        n = 1 << log_n
        precision = rng.choice(["fp64", "fp32_refine"])
        signals = 1
        if call in ("sparse", "mix"):
            signals = int(_log_uniform(rng, 1, min(256, (1 << 27) // n) + 0.99))
        if version == 3:
            # sparse against n; the mix goes up to five times k
            hi = min(400 if call == "mix" else 2000, n >> 10)
            if hi < 10:
                continue
            return _case(None, call, 3, n, int(_log_uniform(rng, 10, hi)), signals, precision)
        k = int(_log_uniform(rng, 10, 2000))
        snr = rng.choice([None, 30.0, 40.0])
        ok, p = derive_params(n, k, version)
        if not ok:
            continue
        located = p["comb_loops"] * p["B_thresh"] * (n // p["W_comb"]) if version == 2 else 0
        if signals * located > (1 << 26):
            continue
        graphs = call == "sparse" and rng.random() < 0.5
        return _case(None, call, version, n, k, signals, precision, snr, graphs)


def _keys(case):
    """(version, n, k) of each signal of the call."""
    S = case["signals"]
    if case["call"] != "mix":
        return [(case["version"], case["n"], case["k"])] * S
    if case["version"] == 3:
        ks = [case["k"], case["k"] * 5 // 2, case["k"] * 5]
        return [(3, case["n"], ks[i % 3]) for i in range(S)]
    return [MIX[i * len(MIX) // S] for i in range(S)]


def _tones(n, k, seed):
    rng = random.Random(seed)
    return rng.sample(range(n), k), [2 * np.pi * rng.random() for _ in range(k)]


def _fill(x, k, seed, snr_db):
    """The signal of one seed into the device vector x."""
    n = x.numel()
    f, ph = _tones(n, k, seed)
    X = torch.zeros(n, dtype=torch.complex128, device=x.device)
    X[torch.tensor(f, device=x.device)] = torch.polar(
        torch.ones(k, dtype=torch.float64), torch.tensor(ph, dtype=torch.float64)).to(x.device)
    torch.fft.ifft(X, norm="forward", out=x)
    if snr_db is not None:
        g = torch.Generator(device=x.device)
        g.manual_seed(seed)
        x += torch.randn(n, dtype=torch.complex128, device=x.device, generator=g) * float(
            np.sqrt(k * 10.0 ** (-snr_db / 10.0)))


def prepare(case, seed):
    dev = torch.device("cuda")
    keys = _keys(case)
    plans = {}
    for key in keys:
        if key not in plans:
            v, n, k = key
            plans[key] = sfft_amd.sfft(n, k, v, strict=False, precision=case["precision"],
                                       seed=(seed % 1000003 + len(plans), seed % 999983))
    xs = []
    if case["call"] == "sparse":  # one array of signals, as a batch is usually held
        x = torch.empty((len(keys), case["n"]), dtype=torch.complex128, device=dev)
        xs = [x[i] for i in range(len(keys))]
    else:
        xs = [torch.empty(n, dtype=torch.complex128, device=dev) for _, n, _ in keys]
    for i, (_, n, k) in enumerate(keys):
        _fill(xs[i], k, seed * 4099 + i, case["snr_db"])
    plan = plans[keys[0]]
    state = {"call": case["call"], "plan": plan}
    if case["call"] == "host":
        state["x"] = xs[0].cpu().numpy()
    elif case["call"] == "dense":
        state["x"], state["out"] = xs[0], torch.empty_like(xs[0])
    elif case["call"] == "sparse":
        plan.enable_graphs(case["graphs"])
        freq, val = plan.make_sparse_outputs(len(keys))
        state.update(x=x, freq=freq.zero_(), val=val.zero_())
    else:
        caps = [plans[key].capacity for key in keys]
        freq = torch.zeros(sum(caps), dtype=torch.int32, device=dev)
        val = torch.zeros(sum(caps), dtype=torch.complex128, device=dev)
        outs = list(zip(freq.split(caps), val.split(caps)))
        state.update(many=ManyPlansCall([plans[key] for key in keys], xs, outs),
                     freq=freq, val=val)
    torch.cuda.synchronize()
    return state


def run(state):
    call = state["call"]
    if call == "host":
        return state["plan"].execute(state["x"])
    if call == "dense":
        return state["plan"].execute_device(state["x"], state["out"])
    if call == "sparse":
        counts = state["plan"].execute_many_sparse(state["x"], state["freq"], state["val"])
    else:
        counts = state["many"].call()
    return {"count": counts, "freq": state["freq"], "val": state["val"]}


def work(case):
    """Samples gathered (16 B each), results written (20 B per located
    coefficient, 16 B per entry of a dense spectrum); a complex
    multiply-add per tap, 5 N log2 N per transform, and per located
    coefficient and loop one complex quotient."""
    nbytes = flops = 0.0
    for v, n, k in _keys(case):
        p = derive_params(n, k, v)[1]
        if v == 3:
            W, B1, B2 = p["W_Man"], p["B_g1"], p["B_g2"]
            samples, located = 2 * W + p["w_g1"] + p["w_g2"], k
            if case["precision"] == "fp32_refine":
                samples += 8 * W
            flops += 8 * (p["w_g1"] + p["w_g2"]) + 10 * (
                W * np.log2(W) + B1 * np.log2(B1) + B2 * np.log2(B2))
        else:
            Ll, Le = p["loc_loops"], p["est_loops"]
            samples = Ll * p["w_loc"] + Le * p["w_est"]
            flops += 8 * samples + 5 * (Ll * p["B_loc"] * np.log2(p["B_loc"]) +
                                        Le * p["B_est"] * np.log2(p["B_est"]))
            located = k
            if v == 2:
                W = p["W_comb"]
                samples += p["comb_loops"] * W
                flops += 5 * p["comb_loops"] * W * np.log2(W)
                # several comb loops may name the same residue
                located = min(n, p["B_thresh"] * (n // W))
            flops += 8.0 * located * (Ll + Le)
        nbytes += 16.0 * samples
        nbytes += 16.0 * n if case["call"] in ("host", "dense") else 20.0 * located
    return {"bytes": nbytes, "flops": float(flops)}


def exact(case, seed):
    """The spectrum by construction, where the dense output is an estimate of
    it to rounding: noiseless v1 and v2 (whose values are conjugated).  With
    noise every located value carries its bucket's share of it, v3 may leave
    tones unresolved, and a sparse result's layout is the located set, which
    the algorithm's own draws decide."""
    if case["call"] not in ("host", "dense") or case["version"] == 3 or case["snr_db"] is not None:
        return None
    f, ph = _tones(case["n"], case["k"], seed * 4099)
    out = np.zeros(case["n"], np.complex128)
    out[f] = np.exp(-1j * np.asarray(ph))
    return out if case["call"] == "host" else torch.from_numpy(out)
