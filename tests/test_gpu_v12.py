"""GPU parity of the sFFT v1/v2 path against the CPU oracle, through the C ABI.

Two levels:
  * bit-exact: the oracle runs with the library's own filter taps, so every
    later step (comb, fold, FFT, selection, votes, median estimation) must
    agree bit for bit with the GPU FP64 form;
  * independent: the oracle designs its own filters; located sets must be
    identical and values within 1e-9 relative (filter designs agree to
    ~1e-12).
The FP32+refine form must give the identical located set and values within
1e-6 of the FP64 form.
"""
import numpy as np
import pytest

import oracle
import sfft_amd
from sfft_amd.signals import signal_np

pytestmark = pytest.mark.gpu

# (version, n, k, snr_db)
CASES = [
    (1, 1 << 14, 50, None),
    (2, 1 << 14, 50, None),
    (1, 1 << 16, 50, None),
    (2, 1 << 16, 50, None),
    (1, 1 << 20, 50, None),     # v1 at the noiseless n=2^20, k=50 workload
    (2, 1 << 22, 64, 40.0),     # one signal of the batched n=2^22, k=64 workload
    (2, 1 << 22, 100, 30.0),    # v2 n=2^22, k=100, SNR 30 dB
    (1, 1 << 18, 300, 20.0),    # v1 on the default parameters (k > 50)
]

# Transforms and selections above one workgroup's LDS: bucket FFTs as LDS
# radix-2 runs plus global passes, comb FFTs likewise, v1 selection over an
# HBM scratch array.
LARGE = [
    (1, 1 << 22, 1500, 30.0),   # B = 16384: one global pass (FP64)
    (1, 1 << 24, 2000, 30.0),   # B = 32768: two passes, selection in HBM
    (1, 1 << 24, 50, None),     # B_loc = 16384, B_est = 1024
    (2, 1 << 24, 10, 30.0),     # W_comb = 2^18: comb FFT with five passes
    (2, 1 << 24, 1000, 30.0),   # v2 with B = 16384 (the comb prefill
                                # locates 2000 * n/W = every frequency)
]


def _gpu_plan(version, n, k, precision="fp64"):
    return sfft_amd.sfft(n, k, version, strict=False, precision=precision,
                         seed=(17, 4242))


def _oracle_run(version, n, k, x, filters=None):
    oracle.seed_glibc(17, 4242)
    P = oracle.V12(n, k, version == 2)
    if filters is not None:
        P.set_filters(*filters)
    a, ai, off = P.draw()
    return P.exec(x, a, ai, off, trace=True)


def _plan_filters(plan):
    """The taps and responses the plan itself uses (for the oracle)."""
    lt, lf = plan.filter(0)
    et, ef = plan.filter(1)
    return lt, lf, et, ef


def _located(ref, version):
    if version == 2:
        return np.unique(ref["hits"][:ref["hits_prefill"]])
    return np.unique(ref["hits"])


def _run_gpu_dense(torch, plan, x):
    xd = torch.from_numpy(x).cuda()
    od = torch.empty_like(xd)
    plan.execute_device(xd, od)
    torch.cuda.synchronize()
    return od.cpu().numpy()


@pytest.mark.parametrize("version,n,k,snr", CASES + LARGE)
def test_fp64_bit_exact_given_filters(torch_cuda, version, n, k, snr):
    print(f"case v{version} n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=1000 + n % 97 + k, snr_db=snr)
    plan = _gpu_plan(version, n, k)
    ref = _oracle_run(version, n, k, x, _plan_filters(plan))
    out = _run_gpu_dense(torch_cuda, plan, x)
    loc_ref = _located(ref, version)
    loc_gpu = np.nonzero(out)[0]
    assert np.array_equal(loc_gpu, loc_ref), (len(loc_gpu), len(loc_ref))
    diff = np.abs(out - ref["out"]).max()
    assert diff == 0.0, diff


@pytest.mark.parametrize("version,n,k,snr", CASES + LARGE[:4])
def test_fp64_buckets_bit_exact_given_filters(torch_cuda, version, n, k, snr):
    """Fold + bucket FFT output of every loop equals the oracle's x_samp."""
    print(f"case v{version} n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=4000 + k, snr_db=snr)
    plan = _gpu_plan(version, n, k)
    ref = _oracle_run(version, n, k, x, _plan_filters(plan))
    plan.execute_sparse_host(x)
    got = plan.debug_buckets(0)
    assert len(got) == len(ref["x_samp"])
    assert np.abs(got - ref["x_samp"]).max() == 0.0


@pytest.mark.parametrize("version,n,k,snr", CASES)
def test_fp64_parity_independent_oracle(torch_cuda, version, n, k, snr):
    print(f"case v{version} n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=2000 + k, snr_db=snr)
    ref = _oracle_run(version, n, k, x)
    plan = _gpu_plan(version, n, k)
    fr, va = plan.execute_sparse_host(x)
    loc_ref = _located(ref, version)
    assert np.array_equal(np.unique(fr), loc_ref)
    # values: norm-wise within 1e-9 of the largest coefficient (leakage-level
    # values carry the ~1e-12 difference of the two filter designs), and
    # every coefficient above 0.1 within 1e-9 relative
    refv = ref["out"][fr]
    diff = np.abs(va - refv)
    assert diff.max() <= 1e-9 * np.abs(refv).max(), diff.max()
    big = np.abs(refv) > 0.1
    assert (diff[big] / np.abs(refv[big])).max(initial=0.0) <= 1e-9
    # every true tone is located and equals conj(X) (reference semantics)
    if snr is None:
        assert np.all(np.isin(f, fr))
        got = dict(zip(fr.tolist(), va.tolist()))
        err = max(abs(got[int(ff)] - np.conj(vv)) for ff, vv in zip(f, v))
        assert err < 1e-6, err


@pytest.mark.parametrize("version,n,k,snr",
                         [c for c in CASES if c[1] >= 1 << 16] + LARGE[:4])
def test_fp32_refine_matches_fp64(torch_cuda, version, n, k, snr):
    print(f"case v{version} n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=3000 + k, snr_db=snr)
    p64 = _gpu_plan(version, n, k)
    p32 = _gpu_plan(version, n, k, precision="fp32_refine")
    f64, v64 = p64.execute_sparse_host(x)
    f32, v32 = p32.execute_sparse_host(x)
    # v2 locates through the FP64 comb and v1 keeps its location loops in
    # FP64, so the located sets are identical in both forms
    assert np.array_equal(f32, f64)
    err = np.abs(v32 - v64)
    assert err.max() <= 1e-6, err.max()


@pytest.mark.parametrize("version,n,k,snr", [
    (2, 1 << 16, 50, None),      # 128 rows: one chunk (plain ascending tap order)
    (2, 1 << 22, 64, 40.0),      # 2048 rows: eight chunks of 256
    (1, 1 << 20, 50, None),      # v1: FP32 estimation loops only (B_est = 512)
    (2, 1 << 20, 64, 30.0),
    (1, 1 << 24, 50, None),      # B_est = 1024: 64 chunks
])
def test_fp32_buckets_bit_exact_model(torch_cuda, version, n, k, snr):
    """The FP32 form's buckets after the bucket FFTs equal, bit for bit, the
    model of its summation order (oracle/fp32_model.c) on the plan's taps
    and draws."""
    print(f"case fp32 buckets v{version} n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=4300 + k, snr_db=snr)
    plan = _gpu_plan(version, n, k, precision="fp32_refine")
    plan.execute_sparse_host(x)
    got = plan.debug_buckets(0)
    p = dict(zip(["B_loc", "B_est", "B_thresh", "W_comb", "comb_loops", "loc_loops",
                  "est_loops", "thr_loops", "w_loc", "w_est"], plan.params()))
    L, Lloc = p["loc_loops"] + p["est_loops"], p["loc_loops"]
    oracle.seed_glibc(17, 4242)
    a, ai, off = oracle.v12_draws(n, L, p["comb_loops"] if version == 2 else 0, p["W_comb"])
    nmax = max(p["B_loc"], p["B_est"], p["W_comb"] if version == 2 else 0)
    lt, _ = plan.filter(0)
    et, _ = plan.filter(1)
    first32 = 0 if version == 2 else Lloc  # v1 keeps its location loops in FP64
    off_l = 0
    for l in range(L):
        B = p["B_loc"] if l < Lloc else p["B_est"]
        if l >= first32:
            want = oracle.fp32_buckets(x, n, B, lt if l < Lloc else et, ai[l], 256, nmax)
            assert np.array_equal(got[off_l:off_l + B], want), (l, np.abs(got[off_l:off_l + B] - want).max())
        off_l += B


@pytest.mark.parametrize("version", [1, 2])
def test_batch_equals_single(torch_cuda, version):
    """exec_many of a batch gives each signal the same result as alone,
    when the RNG draws are replayed in signal order."""
    torch = torch_cuda
    n, k = 1 << 18, 64
    xs = [signal_np(n, k, seed=s, snr_db=30.0)[0] for s in range(6)]
    plan = _gpu_plan(version, n, k)
    xd = [torch.from_numpy(x).cuda() for x in xs]
    fr, va = plan.make_sparse_outputs(len(xs))
    counts = plan.execute_many_sparse(xd, fr, va)
    torch.cuda.synchronize()
    single = _gpu_plan(version, n, k)
    for i, x in enumerate(xs):
        f1, v1 = single.execute_sparse_host(x)
        c = counts[i]
        assert c == len(f1)
        assert np.array_equal(fr[i, :c].cpu().numpy(), f1)
        assert np.abs(va[i, :c].cpu().numpy() - v1).max() == 0.0


@pytest.mark.parametrize("version", [1, 2])
def test_host_pointers_dense(torch_cuda, version):
    """sfft_exec with host in/out (the reference's own calling convention):
    the dense, zero-filled output equals the oracle's bit for bit."""
    n, k = 1 << 16, 50
    x, f, v = signal_np(n, k, seed=5)
    plan = sfft_amd.sfft(n, k, version, seed=(17, 4242))
    out = plan.execute(x)
    ref = _oracle_run(version, n, k, x, _plan_filters(plan))
    assert np.array_equal(out, ref["out"])


def test_host_pointers_dense_v3(torch_cuda):
    """v3 through sfft_exec with host in/out: the oracle's located
    frequencies carry its values, every other entry is zero."""
    n, k = 1 << 18, 100
    x, f, v = signal_np(n, k, seed=6)
    plan = sfft_amd.sfft(n, k, 3, seed=(17, 4242))
    t1, f1 = plan.filter(0)
    t2, f2 = plan.filter(1)
    oracle.seed_glibc(17, 4242)
    P = oracle.V3(n, k)
    P.set_filters(t1, f1, t2, f2)
    ref = P.exec(x, P.draw())
    out = plan.execute(x)
    if ref["early"]:
        assert not np.any(out)
        return
    assert np.array_equal(np.nonzero(out)[0], np.sort(ref["freqs"][ref["vals"] != 0]))
    assert np.abs(out[ref["freqs"]] - ref["vals"]).max() <= 1e-9 * np.abs(ref["vals"]).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32_refine"])
@pytest.mark.parametrize("version,n,k,snr", [(2, 1 << 20, 64, 30.0), (1, 1 << 18, 100, 30.0)])
def test_schedules_give_identical_results(torch_cuda, version, n, k, snr, precision):
    """Fused and streamed folds (any resident-block count) sum every bucket
    in the same tap order, and the alias-row bucket layout (schedule 1, v2
    FP32) feeds estimation the same products: identical bits."""
    print(f"case v{version} n={n} k={k} {precision}", flush=True)
    x, f, v = signal_np(n, k, seed=6000 + k, snr_db=snr)
    res = []
    for mode, blocks in [(0, 0), (1, 0), (1, 96), (1, 1024), (2, 0)]:
        plan = _gpu_plan(version, n, k, precision)
        plan.set_schedule(mode, blocks)
        assert plan.schedule() == (mode, blocks)
        res.append(plan.execute_sparse_host(x))
    for fr, va in res[1:]:
        assert np.array_equal(fr, res[0][0])
        assert np.array_equal(va, res[0][1])


@pytest.mark.parametrize("precision", ["fp64", "fp32_refine"])
def test_unconjugated_values(torch_cuda, precision):
    """With the reference's conjugation undone, every schedule (the alias-row
    estimation of schedule 1 and the natural-order one of schedule 2) gives
    the same bits, the located set and the real parts are the conjugated
    form's, and each tone's value is the conjugate of the default one up to
    the choice between the two middle estimates of its imaginary part."""
    n, k = 1 << 20, 64
    print(f"case v2 n={n} k={k} {precision} unconjugated", flush=True)
    x, f, v = signal_np(n, k, seed=6100, snr_db=30.0)
    base = _gpu_plan(2, n, k, precision).execute_sparse_host(x)
    res = []
    for mode in (1, 2):
        plan = _gpu_plan(2, n, k, precision)
        plan.set_reference_conjugate(False)
        plan.set_schedule(mode, 0)
        res.append(plan.execute_sparse_host(x))
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])
    fr, va = res[0]
    assert np.array_equal(fr, base[0])
    assert np.array_equal(va.real, base[1].real)
    tone = np.isin(fr, f)
    assert tone.sum() == k
    assert np.abs(va[tone] - np.conj(base[1][tone])).max() < 0.05


def test_autotune_keeps_draws_and_results(torch_cuda):
    n, k = 1 << 20, 64
    x, f, v = signal_np(n, k, seed=77, snr_db=30.0)
    tuned = _gpu_plan(2, n, k, "fp32_refine")
    mode, blocks = tuned.autotune(batch=8)
    assert mode in (0, 1, 2) and blocks >= 0
    fresh = _gpu_plan(2, n, k, "fp32_refine")
    a = tuned.execute_sparse_host(x)
    b = fresh.execute_sparse_host(x)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("version,n,k,snr,precision", [
    (2, 1 << 20, 64, 30.0, "fp32_refine"), (1, 1 << 18, 100, 30.0, "fp64")])
def test_graph_replays_match_eager(torch_cuda, version, n, k, snr, precision):
    """Replays of the captured batch (new signals and new draws each time,
    eager torch work in between) equal the eager execs exactly."""
    torch = torch_cuda
    print(f"case graphs v{version} n={n} k={k} {precision}", flush=True)
    g = _gpu_plan(version, n, k, precision)
    g.enable_graphs(True)
    e = _gpu_plan(version, n, k, precision)
    for rep in range(4):
        xs = [torch.from_numpy(signal_np(n, k, seed=700 + 3 * rep + i, snr_db=snr)[0]).cuda()
              for i in range(3)]
        fg, vg = g.make_sparse_outputs(3)
        fe, ve = e.make_sparse_outputs(3)
        cg = g.execute_many_sparse(xs, fg, vg)
        _ = torch.stack(xs).abs().sum().item()   # eager work between replays
        ce = e.execute_many_sparse(xs, fe, ve)
        torch.cuda.synchronize()
        assert np.array_equal(cg, ce)
        for i in range(3):
            c = int(ce[i])
            assert torch.equal(fg[i, :c], fe[i, :c])
            assert torch.equal(vg[i, :c], ve[i, :c])


@pytest.mark.parametrize("version,n,k,snr", [(1, 1 << 18, 100, 30.0), (2, 1 << 20, 64, 30.0)])
def test_stage_timing_keeps_results(torch_cuda, version, n, k, snr):
    """Per-stage HIP-event timing: the stages that ran report time, and the
    timed execs give the untimed results."""
    print(f"case timing v{version} n={n} k={k}", flush=True)
    x, f, v = signal_np(n, k, seed=4100 + k, snr_db=snr)
    plain = _gpu_plan(version, n, k)
    timed = _gpu_plan(version, n, k)
    timed.enable_timing(True)
    for _ in range(3):
        a = plain.execute_sparse_host(x)
        b = timed.execute_sparse_host(x)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    st = timed.stage_times()
    timed.enable_timing(False)
    ran = ["fold", "estimate"] + (["select_vote"] if version == 1 else ["comb"])
    for name in ran:
        assert st[name][1] > 0 and st[name][0] > 0, (name, st)


@pytest.mark.parametrize("precision", ["fp64", "fp32_refine"])
def test_large_batch_tiles_equal_single(torch_cuda, precision):
    """A batch large enough for the wide estimation tiles (16 signals of
    n=2^22, k=64) gives every signal the bits it gets alone, where the
    narrow tiles run."""
    torch = torch_cuda
    from sfft_amd.signals import signals_device
    n, k, S = 1 << 22, 64, 16
    print(f"case wide tiles n={n} k={k} S={S} {precision}", flush=True)
    x, _, _ = signals_device(n, k, list(range(500, 500 + S)), snr_db=40.0)
    batch = _gpu_plan(2, n, k, precision)
    fr, va = batch.make_sparse_outputs(S)
    counts = batch.execute_many_sparse(x, fr, va)
    single = _gpu_plan(2, n, k, precision)
    f1, v1 = single.make_sparse_outputs(1)
    for i in range(S):
        c1 = single.execute_many_sparse(x[i:i + 1], f1, v1)
        torch.cuda.synchronize()
        c = int(counts[i])
        assert int(c1[0]) == c
        assert torch.equal(fr[i, :c], f1[0, :c])
        assert torch.equal(va[i, :c], v1[0, :c])
    del x
    torch.cuda.empty_cache()


def test_concurrent_calls_on_one_plan(torch_cuda):
    """Two host threads calling one plan take turns: each call gets the
    draws of one of the two sequential calls, and together they get both."""
    import threading
    torch = torch_cuda
    n, k = 1 << 18, 64
    x, f, v = signal_np(n, k, seed=2500, snr_db=30.0)
    seq = _gpu_plan(2, n, k)
    ref = [seq.execute_sparse_host(x) for _ in range(2)]
    shared = _gpu_plan(2, n, k)
    got = [None, None]

    def call(i):
        got[i] = shared.execute_sparse_host(x)
    ths = [threading.Thread(target=call, args=(i,)) for i in range(2)]
    [t.start() for t in ths]
    [t.join() for t in ths]
    torch.cuda.synchronize()

    def same(a, b):
        return np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    match = [[same(g, r) for r in ref] for g in got]
    assert (match[0][0] and match[1][1]) or (match[0][1] and match[1][0]), match


@pytest.mark.parametrize("n,k,snr", [(1 << 14, 50, None), (1 << 16, 50, 20.0),
                                     (1 << 20, 50, 30.0), (1 << 22, 64, 40.0)])
def test_v2_comb_votes_match_oracle(torch_cuda, n, k, snr):
    """The v2 location votes (skipped by the exec: they never change the
    output), counted on the GPU on demand, append the oracle's hits in the
    oracle's order (hits after the comb prefill; src/computefourier-1.0-2.0.cc
    125-184), and the output is unchanged by counting them."""
    print(f"case comb votes n={n} k={k} snr={snr}", flush=True)
    x, f, v = signal_np(n, k, seed=8800 + k, snr_db=snr)
    plan = _gpu_plan(2, n, k)
    plain = _gpu_plan(2, n, k)
    plan.debug_comb_votes(True)
    fr, va = plan.execute_sparse_host(x)
    f0, v0 = plain.execute_sparse_host(x)
    assert np.array_equal(fr, f0) and np.array_equal(va, v0)
    got = plan.comb_votes(0)
    ref = _oracle_run(2, n, k, x, _plan_filters(plan))
    appended = ref["hits"][ref["hits_prefill"]:ref["hits_found"]]
    assert ref["hits_found"] - ref["hits_prefill"] == len(got)
    assert np.array_equal(got, appended)
    # every appended frequency duplicates a prefill entry
    assert np.all(np.isin(appended, ref["hits"][:ref["hits_prefill"]]))


@pytest.mark.parametrize("precision", ["fp64", "fp32_refine"])
def test_many_plans_v12_mix_equals_alone(torch_cuda, precision):
    """sfft_exec_many_plans over v1/v2 plans of different (n, k), plus a v3
    plan, interleaved: the v1/v2 groups are enqueued back to back and
    waited for together, and every signal equals its plan's alone run
    (each plan draws for its own signals in order)."""
    torch = torch_cuda
    from sfft_amd.sfft import execute_many_plans
    keys = [(2, 1 << 18, 50), (1, 1 << 18, 20), (2, 1 << 20, 100), (3, 1 << 18, 100),
            (2, 1 << 16, 10)]
    order = [0, 1, 2, 3, 4, 2, 1, 0, 4, 3, 2]
    xs = [torch.from_numpy(signal_np(keys[g][1], keys[g][2], seed=700 + i,
                                     snr_db=None if keys[g][0] == 3 else 30.0)[0]).cuda()
          for i, g in enumerate(order)]

    def plan(g):
        v, n, k = keys[g]
        return sfft_amd.sfft(n, k, v, strict=False, precision=precision,
                             seed=(61 + g, 4242 + g))
    plans = [plan(g) for g in range(len(keys))]
    res = execute_many_plans([plans[g] for g in order], xs)
    torch.cuda.synchronize()
    for g, (v, n, k) in enumerate(keys):
        alone = plan(g)
        idx = [i for i, gg in enumerate(order) if gg == g]
        fr, va = alone.make_sparse_outputs(len(idx))
        counts = alone.execute_many_sparse([xs[i] for i in idx], fr, va)
        torch.cuda.synchronize()
        for j, i in enumerate(idx):
            print(f"case many-plans {precision} v{v} n={n} k={k} signal {i}", flush=True)
            c = int(counts[j])
            assert c > 0 and int(res[i][0].numel()) == c
            assert torch.equal(res[i][0], fr[j, :c])
            assert torch.equal(res[i][1], va[j, :c])


@pytest.mark.parametrize("graphs", [False, True])
def test_parted_batch_equals_single(torch_cuda, graphs):
    """A v2 FP32 batch of 97 signals of n=2^22, k=64 runs in two uneven
    parts (48 + 49: the fold and bucket FFTs of one part beside the
    estimation of the previous one, on two streams, eagerly or replayed from
    a HIP graph); every signal gets the bits it gets alone (a single signal
    runs unparted)."""
    torch = torch_cuda
    from sfft_amd.signals import signals_device
    n, k, S = 1 << 22, 64, 97
    print(f"case parted batch n={n} k={k} S={S} graphs={graphs}", flush=True)
    x, _, _ = signals_device(n, k, list(range(700, 700 + S)), snr_db=40.0)
    batch = _gpu_plan(2, n, k, "fp32_refine")
    batch.enable_graphs(graphs)
    fr, va = batch.make_sparse_outputs(S)
    for rep in range(2 if graphs else 1):   # capture, then a replay
        batch.seed(17, 4242)
        counts = batch.execute_many_sparse(x, fr, va)
        torch.cuda.synchronize()
    single = _gpu_plan(2, n, k, "fp32_refine")
    f1, v1 = single.make_sparse_outputs(1)
    for i in range(S):
        c1 = single.execute_many_sparse(x[i:i + 1], f1, v1)
        torch.cuda.synchronize()
        c = int(counts[i])
        assert int(c1[0]) == c
        assert torch.equal(fr[i, :c], f1[0, :c])
        assert torch.equal(va[i, :c], v1[0, :c])
    del x
    torch.cuda.empty_cache()


# Edges of the sorted fold: few residues (B below a workgroup's), the widest
# spectrum of rows (chunk lists of several passes), 8 and 16 residues per
# workgroup, location and estimation loops of different bucket counts.
SORTED = [
    (2, 1 << 13, 50, 1),    # 23 loops, 32 rows of 256 buckets
    (1, 1 << 14, 50, 3),
    (2, 1 << 24, 10, 1),    # 16,384 and 32,768 rows: up to three list passes
    (2, 1 << 23, 50, 1),    # B_loc != B_est
    (1, 1 << 22, 30, 2),    # v1: FP64 and FP32 loops of one launch
    (2, 1 << 20, 300, 9),   # 16 residues per workgroup
]


@pytest.mark.parametrize("version,n,k,signals", SORTED)
def test_sorted_fold_buckets(torch_cuda, version, n, k, signals):
    """The last signal's buckets of a batch equal the oracle's bit for bit
    (FP64 form) and the model of the FP32 form's summation order."""
    torch = torch_cuda
    print(f"case sorted fold v{version} n={n} k={k} x{signals}", flush=True)
    xs = [signal_np(n, k, seed=8800 + i, snr_db=30.0)[0] for i in range(signals)]
    xd = [torch.from_numpy(x).cuda() for x in xs]
    for precision in ("fp64", "fp32_refine"):
        plan = _gpu_plan(version, n, k, precision)
        fr, va = plan.make_sparse_outputs(signals)
        plan.execute_many_sparse(xd, fr, va)
        got = plan.debug_buckets(signals - 1)
        lt, lf = plan.filter(0)
        et, ef = plan.filter(1)
        P = oracle.V12(n, k, version == 2)
        P.set_filters(lt, lf, et, ef)
        oracle.seed_glibc(17, 4242)
        for _ in range(signals):
            a, ai, off = P.draw()
        ref = P.exec(xs[-1], a, ai, off, trace=True)["x_samp"]
        p = P.p
        nmax = max(p.B_loc, p.B_est, p.W_comb if version == 2 else 0)
        at = 0
        for l in range(P.loops):
            loc = l < p.loc_loops
            B = p.B_loc if loc else p.B_est
            want = ref[at:at + B]
            if precision == "fp32_refine" and not (version == 1 and loc):
                want = oracle.fp32_buckets(xs[-1], n, B, lt if loc else et, ai[l], 256, nmax)
            assert np.array_equal(got[at:at + B], want), (precision, l)
            at += B


@pytest.mark.parametrize("version,n,k,tones", [
    (2, 1 << 20, 50, 0),     # W = 16384, two comb loops: all powers tie at zero
    (2, 1 << 20, 50, 3),     # fewer tones than picks, the rest leakage
    (2, 1 << 24, 10, 0),     # W = 2^18
    (1, 1 << 24, 2000, 0),   # v1: 4000 of 32768 buckets, ties
    (1, 1 << 24, 2000, 5),
])
def test_selection_levels(torch_cuda, version, n, k, tones):
    """Selections above the LDS size pick the oracle's indices, ties at the
    cutoff in index order."""
    print(f"case selection v{version} n={n} k={k} tones={tones}", flush=True)
    x = np.zeros(n, np.complex128)
    if tones:
        x, f, v = signal_np(n, tones, seed=12)
    plan = _gpu_plan(version, n, k)
    ref = _oracle_run(version, n, k, x, _plan_filters(plan))
    out = _run_gpu_dense(torch_cuda, plan, x)
    fr, va = _gpu_plan(version, n, k).execute_sparse_host(x)
    assert np.array_equal(np.unique(fr), _located(ref, version))
    assert np.array_equal(out, ref["out"])


@pytest.mark.parametrize("kind", ["plain", "tiny", "huge", "inf", "nan", "zero", "mixed"])
def test_alias_row_quotients(torch_cuda, kind):
    """The alias-row estimation of the FP64 form (quotients from tabulated
    reciprocals, divisions for buckets outside their range) gives the bits of
    the natural-order one, which divides throughout."""
    torch = torch_cuda
    n, k = 1 << 18, 64
    print(f"case alias-row quotients {kind}", flush=True)
    x, f, v = signal_np(n, k, seed=31, snr_db=30.0)
    xs = [x, x.copy()]
    if kind == "tiny":
        xs[1] *= 1e-230
    elif kind == "huge":
        xs[1] *= 1e250
    elif kind == "inf":
        xs[1][12345] = np.inf
    elif kind == "nan":
        xs[1][777] = np.nan
    elif kind == "zero":
        xs[1][:] = 0
    elif kind == "mixed":  # buckets of few taps on the large samples
        xs[1] *= 1e-300
        xs[1][5000:5003] = 1e200
    res = []
    for mode in (1, 2):
        for conj in (True, False):
            plan = _gpu_plan(2, n, k)
            plan.set_schedule(mode, 0)
            plan.set_reference_conjugate(conj)
            xd = [torch.from_numpy(a).cuda() for a in xs]
            fr, va = plan.make_sparse_outputs(2)
            c = plan.execute_many_sparse(xd, fr, va)
            res.append([(fr[i, :c[i]].cpu().numpy(), va[i, :c[i]].cpu().numpy()) for i in (0, 1)])
    for a, b in ((res[0], res[2]), (res[1], res[3])):
        for i in (0, 1):
            assert np.array_equal(a[i][0], b[i][0])
            assert np.array_equal(a[i][1].view(np.float64), b[i][1].view(np.float64), equal_nan=True)


@pytest.mark.parametrize("zero", [0.0, -0.0])
def test_alias_row_signs_of_zero(torch_cuda, zero):
    """Quotients of zero buckets keep the division's sign: for a signal of
    zeros the alias-row estimation (schedule 1) gives the bits of the
    natural-order one (schedule 2), which divides, estimates of -0 among
    them, with the reference's conjugation and without."""
    n, k = 1 << 18, 64
    print(f"case signs of zero {zero}", flush=True)
    x = np.full(n, complex(zero, zero))
    neg = np.uint64(1 << 63)
    for conj in (True, False):
        bits = []
        for mode in (1, 2):
            plan = _gpu_plan(2, n, k)
            plan.set_schedule(mode, 0)
            plan.set_reference_conjugate(conj)
            bits.append(_run_gpu_dense(torch_cuda, plan, x).view(np.uint64))
        assert np.array_equal(bits[0], bits[1]), conj
        assert (bits[1] == neg).any(), conj


@pytest.mark.parametrize("version,precision,mode", [
    (1, "fp64", 0), (1, "fp64", 1), (1, "fp32_refine", 0), (2, "fp64", 2), (2, "fp32_refine", 1)])
def test_dense_outputs_are_cleared(torch_cuda, version, precision, mode):
    """Dense device outputs that held other values read zero outside the
    located set, for one signal and for several, whatever the schedule."""
    torch = torch_cuda
    n, k = 1 << 16, 50
    print(f"case dense clear v{version} {precision} mode={mode}", flush=True)
    xs = [signal_np(n, k, seed=70 + i)[0] for i in range(3)]
    xd = [torch.from_numpy(x).cuda() for x in xs]
    plan = _gpu_plan(version, n, k, precision)
    plan.set_schedule(mode, 0)
    fr, va = plan.make_sparse_outputs(3)
    counts = plan.execute_many_sparse(xd, fr, va)
    want = torch.zeros((3, n), dtype=torch.complex128, device="cuda")
    for i in range(3):
        want[i, fr[i, :int(counts[i])].long()] = va[i, :int(counts[i])]
    plan.seed(17, 4242)
    outs = [torch.full((n,), 7 + 7j, dtype=torch.complex128, device="cuda") for _ in range(3)]
    plan.execute_many_device(xd, outs)
    for i in range(3):
        assert torch.equal(outs[i], want[i])
    plan.seed(17, 4242)
    plan.execute_device(xd[0], outs[1])
    assert torch.equal(outs[1], want[0])


@pytest.mark.parametrize("version,precision", [(1, "fp64"), (2, "fp64"), (2, "fp32_refine")])
def test_dense_outputs_sharing_memory(torch_cuda, version, precision):
    """A dense device output that shares memory with an input of the call is
    cleared before the inputs are read: the results are those of inputs
    whose shared samples are zero."""
    torch = torch_cuda
    n, k = 1 << 16, 64
    print(f"case shared memory v{version} {precision}", flush=True)
    xs = [torch.from_numpy(signal_np(n, k, seed=90 + i, snr_db=30.0)[0]).cuda() for i in range(3)]
    plan = _gpu_plan(version, n, k, precision)

    def run(ins, outs):
        plan.seed(17, 4242)
        plan.execute_many_device(ins, outs)
        torch.cuda.synchronize()

    def fresh(cnt):
        return [torch.empty(n, dtype=torch.complex128, device="cuda") for _ in range(cnt)]

    # half of the output over half of the input, and the other way round
    for shift in (n // 2, -(n // 2)):
        buf = torch.zeros(2 * n, dtype=torch.complex128, device="cuda")
        a, b = (0, shift) if shift > 0 else (-shift, 0)
        buf[a:a + n] = xs[0]
        x = xs[0].clone()
        x[max(0, b - a):min(n, b - a + n)] = 0
        want = fresh(1)
        run([x], want)
        run([buf[a:a + n]], [buf[b:b + n]])
        assert torch.equal(buf[b:b + n], want[0]), shift
    # an output that is another signal's input, and one that is its own
    want = fresh(3)
    run([xs[0], torch.zeros_like(xs[1]), torch.zeros_like(xs[2])], want)
    ins = [x.clone() for x in xs]
    outs = [ins[1], ins[2], fresh(1)[0]]
    run(ins, outs)
    for i in range(3):
        assert torch.equal(outs[i], want[i]), i


def test_dense_outputs_of_a_parted_batch(torch_cuda):
    """Dense device outputs of 70 FP32 signals, a batch that runs in parts
    (each part's clear on one stream, its estimates on another): every
    output, filled before, holds its signal's located values and zeros.  Two
    signals of different parts that share an output leave both spectra."""
    torch = torch_cuda
    n, k, S = 1 << 16, 64, 70
    print(f"case dense parted n={n} k={k} S={S}", flush=True)
    xs = [torch.from_numpy(signal_np(n, k, seed=300 + i, snr_db=30.0)[0]).cuda() for i in range(S)]
    plan = _gpu_plan(2, n, k, "fp32_refine")
    fr, va = plan.make_sparse_outputs(S)
    counts = plan.execute_many_sparse(xs, fr, va)
    want = torch.zeros((S, n), dtype=torch.complex128, device="cuda")
    for i in range(S):
        want[i, fr[i, :int(counts[i])].long()] = va[i, :int(counts[i])]
    outs = [torch.full((n,), 7 + 7j, dtype=torch.complex128, device="cuda") for _ in range(S)]
    for graphs in (False, True, True):
        plan.enable_graphs(graphs)
        plan.seed(17, 4242)
        for o in outs:
            o.fill_(5 - 3j)
        plan.execute_many_device(xs, outs)
        for i in range(S):
            assert torch.equal(outs[i], want[i]), (graphs, i)
    plan.enable_graphs(False)
    first, last = 1, S - 2
    shared = list(outs)
    shared[last] = shared[first]
    plan.seed(17, 4242)
    plan.execute_many_device(xs, shared)
    only = (want[first] != 0) & (want[last] == 0)
    other = (want[first] == 0) & (want[last] != 0)
    none = (want[first] == 0) & (want[last] == 0)
    got = shared[first]
    assert only.any() and other.any()
    assert torch.equal(got[only], want[first][only])
    assert torch.equal(got[other], want[last][other])
    assert not got[none].any()
    for i in range(S):
        if i not in (first, last):
            assert torch.equal(outs[i], want[i]), i


@pytest.mark.parametrize("version", [1, 2])
def test_refused_dense_call_clears_device_outputs(torch_cuda, version):
    """A batch refused for a null output leaves the device outputs before it
    cleared, as the reference's zero fill comes before anything else."""
    torch = torch_cuda
    n, k = 1 << 14, 50
    print(f"case refused dense call v{version}", flush=True)

    class Null:
        def data_ptr(self):
            return 0

    plan = _gpu_plan(version, n, k)
    xs = [torch.from_numpy(signal_np(n, k, seed=5 + i)[0]).cuda() for i in range(2)]
    out = torch.full((n,), 3 + 4j, dtype=torch.complex128, device="cuda")
    with pytest.raises(sfft_amd.SfftError, match="null output"):
        plan.execute_many_device(xs, [out, Null()])
    torch.cuda.synchronize()
    assert not out.any()


@pytest.mark.parametrize("version,n,k,precision,mode,launches", [
    # comb, fold, bucket FFTs, selection + votes, estimate, v3
    (1, 1 << 18, 100, "fp64", 1, (0, 1, 1, 2, 1, 0)),         # the FFTs select too
    (1, 1 << 18, 100, "fp64", 0, (0, 1, 0, 3, 1, 0)),         # FFTs in the fold, a selection
    (2, 1 << 18, 64, "fp32_refine", 1, (2, 1, 1, 0, 1, 0)),   # comb and alias-row table
    (2, 1 << 16, 50, "fp64", 1, (2, 1, 2, 0, 1, 0)),          # comb and merge; two bucket counts
    (2, 1 << 20, 50, "fp32_refine", 1, (5, 1, 1, 0, 1, 0)),   # runs, columns, level, merge, table
    (3, 1 << 16, 50, "fp64", 1, (0, 0, 0, 0, 0, 1)),
    (3, 1 << 16, 50, "fp32_refine", 1, (0, 0, 0, 0, 0, 5)),   # and the four refine kernels
])
def test_stage_launch_counts(torch_cuda, version, n, k, precision, mode, launches):
    """Stage timing counts the kernels each stage launches."""
    print(f"case stage launches v{version} n={n} k={k} {precision} mode={mode}", flush=True)
    x, f, v = signal_np(n, k, seed=4200 + k)
    plan = _gpu_plan(version, n, k, precision)
    plan.set_schedule(mode, 0)
    plan.enable_timing(True)
    for _ in range(2):
        plan.execute_sparse_host(x)
    st = plan.stage_times()
    assert tuple(int(st[s][1]) for s in plan.STAGES) == tuple(2 * c for c in launches), st
    assert all((st[s][0] > 0) == (c > 0) for s, c in zip(plan.STAGES, launches)), st


def test_autotune_keeps_stream_blocks(torch_cuda):
    """The autotuner chooses the fold mode; the caller's stream_blocks is
    reported back as it was set."""
    print("case autotune stream_blocks", flush=True)
    plan = _gpu_plan(2, 1 << 16, 64, "fp32_refine")
    plan.set_schedule(0, 96)
    mode, blocks = plan.autotune(batch=2)
    assert mode in (0, 1, 2) and blocks == 96


@pytest.mark.parametrize("kind", ["noise", "zeros"])
def test_selection_of_three_levels(torch_cuda, kind):
    """n = 2^26, k = 2000 (v1): 4000 of 65,536 buckets a loop, whose levels
    leave 32,000 and 16,000 candidates.  The located set is that of the votes
    counted over every frequency, with each loop's selection taken from the
    plan's own buckets by sorting (ties to the lower index)."""
    torch = torch_cuda
    n, k = 1 << 26, 2000
    print(f"case three levels {kind}", flush=True)
    plan = _gpu_plan(1, n, k)
    B, _, num, W, _, Lloc, Lest, thr = plan.params()[:8]
    assert (B, num) == (65536, 4000)
    x = torch.zeros(n, dtype=torch.complex128, device="cuda")
    if kind == "noise":
        g = torch.Generator(device="cuda")
        g.manual_seed(26)
        x.real.normal_(generator=g)
        x.imag.normal_(generator=g)
    fr, va = plan.make_sparse_outputs(1)
    count = int(plan.execute_many_sparse([x], fr, va)[0])
    print("transformed", flush=True)
    buckets = plan.debug_buckets(0)[:Lloc * B].reshape(Lloc, B)
    a, ai, off = (np.zeros(Lloc + Lest, np.int32) for _ in range(3))
    oracle.seed_glibc(17, 4242)
    oracle.lib().or_v12_draw(n, Lloc + Lest, 0, W, *(q.ctypes.data for q in (a, ai, off)))
    f = torch.arange(n, dtype=torch.int64, device="cuda")
    score = torch.zeros(n, dtype=torch.int32, device="cuda")
    for l in range(Lloc):
        power = buckets[l].real * buckets[l].real + buckets[l].imag * buckets[l].imag
        sel = np.zeros(B, np.int32)
        sel[np.lexsort((np.arange(B), -power))[:num]] = 1
        bucket = (((f * int(ai[l]) & (n - 1)) + n // B // 2) & (n - 1)) // (n // B)
        score += torch.from_numpy(sel).cuda()[bucket]
    want = torch.nonzero(score >= thr).flatten()
    assert count == want.numel() > 0
    assert torch.equal(torch.sort(fr[0, :count].long()).values, want)
    del x, fr, va, f, score
    torch.cuda.empty_cache()
