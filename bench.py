"""Benchmark: forward + adjoint gradient evaluations per second on one MI355X.

Workload (one step = one gradient evaluation): the 6-mode pure-state circuit
at cutoff 8 (262,144 complex64 amplitudes), 4 layers of the CV layered circuit
(240 operations, 408 real parameters), loss 1 - |<target|psi>|^2 with a seeded
target truncated to total photon number <= 6.  A step rebuilds every gate
matrix from the parameters (FP64 recurrences), runs the forward sweep, the loss
and the hand-written adjoint sweep, and returns all 408 gradients; it is
replayed from one captured HIP graph.  Inputs are resident on the GPU before
timing.

The JSON line also carries
  * fwd_evals_per_s: forward-only evaluations per second (same graph without
    the adjoint), and eager_grad_evals_per_s: the same gradient through
    torch.autograd without graph capture;
  * tf_path_grad_evals_per_s: the TF backend's gradient algorithm restated in
    torch on the same GPU (strawberryfields_amd/tfpath.py: dense per-gate
    matrices with a host round trip, contractions as matrix products, dense
    [D]^4 beamsplitter, autograd tape), with its gradient's relative
    difference from the adjoint's;
  * parity_vs_oracle: max|d psi| and 1 - F of the benchmarked ket against the
    complex128 CPU oracle;
  * roofline: the adjoint sweep (the dominant kernels, fused gate stages),
    algorithmic bytes 4 S per operation (S = state bytes) over the sweep's
    time measured with HIP events on its stream, beside the counter-measured
    HBM traffic per launch;
  * cpu_baseline: the CPU oracle's faithful restatement of the reference fock
    backend (slice loop with np.dot, selection-rule beamsplitter loop in C)
    on a bounded sample (the first layer), median of 5, all threads and one;
    a gradient on that backend needs 2P+1 forward passes (central
    differences), which scales the sample to grad-evals/s;
  * secondary: the 4-mode cutoff-15 forward (both dtypes), the 256-circuit
    batch gradient and the 3-mode cutoff-20 density-matrix gradient, each with
    its algorithmic GB/s and fraction of the 8 TB/s HBM peak.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline sample")
    ap.add_argument("--no-secondary", action="store_true", help="c3: skip the c2 / c4 / c5 lines of the default run")
    ap.add_argument("--fuse", type=int, default=None, help="local modes per fused stage (0 = one kernel per gate)")
    ap.add_argument(
        "--kernels-only",
        action="store_true",
        help="c3: run only the captured evaluator and the event-timed sweeps (no eager, TF-path or CPU legs); "
        "the short run that hardware-counter profiles use",
    )
    ap.add_argument(
        "--workload",
        default="c3",
        choices=["c2", "c3", "c4", "c5", "hbm", "next"],
        help="c3: 6-mode ket gradient (default line); c4: 256 uneven circuits in one graph launch; "
        "c5: 3-mode cutoff-20 density-matrix gradient with loss and layer checkpoints; "
        "hbm: per-kernel HBM rates on a 2 GB ket and the 512 MB DM; "
        "next: S2/MZ/CK/V gates, diagonal runs and measurement kernels on the same states",
    )
    return ap.parse_args()


def _event_us(fn, reps, stream=None):
    import torch

    fn()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    st = stream or torch.cuda.current_stream()
    e0.record(st)
    for _ in range(reps):
        fn()
    e1.record(st)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) * 1e3 / reps


def kernel_rates(n, D, mixed, dtype, reps=10, kinds=None):
    """Average launch time and algorithmic GB/s of each operation kind on one
    state: forward 2 S per operation (two passes on a DM for D, S, BS), adjoint
    4 S (forward state, cotangent in, cotangent out, + recompute on a DM).
    `kinds`: [(name, modes)] or [(name, modes, (p0, p1))]; default the gates of
    the main sweep."""
    import torch

    from strawberryfields_amd import runtime

    dev = torch.device("cuda:0")
    esz = 8 if dtype == torch.complex64 else 16
    S = D ** (2 * n if mixed else n) * esz
    shape = [D] * (2 * n if mixed else n)
    st = torch.randn(shape, dtype=dtype, device=dev)
    out = torch.empty_like(st)
    lam = torch.randn_like(st)
    gin = torch.empty_like(st)
    if kinds is None:
        kinds = [("D", (0,)), ("D", (n - 1,)), ("S", (n // 2,)), ("R", (0,)), ("K", (n - 1,)), ("BS", (0, 1)), ("BS", (n - 2, n - 1))]
        if mixed:
            kinds += [("LOSS", (0,)), ("LOSS", (n - 1,))]
    res = {}
    # plain device copy of the same state: the bandwidth reference (and the
    # kernel whose HBM counters calibrate FETCH_SIZE / WRITE_SIZE)
    tc = _event_us(lambda: out.copy_(st), reps)
    res["copy"] = {"fwd_us": round(tc, 1), "fwd_GBs": round(2 * S / tc / 1e3, 1)}
    for entry in kinds:
        kind, modes = entry[0], entry[1]
        par = entry[2] if len(entry) > 2 else ((0.3, 0.2) if kind != "LOSS" else (0.8, 0.0))
        cc = runtime.CompiledCircuit([(kind, modes)], n, D, mixed, dtype, dev, fuse=0)
        cc.build_table(torch.tensor([list(par)], dtype=torch.float64, device=dev))
        grads = torch.zeros(2, dtype=torch.float64, device=dev)
        tf = _event_us(lambda: cc.forward(0, 1, st, out=out), reps)
        ta = _event_us(lambda: cc.adjoint(0, 1, [st], lam, gin, grads), reps)
        res["%s%s" % (kind, list(modes))] = {
            "fwd_us": round(tf, 1),
            "fwd_GBs": round(2 * S / tf / 1e3, 1),
            "fwd_pct_peak": round(100 * 2 * S / tf / 1e3 / HBM_PEAK_GBS, 1),
            "adj_us": round(ta, 1),
            "adj_GBs": round(4 * S / ta / 1e3, 1),
            "adj_pct_peak": round(100 * 4 * S / ta / 1e3 / HBM_PEAK_GBS, 1),
        }
    return S, res


def _note(msg):
    """A progress line on stderr (stdout carries only the JSON line)."""
    print("[bench] " + msg, file=sys.stderr, flush=True)


def _c5_fixture():
    """Complex128 oracle observables of the full-size c5 forward (written by
    tests/golden/make_c5_fixture.py), or None when absent."""
    import numpy as np

    path = os.path.join(ROOT, "tests", "golden", "c5_forward.npz")
    if not os.path.exists(path):
        return None
    return dict(np.load(path))


def measure_c5(steps, rates=False):
    """3-mode DM at cutoff 20 (64M complex64, 512 MB), 6 layers with loss:
    forward + adjoint gradient of sum_n p(n) (n1+n2+n3-3)^2, checkpoints at
    layer boundaries (24 steps), the rest recomputed in the backward.  The
    TF-path comparator is not timed here: its autograd tape would hold every
    intermediate DM and every permuted matrix-product input (about 200 GB at
    this size); it is timed on the 6-mode ket."""
    import numpy as np
    import torch

    from strawberryfields_amd import circuits, runtime

    dev = torch.device("cuda:0")
    c5 = circuits.config5()
    n, D, ops = c5["n"], c5["D"], c5["ops"]
    dtype = torch.complex64
    cc = runtime.CompiledCircuit([(o[0], o[1]) for o in ops], n, D, True, dtype, dev)
    rows = np.zeros((len(ops), 2))
    for i, (_, _, p) in enumerate(ops):
        rows[i, : len(p)] = p
    params = torch.tensor(rows, dtype=torch.float64, device=dev, requires_grad=True)
    rho0 = torch.zeros([D] * (2 * n), dtype=dtype, device=dev)
    rho0.view(-1)[0] = 1.0
    idx = torch.arange(D, device=dev, dtype=torch.float64)
    w = (idx[:, None, None] + idx[None, :, None] + idx[None, None, :] - 3.0) ** 2

    def step():
        params.grad = None
        rho = runtime.CircuitFunction.apply(params, rho0, cc, c5["layer_len"])
        probs = runtime.all_fock_probs(rho, n, D, True)
        loss = (probs.to(torch.float64) * w).sum()
        loss.backward()
        return loss

    step()
    torch.cuda.synchronize()
    reps = max(2, min(steps, 5))
    t0 = time.perf_counter()
    for _ in range(reps):
        loss = step()
    torch.cuda.synchronize()
    t_grad = (time.perf_counter() - t0) / reps
    if rates:
        _note("c5 gradient: %.1f ms per evaluation" % (t_grad * 1e3))
    with torch.no_grad():
        t0 = time.perf_counter()
        for _ in range(reps):
            rho = runtime.run_circuit(cc, params.detach(), rho0)
        torch.cuda.synchronize()
        t_fwd = (time.perf_counter() - t0) / reps
    S = D ** (2 * n) * 8
    nops = len(ops)
    out = {
        "grad_evals_per_s": round(1.0 / t_grad, 3),
        "ms_per_grad_eval": round(t_grad * 1e3, 2),
        "fwd_ms": round(t_fwd * 1e3, 2),
        "loss": float(loss.detach()),
        "grad_norm": float(params.grad.norm()),
        "trace": float(runtime.norm2(rho, n, D, True)),
        "grad_algorithmic_GBs": round(6 * S * nops / t_grad / 1e9, 1),
        "grad_frac_of_hbm_peak": round(6 * S * nops / t_grad / 1e9 / HBM_PEAK_GBS, 4),
        "fwd_algorithmic_GBs": round(2 * S * nops / t_fwd / 1e9, 1),
        "fwd_frac_of_hbm_peak": round(2 * S * nops / t_fwd / 1e9 / HBM_PEAK_GBS, 4),
        "algorithmic": "2 S per forward operation, 6 S per gradient, S = %d B, %d operations" % (S, nops),
    }
    fx = _c5_fixture()
    if fx is not None:  # forward parity against the complex128 oracle (fixture)
        probs = runtime.all_fock_probs(rho, n, D, True).to(torch.float64).cpu().numpy()
        rdm = runtime.reduced_dm(rho, n, D, True, [0, 1]).to(torch.complex128).cpu().numpy()
        out["max_abs_dprob_vs_oracle"] = float(np.abs(probs - fx["probs"]).max())
        out["max_abs_drho01_vs_oracle"] = float(np.abs(rdm[:10, :10, :10, :10] - fx["rdm01_low"]).max())
    if rates:
        _note("c5 per-kernel rates")
        _, out["kernels"] = kernel_rates(n, D, True, dtype)
    return out


def run_c5(args):
    out = measure_c5(args.steps, rates=True)
    line = {
        "metric": "grad-evals/s (fwd+adjoint), 3-mode cutoff-20 density matrix with loss",
        "value": out["grad_evals_per_s"],
        "unit": "grad-evals/s",
        "n_gpus": 1,
        "dtype": "complex64",
        "data": "synthetic",
        "config": {"workload": "3-mode DM, cutoff 20, 6 layers with loss (144 ops), layer checkpoints"},
    }
    line.update(out)
    print(json.dumps(line))


def measure_c2(steps, cpu=False):
    """4-mode pure ket at cutoff 15 (50,625 amplitudes), 8 layers (256 ops),
    forward only in complex64 and complex128: evals/s launched eagerly (one
    library call per forward) and replayed from a HIP graph, norm and
    fock_prob; with `cpu` the CPU leg times the oracle's faithful fock-backend
    loop, whose complex128 state is also the reference the GPU results are
    compared with."""
    import numpy as np
    import torch

    from strawberryfields_amd import circuits, runtime

    dev = torch.device("cuda:0")
    c2 = circuits.config2()
    n, D, ops = c2["n"], c2["D"], c2["ops"]
    rows = np.zeros((len(ops), 2))
    for i, (_, _, p) in enumerate(ops):
        rows[i, : len(p)] = p
    params = torch.tensor(rows, dtype=torch.float64, device=dev)
    tuner = runtime.Autotuner(path=os.environ.get("SFAMD_AUTOTUNE_CACHE"))
    out = {}
    kets = {}
    for name, dtype in (("complex64", torch.complex64), ("complex128", torch.complex128)):
        K = tuner.best([(o[0], o[1]) for o in ops], n, D, False, dtype, dev, forward_only=True)
        cc = runtime.CompiledCircuit([(o[0], o[1]) for o in ops], n, D, False, dtype, dev, fuse=K)
        vac = torch.zeros([D] * n, dtype=dtype, device=dev)
        vac.view(-1)[0] = 1.0
        psi = runtime.run_circuit(cc, params, vac)
        torch.cuda.synchronize()
        reps = max(10, steps)
        t0 = time.perf_counter()
        for _ in range(reps):
            psi = runtime.run_circuit(cc, params, vac)
        torch.cuda.synchronize()
        t = (time.perf_counter() - t0) / reps
        probs = runtime.all_fock_probs(psi, n, D, False)
        kets[name] = psi.cpu().numpy()
        # the same forward (table build + every step, plus a fidelity readout)
        # replayed from one captured HIP graph, timed with events on its stream
        ev = runtime.GradEvaluator(cc, vac, vac, use_graph=True, forward_only=True)
        ev(params)
        ev.stream.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(ev.stream)
        for _ in range(reps):
            ev(params)
        e1.record(ev.stream)
        e1.synchronize()
        t_graph = e0.elapsed_time(e1) / 1e3 / reps
        dg = float((ev.psi - psi).abs().max())
        del ev
        S = D**n * (8 if dtype == torch.complex64 else 16)
        out[name] = {
            "fwd_evals_per_s": round(1.0 / t, 1),
            "ms": round(t * 1e3, 4),
            "fwd_evals_per_s_graph": round(1.0 / t_graph, 1),
            "ms_graph": round(t_graph * 1e3, 4),
            "fwd_algorithmic_GBs_graph": round(2 * S * len(ops) / t_graph / 1e9, 1),
            "graph_vs_eager_max_abs_diff": dg,
            "fused_local_modes": K,
            "steps": cc.nsteps,
            "norm": float(runtime.norm2(psi, n, D, False)),
            "fock_prob_0000": float(probs[0, 0, 0, 0]),
            "fock_prob_1021": float(probs[1, 0, 2, 1]),
        }
    cpu_line = None
    if cpu:
        from threadpoolctl import threadpool_limits

        from oracle import fock_oracle as fo

        with threadpool_limits(limits=1):
            t0 = time.perf_counter()
            ref, _ = fo.run_ops(ops, n, D, pure=True, faithful=True)
            t_cpu = time.perf_counter() - t0
        cpu_line = {"value": 1.0 / t_cpu, "unit": "forward evals/s", "cores": 1, "kind": "port",
                    "sample": "one complex128 forward through the oracle's faithful fock-backend loop (%.2f s)" % t_cpu}
        r = ref.reshape(-1)
        for name in kets:
            k = kets[name].reshape(-1).astype(np.complex128)
            out[name]["max_abs_dpsi"] = float(np.abs(k - r).max())
            out[name]["one_minus_fidelity"] = float(
                1 - abs(np.vdot(r, k)) ** 2 / (np.vdot(r, r).real * np.vdot(k, k).real)
            )
    return out, cpu_line


def run_c2(args):
    out, cpu = measure_c2(args.steps, cpu=not (args.no_cpu or args.kernels_only))
    print(json.dumps({"metric": "forward evals/s, 4-mode cutoff-15 ket, 256 ops", "results": out, "cpu_baseline": cpu,
                      "dtype": "complex64 and complex128", "data": "synthetic", "n_gpus": 1}))


def measure_c4(steps):
    """256 independent pure circuits (n in 2..5, cutoff 6..20, D^n <= 2^20,
    2-6 layers): forward + adjoint gradient of each circuit's total mean photon
    number, all replayed from one HIP graph; stage tiles from the autotuner."""
    import numpy as np
    import torch

    from strawberryfields_amd import circuits, runtime

    dev = torch.device("cuda:0")
    c4 = circuits.config4()
    circs = c4["circuits"]
    tuner = runtime.Autotuner(path=os.environ.get("SFAMD_AUTOTUNE_CACHE"))
    t0 = time.perf_counter()
    be = runtime.BatchEvaluator(circs, torch.complex64, dev, tuner=tuner)
    t_setup = time.perf_counter() - t0
    plist = []
    for c in circs:
        rows = np.zeros((len(c["ops"]), 2))
        for i, (_, _, p) in enumerate(c["ops"]):
            rows[i, : len(p)] = p
        plist.append(torch.tensor(rows, dtype=torch.float64, device=dev))
    for _ in range(2):
        be(plist)
    torch.cuda.synchronize()
    reps = max(3, min(steps, 20))
    t0 = time.perf_counter()
    for _ in range(reps):
        losses, grads = be(plist)
    torch.cuda.synchronize()
    t_eval = (time.perf_counter() - t0) / reps
    amps = sum(c["D"] ** c["n"] for c in circs)
    alg = sum(6 * 8 * c["D"] ** c["n"] * len(c["ops"]) for c in circs)
    fuse_hist = {}
    for it in be.items:
        fuse_hist[str(it["cc"].fuse)] = fuse_hist.get(str(it["cc"].fuse), 0) + 1
    return {
        "batch_evals_per_s": round(1.0 / t_eval, 3),
        "circuit_grad_evals_per_s": round(len(circs) / t_eval, 1),
        "ms_per_batch": round(t_eval * 1e3, 3),
        "amplitudes": amps,
        "grad_algorithmic_GBs": round(alg / t_eval / 1e9, 1),
        "grad_frac_of_hbm_peak": round(alg / t_eval / 1e9 / HBM_PEAK_GBS, 4),
        "algorithmic": "6 S per operation per circuit (S = 8 D^n B), summed over the 256 circuits",
        "setup_s_incl_autotune": round(t_setup, 2),
        "autotuned_tiles": fuse_hist,
        "mean_loss": float(losses.mean()),
    }


def run_c4(args):
    out = measure_c4(args.steps)
    line = {
        "metric": "batch grad-evals/s (256 circuits per evaluation, one graph launch)",
        "value": out["batch_evals_per_s"],
        "unit": "batch-evals/s",
        "n_gpus": 1,
        "dtype": "complex64",
        "data": "synthetic",
        "config": {"workload": "256 uneven pure circuits, loss = total mean photon number"},
    }
    line.update(out)
    print(json.dumps(line))


def run_hbm(args):
    """Per-operation HBM rates on a 2 GB pure state (7 modes, cutoff 16) and on
    the 512 MB density matrix (3 modes, cutoff 20), complex64."""
    import torch

    S1, r1 = kernel_rates(7, 16, False, torch.complex64)
    S2, r2 = kernel_rates(3, 20, True, torch.complex64)
    print(
        json.dumps(
            {
                "metric": "algorithmic HBM GB/s per operation (peak %d GB/s)" % HBM_PEAK_GBS,
                "ket_7modes_cutoff16": {"state_MB": S1 / 2**20, "ops": r1},
                "dm_3modes_cutoff20": {"state_MB": S2 / 2**20, "ops": r2},
            }
        )
    )


def run_next(args):
    """The operations past the core gate set, on the same large states as the HBM
    sweep (complex64): S2, MZ, CK and V gates (forward and adjoint), a run of
    three R / K gates in one pass, and the measurement / preparation kernels
    (marginal distribution, |0><x| projection, homodyne density, multi-mode
    embedding)."""
    import torch

    from strawberryfields_amd import runtime

    dev = torch.device("cuda:0")
    c64 = torch.complex64
    ket_kinds = [("S2", (0, 1)), ("S2", (5, 6)), ("MZ", (0, 1)), ("MZ", (5, 6)), ("CK", (0, 1)), ("V", (0,), (0.2, 0.0))]
    dm_kinds = [("S2", (0, 1)), ("S2", (1, 2)), ("MZ", (1, 2)), ("CK", (0, 1)), ("V", (0,), (0.2, 0.0))]
    S1, r1 = kernel_rates(7, 16, False, c64, kinds=ket_kinds)
    S2, r2 = kernel_rates(3, 20, True, c64, kinds=dm_kinds)
    meas = {}
    for label, n, D, mixed in [("ket_7modes_cutoff16", 7, 16, False), ("dm_3modes_cutoff20", 3, 20, True)]:
        shape = [D] * (2 * n if mixed else n)
        st = torch.randn(shape, dtype=c64, device=dev)
        S = st.numel() * 8
        m = {}
        # a run of three diagonal gates on three modes, one pass
        ops = [("R", (0,)), ("K", (1,)), ("R", (n - 1,))]
        cc = runtime.CompiledCircuit(ops, n, D, mixed, c64, dev, fuse=0)
        cc.build_table(torch.tensor([[0.3, 0.0]] * 3, dtype=torch.float64, device=dev))
        out = torch.empty_like(st)
        lam = torch.randn_like(st)
        gin = torch.empty_like(st)
        grads = torch.zeros(6, dtype=torch.float64, device=dev)
        tf = _event_us(lambda: cc.forward(0, cc.nsteps, st, out=out), 10)
        ta = _event_us(lambda: cc.adjoint(0, cc.nsteps, [st], lam, gin, grads), 10)
        m["R,K,R run (one pass)"] = {
            "fwd_us": round(tf, 1),
            "fwd_pct_peak": round(100 * 2 * S / tf / 1e3 / HBM_PEAK_GBS, 1),
            "adj_us": round(ta, 1),
            "adj_pct_peak": round(100 * 3 * S / ta / 1e3 / HBM_PEAK_GBS, 1),
        }
        for k in (1, 2):
            t = _event_us(lambda: runtime.marginal_probs(st, n, D, mixed, list(range(k))), 10)
            read = (D**n) * 8 if mixed else S  # a DM's marginal reads its diagonal only
            m["marginal_probs %d mode(s)" % k] = {"us": round(t, 1), "GBs_read": round(read / t / 1e3, 1)}
        t = _event_us(lambda: runtime.project_reset(st, n, D, mixed, [0], [1], 1.0), 10)
        m["project_reset 1 mode"] = {"us": round(t, 1), "pct_peak": round(100 * 2 * S / t / 1e3 / HBM_PEAK_GBS, 1)}
        if mixed:
            rho = runtime.reduced_dm(st, n, D, True, [1])
            t = _event_us(lambda: runtime.homodyne_pdf(rho, D, 0.3, 10.0, 100000, 2.0), 10)
            m["homodyne_pdf 100000 bins"] = {"us": round(t, 1), "GFLOPs": round(100000 * D * D * 2 / t / 1e3, 1)}
            rest = runtime.reduced_dm(st, n, D, True, [0])
            sig = torch.randn([D] * 4, dtype=c64, device=dev)
            t = _event_us(lambda: runtime.embed_modes(rest, sig, n, D, [2, 1], True), 10)
            m["embed 2-mode DM"] = {"us": round(t, 1), "pct_peak": round(100 * S / t / 1e3 / HBM_PEAK_GBS, 1)}
        meas[label] = m
        del st, out, lam, gin
        torch.cuda.empty_cache()
    print(
        json.dumps(
            {
                "metric": "S2/MZ/CK/V gates, diagonal runs and measurement kernels on large states (peak %d GB/s)" % HBM_PEAK_GBS,
                "ket_7modes_cutoff16": {"state_MB": S1 / 2**20, "gates": r1},
                "dm_3modes_cutoff20": {"state_MB": S2 / 2**20, "gates": r2},
                "measurement": meas,
            }
        )
    )


def stage_adj_traffic():
    """HBM bytes per k_mst_adj launch measured by the FETCH_SIZE / WRITE_SIZE
    counter runs recorded in profiles/ (calibrated against a device copy)."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", "c3_matrix_stage_hbm_traffic.txt")
    try:
        with open(path) as f:
            for line in f:
                if line.startswith("traffic_bytes_per_launch k_mst_adj:"):
                    return int(line.split(":")[1]), "profiles/c3_matrix_stage_hbm_traffic.txt"
    except OSError:
        pass
    return None, None


def comparators(args, cc, params, vac, target, grads, ops, n, D, timed):
    """Eager autograd (same kernels, no graph) and the TF-backend gradient path
    restated in torch (dense contractions + autograd) on the same GPU."""
    import torch

    from strawberryfields_amd import runtime

    dtype = vac.dtype
    dev = vac.device
    p_leaf = params.clone().requires_grad_(True)

    def eager():
        p_leaf.grad = None
        psi = runtime.CircuitFunction.apply(p_leaf, vac, cc, None)
        runtime.fidelity_loss(psi, target).backward()

    t_eager = timed(eager, max(10, args.steps // 4), 3)
    eager_rate = max(10, args.steps // 4) / t_eager
    eager_diff = float((p_leaf.grad - grads).abs().max())

    from strawberryfields_amd import tfpath

    tfc = tfpath.TFPathCircuit([(o[0], o[1]) for o in ops], n, D, dtype, dev)
    p_tf = params.clone().requires_grad_(True)

    def tf_step():
        p_tf.grad = None
        psi = tfc.forward(p_tf)
        ov = torch.vdot(target.reshape(-1), psi.reshape(-1))
        (1 - ov.real**2 - ov.imag**2).backward()

    tf_steps = 5
    t_tf = timed(tf_step, tf_steps, 1)
    tf_rate = tf_steps / t_tf
    tf_diff = float((p_tf.grad - grads).norm() / grads.norm())

    return eager_rate, eager_diff, tf_rate, tf_diff


def _cpu_model():
    try:
        import subprocess

        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            if line.lower().startswith("model name"):
                return line.split(":", 1)[1].strip()
    except (OSError, ValueError, Exception):  # noqa: BLE001 -- lscpu may be absent
        pass
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def cpu_baseline_c3(ops, n, D, layers, nparam, psi_gpu):
    """The CPU fock-backend algorithm on the host cores: the oracle's faithful
    restatement (apply_gate_BLAS's slice loop with np.dot; the selection-rule
    beamsplitter loop in C, oracle/fock_cpu.c, standing in for the reference's
    numba loop), complex128, on a bounded sample -- the first layer of the
    workload (its layers have identical structure) -- one warm-up, then the
    median of 5 runs, with all BLAS threads and with one; a gradient on that
    backend is 2P+1 forward passes (central differences).  The oracle's
    vectorised forward of the whole circuit also gives the complex128
    reference the GPU ket is compared with."""
    import statistics

    import numpy as np
    from threadpoolctl import threadpool_limits

    from oracle import fock_oracle as fo

    per_layer = len(ops) // layers
    sample = ops[:per_layer]
    med = {}
    for label, lim in (("all_threads", None), ("one_thread", 1)):
        with threadpool_limits(limits=lim):
            fo.run_ops(sample, n, D, pure=True, faithful=True)
            ts = []
            for _ in range(5):
                t0 = time.perf_counter()
                fo.run_ops(sample, n, D, pure=True, faithful=True)
                ts.append(time.perf_counter() - t0)
        med[label] = statistics.median(ts)
    t_fwd = med["all_threads"] * layers
    ref, _ = fo.run_ops(ops, n, D, pure=True)
    r = ref.reshape(-1)
    k = psi_gpu.reshape(-1).astype(np.complex128)
    parity = {
        "max_abs_dpsi": float(np.abs(k - r).max()),
        "one_minus_fidelity": float(1 - abs(np.vdot(r, k)) ** 2 / (np.vdot(r, r).real * np.vdot(k, k).real)),
    }
    cpu = {
        "value": 1.0 / (t_fwd * (2 * nparam + 1)),
        "unit": "grad-evals/s",
        "cores": 1,
        "kind": "port",
        "sample": "layer 1 of %d (%d ops) of the workload through the oracle's faithful fock-backend loop, "
        "complex128, median of 5 after a warm-up: %.3f s with all BLAS threads, %.3f s with one; "
        "x%d layers = %.2f s per forward; central-difference gradient = 2P+1 = %d forwards"
        % (layers, per_layer, med["all_threads"], med["one_thread"], layers, t_fwd, 2 * nparam + 1),
        "fwd_evals_per_s": 1.0 / t_fwd,
        "fwd_s_one_thread": med["one_thread"] * layers,
        "native_selection_rule_loop": fo.native_lib() is not None,
        "host_cpu_count": os.cpu_count(),
        "host_cpu_model": _cpu_model(),
        "threads_note": "the slice loop and the selection-rule loop are single-threaded, as in the reference; "
        "only the tiny np.dot calls could use BLAS threads",
    }
    return cpu, parity


def secondary(args):
    """The other workloads, measured in the same run: c2 forward (both dtypes,
    graph replay), c4 batch gradient and c5 density-matrix gradient, each with
    its algorithmic GB/s and fraction of the HBM peak."""
    import torch

    out = {}
    c2, _ = measure_c2(max(20, args.steps // 10), cpu=not (args.no_cpu or args.kernels_only))
    out["c2_4mode_cutoff15_forward"] = c2
    torch.cuda.empty_cache()
    out["c4_256_uneven_circuits_gradient"] = measure_c4(10)
    torch.cuda.empty_cache()
    out["c5_3mode_cutoff20_dm_gradient"] = measure_c5(3)
    torch.cuda.empty_cache()
    return out


def main():
    args = parse()
    if args.gpus != 1:
        print(
            "bench.py measures one GPU: there is no multi-GPU path "
            "(one state would be sharded along its most significant mode axis); run with --gpus 1",
            file=sys.stderr,
        )
        sys.exit(2)

    import numpy as np
    import torch

    from strawberryfields_amd import circuits, runtime

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.workload == "c5":
        return run_c5(args)
    if args.workload == "c4":
        return run_c4(args)
    if args.workload == "c2":
        return run_c2(args)
    if args.workload == "hbm":
        return run_hbm(args)
    if args.workload == "next":
        return run_next(args)
    c3 = circuits.config3()
    n, D, ops = c3["n"], c3["D"], c3["ops"]
    dtype = torch.complex64
    nparam = circuits.n_params(ops)

    cc = runtime.CompiledCircuit([(o[0], o[1]) for o in ops], n, D, False, dtype, dev, fuse=args.fuse)
    rows = np.zeros((len(ops), 2))
    for i, (_, _, p) in enumerate(ops):
        rows[i, : len(p)] = p
    params = torch.tensor(rows, dtype=torch.float64, device=dev)
    vac = torch.zeros([D] * n, dtype=dtype, device=dev)
    vac.view(-1)[0] = 1.0
    target = torch.as_tensor(c3["target"], dtype=dtype, device=dev)

    def timed(fn, steps, warmup):
        for _ in range(warmup):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return time.perf_counter() - t0

    # ---- captured gradient evaluation (the measured step)
    ev = runtime.GradEvaluator(cc, vac, target, use_graph=True)
    t_grad = timed(lambda: ev(params), args.steps, args.warmup)
    loss, grads = ev(params)
    torch.cuda.synchronize()
    loss = float(loss)
    grad_norm = float(grads.norm())
    grads = grads.clone()
    psi_gpu = ev.psi.cpu().numpy()
    value = args.steps / t_grad

    evf = runtime.GradEvaluator(cc, vac, target, use_graph=True, forward_only=True)
    t_fwd = timed(lambda: evf(params), args.steps, args.warmup)
    fwd_rate = args.steps / t_fwd

    eager_rate = eager_diff = tf_rate = tf_diff = None
    if not args.kernels_only:
        eager_rate, eager_diff, tf_rate, tf_diff = comparators(args, cc, params, vac, target, grads, ops, n, D, timed)

    # ---- sweep timing with HIP events on the evaluator's stream
    S = (D**n) * 8
    stream = ev.stream

    def event_time(fn, reps):
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        with torch.cuda.stream(stream):
            fn()
            e0.record(stream)
            for _ in range(reps):
                fn()
            e1.record(stream)
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) * 1e-3 / reps

    reps = 20
    with torch.cuda.stream(stream):
        cc.build_table(ev.params)
    t_fsweep = event_time(lambda: cc.forward(0, cc.nsteps, ev.state_in, out=ev.psi, saved=ev.saved), reps)
    t_asweep = event_time(lambda: cc.adjoint(0, cc.nsteps, ev.saved, ev.g_psi, ev.g_in, ev.grads), reps)
    nops = len(ops)
    # the traffic was counted on the default plan's matrix-core stages
    matrix = args.fuse is None and set(cc.step_kinds()) == {"matrix"}
    traffic, traffic_src = stage_adj_traffic() if matrix else (None, None)
    adj_bytes = 4 * S * nops
    fwd_bytes = 2 * S * nops
    achieved = adj_bytes / t_asweep / 1e9
    per_launch = t_asweep / cc.nsteps
    roofline = {
        "bound": "hbm",
        "kernel": "k_mst_adj (matrix-core adjoint gate stages, %d launches per sweep)" % cc.nsteps,
        "achieved": round(achieved, 1),
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 4),
        "traffic": traffic,
        "traffic_source": traffic_src,
        "bytes_per_launch": int(adj_bytes / cc.nsteps),
        "avg_launch_us": round(per_launch * 1e6, 3),
        "algorithmic": "4 S per adjoint operation, S = %d B; %d operations in %d fused launches" % (S, nops, cc.nsteps),
        "fwd_sweep_GBs": round(fwd_bytes / t_fsweep / 1e9, 1),
        "measured_traffic_GBs": round(traffic / per_launch / 1e9, 1) if traffic else None,
        "measured_traffic_frac": round(traffic / per_launch / 1e9 / HBM_PEAK_GBS, 4) if traffic else None,
        "limiter": "not HBM: the 2 MiB state stays in cache and a fused stage moves memory once for ~5 gates; "
        "the stage kernels are bound by launch latency and by LDS, barriers and reductions per gate (frac is algorithmic bytes "
        "over time, not HBM utilisation)",
    }

    # ---- CPU baseline: faithful fock-backend restatement, bounded sample
    cpu = parity = None
    if not (args.no_cpu or args.kernels_only):
        cpu, parity = cpu_baseline_c3(c3["ops"], n, D, 4, nparam, psi_gpu)

    line = {
        "metric": "grad-evals/s (fwd+adjoint) vs fwd-only & CPU fockbackend; HBM GB/s % peak",
        "value": round(value, 2),
        "unit": "grad-evals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * t_grad / args.steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "complex64",
        "data": "synthetic",
        "config": {
            "workload": "6-mode pure ket, cutoff 8, 4-layer CV layered circuit "
            "(240 ops, %d params), loss 1-|<t|psi>|^2, forward + adjoint" % nparam,
            "modes": n,
            "cutoff": D,
            "layers": 4,
            "params": nparam,
            "fused_local_modes": cc.fuse,
            "steps_per_sweep": cc.nsteps,
        },
        "fwd_evals_per_s": round(fwd_rate, 2),
        "eager_grad_evals_per_s": round(eager_rate, 2) if eager_rate else None,
        "tf_path_grad_evals_per_s": round(tf_rate, 3) if tf_rate else None,
        "speedup_vs_tf_path": round(value / tf_rate, 1) if tf_rate else None,
        "tf_path_grad_rel_diff": tf_diff,
        "graph_vs_eager_max_grad_diff": eager_diff,
        "loss": loss,
        "grad_norm": grad_norm,
        "parity_vs_oracle": parity,
        "roofline": roofline,
        "cpu_baseline": cpu,
    }
    if not (args.no_secondary or args.kernels_only):
        line["secondary"] = secondary(args)
    print(json.dumps(line))


if __name__ == "__main__":
    main()
