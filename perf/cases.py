"""Timed workloads of this package: what a program that uses it has it do, over
the sizes that its circuits take.

Each case runs through the public entry points: the Engine with the HIP
backend, planned circuits (``CompiledCircuit`` / ``run_circuit``), gradients
through autograd or a captured ``GradEvaluator``, batches of circuits, and the
readouts of ``FockStateHIP``.  ``exact`` restates every case with dense gate
matrices in 64 bits, independent of the package.

Circuit parameters are float32 leaves in complex64 programs and float64 leaves
in complex128 ones, so losses and gradients come back in that type.
"""
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from strawberryfields_amd import HIPFockBackend, circuits, frontend, runtime
from strawberryfields_amd.states import FockStateHIP

DTYPES = {"c64": torch.complex64, "c128": torch.complex128}
REAL = {"c64": torch.float32, "c128": torch.float64}
NUMPY = {"c64": np.float32, "c128": np.float64}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the plain method at its smallest: a 3-mode program run by the Engine in the default
        # precision, as one evaluates a circuit interactively (dominated by calls and launches)
        dict(name="engine 3x8 c128", kind="engine", n=3, D=8, dtype="c128"),
        # forward of a layered circuit on a small ket, in both precisions: sampling and
        # inference with a trained circuit
        dict(name="ket fwd 4x15 c64", kind="fwd", n=4, D=15, layers=8, dtype="c64"),
        dict(name="ket fwd 4x15 c128", kind="fwd", n=4, D=15, layers=8, dtype="c128"),
        # forward on a ket much larger than the caches (2 GiB)
        dict(name="ket fwd 7x16 c64", kind="fwd", n=7, D=16, layers=1, dtype="c64"),
        # a training step replayed from one graph: the 6-mode cutoff-8 circuit
        dict(name="ket grad 6x8 c64 graph", kind="graph", n=6, D=8, layers=4, dtype="c64"),
        # training steps through autograd: a ragged cutoff in the default precision, and a
        # state of 128 MiB
        dict(name="ket grad 3x11 c128", kind="grad", n=3, D=11, layers=3, dtype="c128"),
        dict(name="ket grad 6x16 c64", kind="grad", n=6, D=16, layers=1, dtype="c64"),
        # the gates beyond the layered circuit (S2, MZ, CK, V) in a random program, trained
        dict(name="gates grad 5x10 c64", kind="gates", n=5, D=10, count=40, structure=11, dtype="c64"),
        # many uneven circuits trained together
        dict(name="batch of 32 c64", kind="batch", count=32, maxamps=200000, structure=5, dtype="c64"),
        # noisy circuits: density matrices with loss, trained with checkpoints at layers
        dict(name="dm grad 3x20 c64", kind="dm", n=3, D=20, layers=6, dtype="c64"),
        dict(name="dm grad 3x9 c128", kind="dm", n=3, D=9, layers=2, dtype="c128"),
        # reading a state out: probabilities, moments, reduced states, marginals, homodyne density
        dict(name="readout 6x8 c128", kind="readout", n=6, D=8, mixed=False, dtype="c128"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ket_size(rng, lo, hi, nmin=2, nmax=8, dmax=24):
    """Modes and cutoff of a ket of about lo..hi amplitudes (spread over the logarithm)."""
    while True:
        want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        n = rng.randint(nmin, nmax)
        D = int(round(want ** (1.0 / n))) + rng.randint(-1, 1)
        if 3 <= D <= dmax and lo / 2 <= D**n <= hi:
            return n, D


def draw(rng):
    kind = rng.choice(["engine", "fwd", "fwd", "graph", "graph", "grad", "grad", "gates", "batch", "dm", "dm", "readout"])
    dtype = rng.choice(["c64", "c64", "c128"])
    if kind == "engine":
        n = rng.randint(2, 4)
        return dict(kind=kind, n=n, D=rng.randint(4, 24 if n < 4 else 14), dtype=rng.choice(["c64", "c128"]))
    if kind == "fwd":
        n, D = _ket_size(rng, 200, 2e8)
        return dict(kind=kind, n=n, D=D, layers=_logint(rng, 1, 8) if D**n < 1e7 else 1, dtype=dtype)
    if kind in ("graph", "grad"):
        n, D = _ket_size(rng, 200, 2e6 if kind == "graph" else 1.5e7)
        return dict(kind=kind, n=n, D=D, layers=rng.randint(1, 5) if D**n < 1e6 else 1, dtype=dtype)
    if kind == "gates":
        n, D = _ket_size(rng, 200, 5e6, dmax=20)
        return dict(kind=kind, n=n, D=D, count=_logint(rng, 8, 60), structure=rng.randrange(10**6), dtype=dtype)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(4, 40), maxamps=_logint(rng, 3000, 300000),
                    structure=rng.randrange(10**6), dtype="c64")
    if kind == "dm":
        while True:
            n, D = rng.randint(1, 3), rng.randint(4, 20)
            N = D ** (2 * n)
            if 200 <= N <= (64e6 if dtype == "c64" else 16e6):
                return dict(kind=kind, n=n, D=D, layers=rng.randint(1, 5) if N < 2e7 else rng.randint(1, 2), dtype=dtype)
    mixed = rng.random() < 0.4
    n, D = _ket_size(rng, 30, 3000, nmin=2, nmax=4) if mixed else _ket_size(rng, 500, 4e6)
    return dict(kind="readout", n=n, D=D, mixed=mixed, dtype="c128")


# ---------------------------------------------------------------- circuits of a case
def _random_gates(n, D, count, structure):
    """A seeded random program over every pure-state gate kind: (name, modes) list."""
    r = np.random.default_rng([structure, n, D])
    ops = [("S", (i,)) for i in range(n)]
    kinds = ["D", "R", "K", "BS", "BS", "S2", "MZ", "CK", "V"]
    while len(ops) < n + count:
        k = kinds[int(r.integers(len(kinds)))]
        a, b = (int(v) for v in r.choice(n, 2, replace=False))
        ops.append((k, (a, b) if k in ("BS", "S2", "MZ", "CK") else (a,)))
    return ops


def _ops(case):
    """The circuit's operations (name, modes); its parameters come from _params."""
    if case["kind"] == "gates":
        return _random_gates(case["n"], case["D"], case["count"], case["structure"])
    if case["kind"] == "engine":
        n, ops = case["n"], []
        for i in range(n):
            ops += [("S", (i,)), ("D", (i,)), ("R", (i,))]
        ops += [("BS", p) for p in circuits.mesh_pairs(n)]
        return ops + [("K", (i,)) for i in range(n)]
    loss = case["kind"] == "dm"
    return [o[:2] for o in circuits.layered(case["n"], case["layers"], np.random.default_rng(0), loss=loss)]


def _params(ops, dtype, rng, sd=0.1):
    """Gate parameters [nops, 2] of a circuit in training: beamsplitters anywhere, the rest small."""
    rows = np.zeros((len(ops), 2))
    for i, (name, _) in enumerate(ops):
        if name == "BS":
            rows[i] = rng.uniform(0, np.pi / 2), rng.normal(0, sd)
        elif name == "MZ":
            rows[i] = rng.uniform(0, 2 * np.pi, 2)
        elif name == "LOSS":
            rows[i, 0] = rng.uniform(0.7, 1.0)
        elif name in ("D", "S", "S2"):
            rows[i] = rng.normal(0, sd, 2)
        elif name == "V":
            rows[i, 0] = rng.normal(0, sd / 4)
        else:
            rows[i, 0] = rng.normal(0, sd)
    return torch.tensor(rows, dtype=torch.float64).to(REAL[dtype])


def _batch(case):
    r = np.random.default_rng(case["structure"])
    out = []
    while len(out) < case["count"]:
        n, D, L = int(r.integers(2, 6)), int(r.integers(6, 21)), int(r.integers(2, 5))
        if D**n <= case["maxamps"]:
            out.append(dict(n=n, D=D, ops=[o[:2] for o in circuits.layered(n, L, np.random.default_rng(0))]))
    return out


def _vacuum(n, D, dtype, mixed=False):
    st = torch.zeros([D] * (2 * n if mixed else n), dtype=DTYPES[dtype], device="cuda")
    st.view(-1)[0] = 1.0
    return st


def _photons(n, D, device="cuda"):
    """Total photon number of every Fock state, [D]*n float64."""
    k = torch.arange(D, dtype=torch.float64, device=device)
    tot = torch.zeros([D] * n, dtype=torch.float64, device=device)
    for m in range(n):
        tot = tot + k.reshape([-1 if i == m else 1 for i in range(n)])
    return tot


def _target(case, gen):
    """A seeded normalised target ket over at most n photons, mostly vacuum-like as a goal state is."""
    n, D = case["n"], case["D"]
    tot = _photons(n, D)
    v = torch.randn([D] * n, dtype=torch.complex128, device="cuda", generator=gen)
    v = v * torch.exp(-tot) * (tot <= n)
    v = (v / v.abs().square().sum().sqrt()).to(DTYPES[case["dtype"]])
    return v


def _readout_state(case, gen):
    """A normalised state whose amplitudes fall with the photon number."""
    n, D = case["n"], case["D"]
    amp = torch.exp(-0.35 * _photons(n, D))
    kets = [torch.randn([D] * n, dtype=torch.complex128, device="cuda", generator=gen) * amp
            for _ in range(2 if case["mixed"] else 1)]
    kets = [k / k.abs().square().sum().sqrt() for k in kets]
    if not case["mixed"]:
        return kets[0]
    perm = [a for m in range(n) for a in (m, n + m)]
    rho = sum(w * torch.outer(k.reshape(-1), k.reshape(-1).conj()) for w, k in zip((0.7, 0.3), kets))
    return rho.reshape([D] * (2 * n)).permute(perm).contiguous()


def _inputs(case, seed):
    """What the seed determines, shared by prepare and exact."""
    rng = np.random.default_rng([seed, 7])
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)
    kind = case["kind"]
    if kind == "readout":
        return dict(state=_readout_state(case, gen), phi=float(rng.uniform(0, np.pi)))
    if kind == "batch":
        return dict(params=[_params(c["ops"], case["dtype"], rng).cuda() for c in _batch(case)])
    ops = _ops(case)
    got = dict(ops=ops, params=_params(ops, case["dtype"], rng, 0.25 if kind == "engine" else 0.1))
    if kind != "engine":
        got["params"] = got["params"].cuda()
    if kind in ("graph", "grad", "gates"):
        got["target"] = _target(case, gen)
    return got


# ---------------------------------------------------------------- prepare and run
_GATES = {"S": frontend.Sgate, "D": frontend.Dgate, "R": frontend.Rgate, "K": frontend.Kgate, "BS": frontend.BSgate}
BINS = 20000


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    s["case"] = dict(case)
    if kind == "readout":
        s["fock"] = FockStateHIP(s["state"], case["n"], not case["mixed"], case["D"])
        return s
    if kind == "batch":
        circs = _batch(case)
        s["batch"] = runtime.BatchEvaluator(circs, DTYPES[case["dtype"]], "cuda")
        return s
    n, D, ops = case["n"], case["D"], s["ops"]
    if kind == "engine":
        prog = frontend.Program(n)
        with prog.context as q:
            for (name, modes), row in zip(ops, s["params"].tolist()):
                args = row if name in ("S", "D", "BS") else row[:1]
                _GATES[name](*args) | tuple(q[m] for m in modes)
        s["prog"] = prog
        s["engine"] = frontend.Engine(HIPFockBackend(), backend_options={"cutoff_dim": D, "dtype": DTYPES[case["dtype"]]})
        return s
    mixed = kind == "dm"
    s["plan"] = runtime.CompiledCircuit(ops, n, D, mixed, DTYPES[case["dtype"]], torch.device("cuda:0"))
    s["vacuum"] = _vacuum(n, D, case["dtype"], mixed)
    if kind == "graph":
        s["evaluator"] = runtime.GradEvaluator(s["plan"], s["vacuum"], s["target"])
    elif kind == "dm":
        s["weight"] = (_photons(n, D) - n) ** 2
    if kind in ("grad", "gates", "dm"):
        s["params"].requires_grad_(True)
    elif kind == "fwd":
        s["params64"] = s["params"].double()
    return s


def run(s):
    case = s["case"]
    kind, real = case["kind"], REAL[case["dtype"]]
    if kind == "readout":
        st, n, D, mixed = s["fock"], case["n"], case["D"], case["mixed"]
        probs = st.all_fock_probs()
        mean = [st.mean_photon(m) for m in range(n)]
        pair = st.reduced_dm([0, 1])
        one = st.reduced_dm([n - 1])
        marg = runtime.marginal_probs(s["state"], n, D, mixed, [0, n - 1] if n > 1 else [0])
        pdf = runtime.homodyne_pdf(one, D, s["phi"], 8.0, BINS, 2.0)
        return dict(probs=probs, mean=[v for p in mean for v in p], pair=pair, one=one, marginal=marg, pdf=pdf, trace=st.trace())
    if kind == "batch":
        losses, grads = s["batch"]([p.double() for p in s["params"]])
        return dict(loss=losses.to(real), grad=[g.to(real) for g in grads])
    if kind == "engine":
        s["engine"].reset()
        st = s["engine"].run(s["prog"]).state
        return dict(ket=st.ket(), probs=st.all_fock_probs(), mean=[NUMPY[case["dtype"]](st.mean_photon(m)[0]) for m in range(case["n"])])
    if kind == "fwd":
        return dict(ket=runtime.run_circuit(s["plan"], s["params64"], s["vacuum"]))
    if kind == "graph":
        loss, grads = s["evaluator"](s["params"])
        return dict(loss=loss.to(real), grad=grads.to(real), ket=s["evaluator"].psi)
    s["params"].grad = None
    out = runtime.run_circuit(s["plan"], s["params"].double(), s["vacuum"], 24 if kind == "dm" else None)
    if kind == "dm":
        probs = runtime.all_fock_probs(out, case["n"], case["D"], True)
        loss = (probs.double() * s["weight"]).sum()
        loss.backward()
        return dict(loss=loss.detach().to(real), grad=s["params"].grad, probs=probs.detach(), rho=out.detach())
    loss = runtime.fidelity_loss(out, s["target"])
    loss.backward()
    return dict(loss=loss.detach().to(real), grad=s["params"].grad, ket=out.detach())


# ---------------------------------------------------------------- what a pass cannot do without
_TWO = ("BS", "S2", "MZ", "CK")


def _op_flops(name, n, D, mixed):
    N = float(D) ** (2 * n if mixed else n)
    if name in ("R", "K"):
        f = 6.0 * N
    elif name == "CK":
        f = 6.0 * N
    elif name in _TWO:  # sum of c(s)^2 over the blocks of D^2 amplitudes
        f = 8.0 * N * (2.0 * D * D + 1) / (3.0 * D)
    elif name == "LOSS":
        return 4.0 * N * (D + 1) / 3.0
    else:
        f = 8.0 * N * (D if name != "S" else D / 2.0)
    return 2.0 * f if mixed else f


def work(case):
    kind = case["kind"]
    esz = 8 if case["dtype"] == "c64" else 16
    if kind == "readout":
        n, D = case["n"], case["D"]
        N = float(D) ** (2 * n if case["mixed"] else n)
        out = float(D) ** n * 8 + D**4 * esz + BINS * 8
        fl = 8.0 * (D**2) * float(D) ** n if not case["mixed"] else 2.0 * N / D ** max(0, n - 2)
        return dict(bytes=(N * esz if not case["mixed"] else float(D) ** (n + 2) * esz) + out, flops=fl + BINS * 2.0 * D * D)
    parts = _batch(case) if kind == "batch" else [dict(n=case["n"], D=case["D"], ops=_ops(case))]
    mixed = kind == "dm"
    grad = kind in ("graph", "grad", "gates", "batch", "dm")
    nbytes = flops = 0.0
    for c in parts:
        N = float(c["D"]) ** (2 * c["n"] if mixed else c["n"])
        flops += (3.0 if grad else 1.0) * sum(_op_flops(o[0], c["n"], c["D"], mixed) for o in c["ops"])
        nbytes += 16.0 * len(c["ops"]) * (2 if grad else 1)
        if kind in ("fwd", "engine", "grad", "gates"):
            nbytes += N * esz  # the state returned
        if kind in ("graph", "grad", "gates"):
            nbytes += N * esz  # the target read
        if kind != "batch":
            nbytes += N * esz  # the input state read
    return dict(bytes=nbytes, flops=flops)


# ---------------------------------------------------------------- the same in 64 bits
def _ladder(M):
    return torch.diag(torch.sqrt(torch.arange(1, M, dtype=torch.float64)), 1)


def _phase(w, p):
    return torch.polar(torch.ones_like(w), w * p)


def _single(name, p, D):
    """The truncated [D, D] matrix of a single-mode gate, differentiable in p (CPU, 64 bits)."""
    k = torch.arange(D, dtype=torch.float64)
    if name == "R":
        return torch.diag(_phase(k, p[0]))
    if name == "K":
        return torch.diag(_phase(k * k, p[0]))
    if name == "V":
        x = _ladder(D)
        x = (x + x.T).to(torch.complex128)
        return torch.linalg.matrix_exp(1j * p[0] / 6.0 * (x @ x @ x))
    M = D + 70
    a = _ladder(M)
    if name == "D":
        U, w = torch.linalg.matrix_exp(p[0] * (a.T - a))[:D, :D], 1.0
    else:
        U, w = torch.linalg.matrix_exp(0.5 * p[0] * (a @ a - a.T @ a.T))[:D, :D], 0.5
    return _phase(w * (k[:, None] - k[None, :]), p[1]) * U


def _conserving(theta, D):
    """exp(theta (a b^+ - a^+ b)) as [N, M, n, m] for N, n, M, m < D, block by total photon number."""
    S = 2 * D - 1
    s, k = torch.arange(S, dtype=torch.float64)[:, None], torch.arange(S - 1, dtype=torch.float64)[None, :]
    off = torch.sqrt(torch.clamp((k + 1) * (s - k), min=0.0)) * (k < s)  # <k| a b^+ |k + 1>
    gen = torch.diag_embed(off, 1) - torch.diag_embed(off, -1)
    E = torch.linalg.matrix_exp(theta * gen)  # [s, N, n]
    N, M, n, m = _grid(D)
    return E[(N + M).clamp(max=S - 1), N, n] * (N + M == n + m)


def _grid(D):
    return torch.meshgrid(*[torch.arange(D)] * 4, indexing="ij")


def _double(name, p, D):
    """The truncated [N, M, n, m] tensor of a two-mode gate, differentiable in p (CPU, 64 bits)."""
    N, M, n, m = _grid(D)
    if name == "CK":
        return _phase((n * m).double(), p[0]) * ((N == n) & (M == m))
    if name == "BS":
        return _phase((n - N).double(), p[1]) * _conserving(p[0], D)
    if name == "S2":
        Z = D + 70  # difference blocks d = n - m >= 0 of the pairs (k + d, k)
        d, k = torch.arange(D, dtype=torch.float64)[:, None], torch.arange(Z - 1, dtype=torch.float64)[None, :]
        off = torch.sqrt((k + d + 1) * (k + 1))
        E = torch.linalg.matrix_exp(p[0] * (torch.diag_embed(off, -1) - torch.diag_embed(off, 1)))
        lo_out, lo_in = torch.minimum(N, M), torch.minimum(n, m)
        return _phase((N - n).double(), p[1]) * E[(n - m).abs(), lo_out, lo_in] * (N - M == n - m)
    # MZ = B R(phi_in) B R(phi_ex) with B = BS(pi/4, pi/2), exact at cutoff 2 D - 1
    L = 2 * D - 1
    s, k = torch.arange(L, dtype=torch.float64)[:, None], torch.arange(L - 1, dtype=torch.float64)[None, :]
    off = torch.sqrt(torch.clamp((k + 1) * (s - k), min=0.0)) * (k < s)
    gen = torch.diag_embed(off, 1) - torch.diag_embed(off, -1)
    j = torch.arange(L, dtype=torch.float64)
    B = _phase(j[None, :] - j[:, None], torch.tensor(math.pi / 2, dtype=torch.float64)) * torch.linalg.matrix_exp(math.pi / 4 * gen)
    E = (B * _phase(j, p[0])) @ (B * _phase(j, p[1]))
    return E[(N + M).clamp(max=L - 1), N, n] * (N + M == n + m)


def _axis(x, U, axes):
    """U [k, k] on the listed axes of x (taken together as one index)."""
    k = len(axes)
    y = torch.movedim(x, axes, list(range(k)))
    shape = y.shape
    return torch.movedim((U @ y.reshape(U.shape[1], -1)).reshape(shape), list(range(k)), axes)


def _loss64(x, T, D, bra, ket):
    y = torch.movedim(x, (bra, ket), (0, 1))
    lg = torch.lgamma(torch.arange(2 * D, dtype=torch.float64, device=x.device) + 1)
    k = torch.arange(D, device=x.device)
    out = torch.zeros_like(y)
    for l in range(D):
        i = k[: D - l]
        binom = 0.5 * (lg[i + l] - lg[i] - lg[l])
        c = torch.exp(binom[:, None] + binom[None, :]) * T ** ((i[:, None] + i[None, :]).double() / 2) * (1 - T) ** l
        part = y[l:, l:] * c.reshape(list(c.shape) + [1] * (x.dim() - 2))
        a = D - l
        out = out.clone() if out.requires_grad else out
        out[:a, :a] += part
    return torch.movedim(out, (0, 1), (bra, ket))


def _apply64(x, name, modes, p, n, D, mixed):
    if name == "LOSS":
        return _loss64(x, p[0].to(x.device), D, 2 * modes[0], 2 * modes[0] + 1)
    p = p.cpu()
    if name in _TWO:
        U = _double(name, p, D).reshape(D * D, D * D)
    else:
        U = _single(name, p, D)
    U = U.to(torch.complex128).to(x.device)
    if not mixed:
        return _axis(x, U, list(modes))
    x = _axis(x, U, [2 * m for m in modes])
    return _axis(x, U.conj(), [2 * m + 1 for m in modes])


def _run64(ops, params, x, n, D, mixed, chunk=6):
    """The circuit on x; with gradients, states are kept every `chunk` operations."""

    def part(x, params, b, e):
        for i in range(b, e):
            x = _apply64(x, ops[i][0], ops[i][1], params[i], n, D, mixed)
        return x

    if not params.requires_grad:
        return part(x, params, 0, len(ops))
    for b in range(0, len(ops), chunk):
        x = checkpoint(part, x, params, b, min(b + chunk, len(ops)), use_reentrant=False)
    return x


def _vacuum64(n, D, mixed=False):
    return _vacuum(n, D, "c128", mixed)


def _loss_grad64(ops, params, n, D, mixed, loss_of):
    p = params.detach().double().requires_grad_(True)
    out = _run64(ops, p, _vacuum64(n, D, mixed), n, D, mixed)
    loss = loss_of(out)
    loss.backward()
    return loss.detach(), p.grad, out.detach()


def _hermite_pdf(rho, D, phi, q, hbar=2.0):
    """sum_ab rho[a, b] e^{-i phi (a - b)} u_a(x) u_b(x) dx with the oscillator functions u_n."""
    x = q / math.sqrt(hbar)
    u = [math.pi**-0.25 * torch.exp(-0.5 * x * x)]
    for k in range(1, D):
        v = math.sqrt(2.0 / k) * x * u[-1]
        u.append(v - math.sqrt((k - 1.0) / k) * u[-2] if k > 1 else v)
    k = torch.arange(D, dtype=torch.float64, device=rho.device)
    u = torch.stack(u).to(torch.complex128) * torch.exp(-1j * phi * k)[:, None]
    dx = (q[1] - q[0]) / math.sqrt(hbar)
    return ((rho @ u.conj()) * u).sum(0).real * dx


def _reduced64(x, n, D, mixed, modes):
    rest = [m for m in range(n) if m not in modes]
    k = len(modes)
    if mixed:
        perm = [a for m in modes for a in (2 * m, 2 * m + 1)] + [2 * r for r in rest] + [2 * r + 1 for r in rest]
        y = x.permute(perm).reshape(D ** (2 * k), D ** (n - k), D ** (n - k))
        return y.diagonal(dim1=1, dim2=2).sum(-1).reshape([D] * (2 * k))
    y = x.permute(list(modes) + rest).reshape(D**k, D ** (n - k))
    r = (y @ y.conj().T.contiguous()).reshape([D] * (2 * k))
    return r.permute([a for i in range(k) for a in (i, k + i)])


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batch":
        losses, grads = [], []
        for c, p in zip(_batch(case), s["params"]):
            w = _photons(c["n"], c["D"])
            l, g, _ = _loss_grad64(c["ops"], p, c["n"], c["D"], False, lambda x: (x.abs().square() * w).sum())
            losses.append(l)
            grads.append(g)
        return dict(loss=torch.stack(losses), grad=grads)
    n, D = case["n"], case["D"]
    if kind == "readout":
        x, mixed = s["state"], case["mixed"]
        if mixed:
            perm = [2 * m for m in range(n)] + [2 * m + 1 for m in range(n)]
            probs = x.permute(perm).reshape(D**n, D**n).diagonal().real.reshape([D] * n)
        else:
            probs = x.real**2 + x.imag**2
        k = torch.arange(D, dtype=torch.float64, device="cuda")
        mean = []
        for m in range(n):
            pm = probs.sum([a for a in range(n) if a != m])
            mu = float((pm * k).sum())
            mean += [mu, float((pm * k * k).sum()) - mu * mu]
        one = _reduced64(x, n, D, mixed, [n - 1])
        marg = probs.sum(list(range(1, n - 1))) if n > 2 else probs
        q = torch.linspace(-8.0, 8.0, BINS, dtype=torch.float64, device="cuda")
        return dict(probs=probs, mean=mean, pair=_reduced64(x, n, D, mixed, [0, 1]), one=one, marginal=marg,
                    pdf=_hermite_pdf(one, D, s["phi"], q), trace=float(probs.sum()))
    ops = s["ops"]
    if kind in ("engine", "fwd"):
        ket = _run64(ops, s["params"].detach().double().cpu(), _vacuum64(n, D), n, D, False)
        if kind == "fwd":
            return dict(ket=ket)
        probs = ket.real**2 + ket.imag**2
        k = torch.arange(D, dtype=torch.float64, device="cuda")
        mean = [(probs.sum([a for a in range(n) if a != m]) * k).sum() for m in range(n)]
        return dict(ket=ket, probs=probs, mean=mean)
    if kind == "dm":
        w = (_photons(n, D) - n) ** 2
        perm = [2 * m for m in range(n)] + [2 * m + 1 for m in range(n)]

        def probs_of(x):
            return x.permute(perm).reshape(D**n, D**n).diagonal().real.reshape([D] * n)

        l, g, x = _loss_grad64(ops, s["params"], n, D, True, lambda x: (probs_of(x) * w).sum())
        return dict(loss=l, grad=g, probs=probs_of(x).contiguous(), rho=x)
    t = s["target"].to(torch.complex128)

    def infidelity(x):
        ov = (t.conj() * x).sum()
        return 1.0 - ov.real**2 - ov.imag**2

    l, g, x = _loss_grad64(ops, s["params"], n, D, False, infidelity)
    return dict(loss=l, grad=g, ket=x)
