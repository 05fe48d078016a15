"""Device runtime: planned circuits, the differentiable circuit Function, readout.

A circuit is a list of ``(name, modes)`` operations with one row of two real
parameters per operation.  ``CompiledCircuit`` plans it once on the library
(``sfamd_prog_create``), owns the device workspaces, and runs

* the gate-table build (all matrices of the circuit, FP64 recurrences, one
  launch per 96 operations) from a device parameter vector,
* the forward sweep, writing requested operation inputs as checkpoints,
* the adjoint sweep, which returns the state cotangent and every parameter
  gradient.

``CircuitFunction`` wraps this in ``torch.autograd.Function``: the backward
recomputes each checkpoint segment forward and runs the hand-written adjoint
kernels over it (truncated Fock gates are not unitary, so the reverse sweep
needs the forward states; it cannot un-compute them).

This replaces the TF backend's tape (``tfbackend/circuit.py:72-76`` keeps every
state; ``tfbackend/ops.py:190-204,318-366`` give the per-gate VJPs).
"""
import collections
import ctypes
import math
import threading

import numpy as np
import torch

from . import _lib

# default memory budget for keeping every operation input alive in backward
DEFAULT_SAVE_BUDGET = 16 * 2**30
# step inputs that the differentiable forwards on a device keep, all together,
# without a look at its free memory (a 4500th of the card)
KEEP_ALWAYS = 64 * 2**20


def _elem_bytes(dtype):
    return 8 if dtype == torch.complex64 else 16


def default_fuse(n, D):
    """Local modes per fused stage (stage kernels exist for cutoffs 2..20).

    Three, and more at the lowest cutoffs, where a tile of three modes leaves
    the matrix cores idle and a stage takes few gates: one layer of the layered
    circuit, forward and adjoint, with 3 / 4 / 5 / 6 local modes took 541 / 414 /
    339 / 407 us on 10 modes at cutoff 3, 300 / 221 / 255 us on 8 at cutoff 4, 1024 /
    727 / 787 us on 8 at cutoff 5, 395 / 337 us on 7 and 2074 / 1730 us on 8 at cutoff
    6, but 132 / 161 us on 5 modes at cutoff 6.  Cutoffs above 16 take two (three
    keep too few gates' tiles in LDS for the adjoint)."""
    if n < 2 or D < 2 or D > 20:
        return 0
    want = 5 if D <= 3 else 4 if D <= 5 or (D == 6 and n >= 7) else 3 if D <= 16 else 2
    return min(want, n)


class _KeptInputs:
    """A share of the bytes that differentiable forwards may keep on a device, held
    with what is kept and given back when the backward is done with it or the
    graph is freed."""

    _lock = threading.Lock()
    _held = {}  # by device, what was given back not yet subtracted
    _back = collections.deque()  # appended to by __del__, which may run anywhere and takes no lock

    def __init__(self, device, nbytes):
        self.share = (device, nbytes)

    def __del__(self):
        self._back.append(self.share)

    @classmethod
    def reserve(cls, device, nbytes):
        """The share, or None: beyond KEEP_ALWAYS bytes in all, at most a quarter of
        the free memory goes to one forward and DEFAULT_SAVE_BUDGET to all."""
        with cls._lock:
            while cls._back:
                dev, n = cls._back.popleft()
                cls._held[dev] -= n
            held = cls._held.get(device, 0) + nbytes
            if held > KEEP_ALWAYS and (
                held > DEFAULT_SAVE_BUDGET
                or torch.cuda.is_current_stream_capturing()
                or nbytes > torch.cuda.mem_get_info(device)[0] // 4
            ):
                return None
            cls._held[device] = held
            return cls(device, nbytes)


class CompiledCircuit:
    """A planned circuit (structure only) bound to one device and dtype.

    The plan is a list of steps: fused stages (many gates on LDS tiles of
    ``fuse`` local modes) or single operations.  The default (``fuse=None``)
    stages gates where enough of them share a tile to pay; a number asks for
    stages of that many local modes however few gates they hold, and 0 for
    none.  Checkpoints and segments are expressed in steps; gradients are
    indexed by operation.
    """

    def __init__(self, ops, n, D, mixed_in, dtype, device, fuse=None):
        self.lib = _lib.load()
        self.ops = [(name, tuple(int(m) for m in modes)) for name, modes in ops]
        self.n, self.D, self.mixed_in = int(n), int(D), bool(mixed_in)
        self.dtype = dtype
        self.code = _lib.dtype_code(dtype)
        self.device = torch.device(device)
        arr = (_lib.OpDesc * max(1, len(self.ops)))()
        for i, (name, modes) in enumerate(self.ops):
            arr[i].kind = _lib.OP_KINDS[name]
            arr[i].mode0 = modes[0] if len(modes) > 0 else -1
            arr[i].mode1 = modes[1] if len(modes) > 1 else -1
            arr[i].pad = 0
        handle = ctypes.c_void_p()
        self.fuse = default_fuse(self.n, self.D) if fuse is None else int(fuse)
        fuse_K = self.fuse | _lib.FUSE_MIXED if self.fuse >= 2 else self.fuse
        if fuse is None and self.fuse >= 2:
            fuse_K |= _lib.FUSE_PAYING
        st = self.lib.sfamd_prog_create(
            arr, len(self.ops), self.n, self.D, int(self.mixed_in), self.code, fuse_K, ctypes.byref(handle)
        )
        _lib.check(st, "sfamd_prog_create")
        self.handle = handle
        info = _lib.ProgInfo()
        _lib.check(self.lib.sfamd_prog_info(handle, ctypes.byref(info)), "sfamd_prog_info")
        self.info = info
        self.nops = len(self.ops)
        self.nsteps = info.nsteps
        self.final_mixed = bool(info.final_mixed)
        self.state_elems = [self.lib.sfamd_prog_state_elems(handle, i) for i in range(self.nsteps + 1)]
        full = self.D ** (2 * self.n)
        self.mixed_at = [e == full and (self.n > 0 and (self.D > 1 or self.mixed_in)) for e in self.state_elems]
        if self.D == 1:  # sizes cannot tell kets from DMs
            self.mixed_at = [self.mixed_in] * (self.nsteps + 1)
            self.mixed_at[-1] = self.final_mixed
        buf = (ctypes.c_int32 * max(1, self.nops))()
        self.step_ops = []
        for i in range(self.nsteps):
            k = self.lib.sfamd_prog_step_ops(handle, i, buf, self.nops)
            self.step_ops.append([buf[j] for j in range(k)])
        dev = self.device
        self.table = torch.empty(max(1, info.table_elems), dtype=dtype, device=dev)
        self.ws = torch.empty(max(1, info.ws_elems), dtype=dtype, device=dev)
        self.partial = torch.empty(max(1, info.partial_doubles), dtype=torch.float64, device=dev)
        self._built = None

    def __del__(self):
        h = getattr(self, "handle", None)
        if h is not None and h.value:
            try:
                self.lib.sfamd_prog_destroy(h)
            except Exception:  # interpreter shutdown
                pass
            self.handle = None

    def step_kinds(self, forward_only=False):
        """How each step runs: "op", "diag" (a run of R / K gates), "vector" or
        "matrix" (stages); forward_only: the steps of a run without gradients."""
        kinds, i = [], 0
        while (k := self.lib.sfamd_prog_step_kind(self.handle, int(forward_only), i)) >= 0:
            kinds.append(("op", "diag", "vector", "matrix")[k])
            i += 1
        return kinds

    # ---- shapes
    def state_shape(self, i):
        return [self.D] * (2 * self.n if self.mixed_at[i] else self.n)

    def state_bytes(self, i):
        return self.state_elems[i] * _elem_bytes(self.dtype)

    def new_state(self, i):
        return torch.empty(self.state_shape(i), dtype=self.dtype, device=self.device)

    # ---- launches
    def _stream(self):
        return _lib.stream_ptr(self.device)

    def build_table(self, params, force=True):
        """Gate tables from params (float64 [nops, 2] on the device).

        With force=False the build is skipped when the table already holds
        this exact parameter tensor (same object, unmodified), as between the
        forward and the backward of one evaluation.
        """
        assert params.dtype == torch.float64 and params.is_contiguous()
        if self.nops == 0:
            return
        key = (id(params), params._version)
        if not force and self._built is not None and self._built[0] is params and self._built[1] == key:
            return
        _lib.call(
            "sfamd_prog_build_table", self.handle, _lib.ptr(params), _lib.ptr(self.table), self._stream()
        )
        self._built = (params, key)

    def forward(self, begin, end, state_in, out=None, saved=None):
        """Run steps [begin, end) on state_in; saved[j] receives the input of step begin+j."""
        if out is None:
            out = self.new_state(end)
        sv = None
        if saved is not None:
            sv = (ctypes.c_void_p * max(1, end - begin))()
            for j, t in enumerate(saved):
                sv[j] = t.data_ptr() if t is not None else None
        _lib.call(
            "sfamd_prog_forward",
            self.handle,
            begin,
            end,
            _lib.ptr(self.table),
            _lib.ptr(state_in),
            _lib.ptr(out),
            sv,
            _lib.ptr(self.ws),
            self._stream(),
        )
        return out

    def run(self, state_in, out=None):
        """The whole program without checkpoints (nothing is differentiated)."""
        if out is None:
            out = self.new_state(self.nsteps)
        _lib.call(
            "sfamd_prog_run",
            self.handle,
            _lib.ptr(self.table),
            _lib.ptr(state_in),
            _lib.ptr(out),
            _lib.ptr(self.ws),
            self._stream(),
        )
        return out

    def adjoint(self, begin, end, saved, g_out, g_in, grads):
        sv = (ctypes.c_void_p * max(1, end - begin))()
        for j, t in enumerate(saved):
            sv[j] = t.data_ptr()
        _lib.call(
            "sfamd_prog_adjoint",
            self.handle,
            begin,
            end,
            _lib.ptr(self.table),
            sv,
            _lib.ptr(g_out),
            _lib.ptr(g_in),
            _lib.ptr(grads),
            _lib.ptr(self.partial),
            _lib.ptr(self.ws),
            self._stream(),
        )

    # ---- checkpoint plan
    def segments(self, segment=None, budget=DEFAULT_SAVE_BUDGET):
        """Split the steps [0, nsteps) into checkpoint segments.

        segment=None keeps every step input when they fit in `budget` bytes,
        else uses segments of ~sqrt(nsteps) steps; an int gives the segment
        length in steps.  Within a segment the backward recomputes the
        forward from the segment's checkpoint (the last segment's inputs may be
        kept, see keeps_inputs).
        """
        ns = self.nsteps
        if ns == 0:
            return []
        if segment is None:
            total = sum(self.state_bytes(i) for i in range(ns))
            if total <= budget:
                segment = ns
            else:
                segment = max(1, int(math.ceil(math.sqrt(ns))))
        segment = max(1, int(segment))
        return [(b, min(b + segment, ns)) for b in range(0, ns, segment)]

    def keeps_inputs(self, b, e):
        """May a differentiable forward keep the inputs of the last segment's steps b..e?

        The backward begins with that segment, so keeping them saves one
        recomputation (3 modes, cutoff 11, 3 layers, complex128: 478 -> 388 us
        a gradient; 6 modes, cutoff 16, 1 layer, complex64, 45 states of 134 MB:
        11.2 -> 8.7 ms).  The first backward takes them and frees them with that
        segment, so that it never holds two segments; a further one over a
        retained graph recomputes them.  Under saved-tensor hooks (checkpointing,
        offloading) none are kept: those save as little as they can.
        Returns the share of the memory that the forward holds on to (see
        _KeptInputs), or None.
        """
        if e - b < 2 or torch._C._autograd._top_saved_tensors_default_hooks(True) is not None:
            return None
        return _KeptInputs.reserve(self.table.device, sum(self.state_bytes(i) for i in range(b + 1, e)))


def _params_row(p):
    """Two float64 parameter slots (tensor, keeps autograd) of one operation."""
    out = []
    for v in list(p)[:2]:
        if isinstance(v, torch.Tensor):
            out.append(v.reshape(()).to(torch.float64))
        else:
            out.append(torch.tensor(float(v), dtype=torch.float64))
    while len(out) < 2:
        out.append(torch.tensor(0.0, dtype=torch.float64))
    return out


def params_tensor(ops_params, device):
    """Stack per-op parameters into a float64 [nops, 2] device tensor (differentiable)."""
    rows = []
    for p in ops_params:
        rows.extend(_params_row(p))
    if not rows:
        return torch.zeros((0, 2), dtype=torch.float64, device=device)
    flat = torch.stack([r.cpu() if r.device.type != "cpu" else r for r in rows])
    return flat.reshape(-1, 2).to(device)


class CircuitFunction(torch.autograd.Function):
    """state_out = circuit(params, state_in), with the hand-written adjoint as backward."""

    @staticmethod
    def forward(ctx, params, state_in, cc, segment):
        params = params.detach().contiguous()
        state_in = state_in.detach().contiguous()
        cc.build_table(params)
        segs = cc.segments(segment)
        ckpts = []
        inner = []
        ctx.kept = None
        cur = state_in
        for (b, e) in segs:
            ckpts.append(cur)
            if e == cc.nsteps:
                ctx.kept = cc.keeps_inputs(b, e)
                if ctx.kept:
                    inner = [cc.new_state(i) for i in range(b + 1, e)]
            cur = cc.forward(b, e, cur, saved=[cur] + inner if inner else None)
        ctx.cc = cc
        ctx.segs = segs
        ctx.params = params
        ctx.inner = inner  # the last segment's step inputs, until the first backward
        ctx.save_for_backward(*ckpts)
        return cur if segs else state_in.clone()

    @staticmethod
    def backward(ctx, g_out):
        cc = ctx.cc
        if not ctx.segs:
            return None, g_out, None, None
        ckpts = ctx.saved_tensors  # read once: every read unpacks them again under saved-tensor hooks
        inner, ctx.inner = ctx.inner, []
        kept, ctx.kept = ctx.kept, None
        # the gate table may have been rebuilt by another run of the same plan
        cc.build_table(ctx.params, force=False)
        grads = torch.zeros(cc.nops * 2, dtype=torch.float64, device=cc.device)
        lam = g_out.to(cc.dtype).contiguous()
        for si in range(len(ctx.segs) - 1, -1, -1):
            b, e = ctx.segs[si]
            saved = [ckpts[si]] + inner
            if not inner:
                saved += [cc.new_state(i) for i in range(b + 1, e)]
                if e - b > 1:
                    cc.forward(b, e - 1, ckpts[si], out=saved[-1], saved=saved[:-1])
            g_in = cc.new_state(b)
            cc.adjoint(b, e, saved, lam, g_in, grads)
            lam = g_in
            # one segment at a time (the device frees in stream order)
            inner, saved, kept = [], None, None
        return grads.reshape(-1, 2), lam, None, None


def run_circuit(cc, params, state_in, segment=None):
    """Differentiable execution when params or state_in require grad, plain otherwise."""
    if torch.is_grad_enabled() and (params.requires_grad or state_in.requires_grad):
        return CircuitFunction.apply(params, state_in, cc, segment)
    params = params.detach().contiguous()
    cc.build_table(params)
    if cc.nsteps == 0:
        return state_in.clone()
    return cc.run(state_in.detach().contiguous())


# --------------------------------------------------------------------- readout
def _scratch(n, dtype, device):
    return torch.empty(max(1, n), dtype=dtype, device=device)


def norm2(state, n, D, mixed):
    """<psi|psi> or Tr rho, FP64 accumulation; returns a 0-dim float64 device tensor."""
    lib = _lib.load()
    dev = state.device
    part = _scratch(lib.sfamd_reduce_partials(n, D, int(mixed)), torch.float64, dev)
    out = torch.empty(1, dtype=torch.float64, device=dev)
    _lib.call(
        "sfamd_norm",
        _lib.ptr(state),
        n,
        D,
        int(mixed),
        _lib.ptr(part),
        _lib.ptr(out),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(dev),
    )
    return out[0]


class _ProbsFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, state, n, D, mixed):
        state = state.detach().contiguous()
        probs = torch.empty([D] * n, dtype=_lib.real_dtype(state.dtype), device=state.device)
        _lib.call(
            "sfamd_all_fock_probs",
            _lib.ptr(state),
            _lib.ptr(probs),
            n,
            D,
            int(mixed),
            _lib.dtype_code(state.dtype),
            _lib.stream_ptr(state.device),
        )
        ctx.save_for_backward(state)
        ctx.n, ctx.D, ctx.mixed = n, D, mixed
        return probs

    @staticmethod
    def backward(ctx, g):
        (state,) = ctx.saved_tensors
        g = g.to(_lib.real_dtype(state.dtype)).contiguous()
        gs = torch.empty_like(state)
        _lib.call(
            "sfamd_all_fock_probs_vjp",
            _lib.ptr(state),
            _lib.ptr(g),
            _lib.ptr(gs),
            ctx.n,
            ctx.D,
            int(ctx.mixed),
            _lib.dtype_code(state.dtype),
            _lib.stream_ptr(state.device),
        )
        return gs, None, None, None


def all_fock_probs(state, n, D, mixed):
    return _ProbsFunction.apply(state, n, D, mixed)


def reduced_dm(state, n, D, mixed, modes):
    """Reduced DM of sorted `modes` ([D]*2k, interleaved) straight from the state."""
    lib = _lib.load()
    k = len(modes)
    dev = state.device
    part = _scratch(lib.sfamd_reduced_dm_partials(n, D, k, int(mixed)), torch.float64, dev)
    out = torch.empty([D] * (2 * k), dtype=state.dtype, device=dev)
    arr = (ctypes.c_int * max(1, k))(*modes)
    _lib.call(
        "sfamd_reduced_dm",
        _lib.ptr(state.contiguous()),
        _lib.ptr(out),
        n,
        D,
        int(mixed),
        arr,
        k,
        _lib.ptr(part),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(dev),
    )
    return out


def _reduced_dm_torch(state, n, D, mixed, modes):
    """The reduced DM as torch contractions on the device (differentiable):
    rho_red = M M^H with M the ket's kept modes x the rest, or the trace of
    the DM over the rest modes' (bra, ket) pairs (states.py:613-642)."""
    rest = [m for m in range(n) if m not in modes]
    k = len(modes)
    if mixed:
        perm = [a for m in modes for a in (2 * m, 2 * m + 1)] + [2 * r for r in rest] + [2 * r + 1 for r in rest]
        x = state.permute(perm).reshape(D ** (2 * k), D ** (n - k), D ** (n - k))
        return x.diagonal(dim1=1, dim2=2).sum(-1).reshape([D] * (2 * k))
    m = state.permute(list(modes) + rest).reshape(D**k, D ** (n - k))
    r = (m @ m.conj().transpose(0, 1).contiguous()).reshape([D] * (2 * k))
    return r.permute([a for i in range(k) for a in (i, k + i)])


class ReducedDM(torch.autograd.Function):
    """Reduced DM of sorted `modes` with a gradient: the forward is the
    library's reduction kernel; the backward differentiates the same
    contraction written as torch matrix products on the device (the TF
    backend's reduced_dm is differentiable, tfbackend/states.py:307)."""

    @staticmethod
    def forward(ctx, state, n, D, mixed, modes):
        ctx.save_for_backward(state)
        ctx.meta = (n, D, mixed, list(modes))
        return reduced_dm(state.detach(), n, D, mixed, list(modes))

    @staticmethod
    def backward(ctx, g):
        (state,) = ctx.saved_tensors
        n, D, mixed, modes = ctx.meta
        with torch.enable_grad():
            s = state.detach().requires_grad_(True)
            (gs,) = torch.autograd.grad(_reduced_dm_torch(s, n, D, mixed, modes), s, g)
        return gs, None, None, None, None


def diagonal_expectation(state, n, D, mixed, modes, values):
    """sum_I p(I) prod_{m in modes} values[I_m] (FP64); returns a 0-dim float64 tensor."""
    lib = _lib.load()
    dev = state.device
    k = len(modes)
    part = _scratch(lib.sfamd_reduce_partials(n, D, int(mixed)), torch.float64, dev)
    out = torch.empty(1, dtype=torch.float64, device=dev)
    vals = torch.as_tensor(np.asarray(values, dtype=np.float64)).to(dev)
    arr = (ctypes.c_int * max(1, k))(*modes)
    _lib.call(
        "sfamd_diagonal_expectation",
        _lib.ptr(state.contiguous()),
        n,
        D,
        int(mixed),
        arr,
        k,
        _lib.ptr(vals),
        _lib.ptr(part),
        _lib.ptr(out),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(dev),
    )
    return out[0]


def mix(ket, n, D):
    dm = torch.empty([D] * (2 * n), dtype=ket.dtype, device=ket.device)
    _lib.call(
        "sfamd_mix",
        _lib.ptr(ket.contiguous()),
        _lib.ptr(dm),
        n,
        D,
        _lib.dtype_code(ket.dtype),
        _lib.stream_ptr(ket.device),
    )
    return dm


def replace_mode(dm, n, D, mode, sigma):
    """rho' = sigma (x) Tr_mode(rho) with sigma a [D, D] device matrix."""
    out = torch.empty_like(dm)
    _lib.call(
        "sfamd_replace_mode",
        _lib.ptr(dm.contiguous()),
        _lib.ptr(out),
        n,
        D,
        mode,
        _lib.ptr(sigma.to(dm.dtype).contiguous()),
        _lib.dtype_code(dm.dtype),
        _lib.stream_ptr(dm.device),
    )
    return out


def marginal_probs(state, n, D, mixed, modes):
    """Fock distribution of the sorted `modes` (float64 device tensor [D]*k)."""
    lib = _lib.load()
    k = len(modes)
    dev = state.device
    part = _scratch(lib.sfamd_marginal_partials(n, D, k), torch.float64, dev)
    out = torch.empty([D] * k, dtype=torch.float64, device=dev)
    arr = (ctypes.c_int * max(1, k))(*modes)
    _lib.call(
        "sfamd_marginal_probs",
        _lib.ptr(state.contiguous()),
        n,
        D,
        int(mixed),
        arr,
        k,
        _lib.ptr(part),
        _lib.ptr(out),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(dev),
    )
    return out


def project_reset(state, n, D, mixed, modes, outcome, scale):
    """scale * |0><outcome| on `modes` (both sides of a DM)."""
    k = len(modes)
    out = torch.empty_like(state)
    _lib.call(
        "sfamd_project_reset",
        _lib.ptr(state.contiguous()),
        _lib.ptr(out),
        n,
        D,
        int(mixed),
        (ctypes.c_int * max(1, k))(*[int(m) for m in modes]),
        (ctypes.c_int * max(1, k))(*[int(x) for x in outcome]),
        k,
        float(scale),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(state.device),
    )
    return out


def homodyne_pdf(rho, D, phi, q_mag, num_bins, hbar):
    """Homodyne density of a single-mode DM on the linspace(-q_mag, q_mag, num_bins)
    grid (float64 device tensor, sums to ~1 for a state inside the cutoff)."""
    out = torch.empty(num_bins, dtype=torch.float64, device=rho.device)
    _lib.call(
        "sfamd_homodyne_pdf",
        _lib.ptr(rho.contiguous()),
        D,
        float(phi),
        float(q_mag),
        int(num_bins),
        float(hbar),
        _lib.ptr(out),
        _lib.dtype_code(rho.dtype),
        _lib.stream_ptr(rho.device),
    )
    return out


def apply_matrix(state, n, D, mixed, mode, U):
    """Single-mode matrix U [D, D] on `mode` (U rho U^dagger on a DM)."""
    out = torch.empty_like(state)
    tmp = torch.empty_like(state) if mixed else None
    _lib.call(
        "sfamd_apply_matrix",
        _lib.ptr(state.contiguous()),
        _lib.ptr(out),
        _lib.ptr(tmp) if tmp is not None else None,
        n,
        D,
        mode,
        int(mixed),
        _lib.ptr(U.to(state.dtype).contiguous()),
        _lib.dtype_code(state.dtype),
        _lib.stream_ptr(state.device),
    )
    return out


def embed_modes(rest, sigma, n, D, modes, mixed):
    """rest (x) sigma with sigma's axes on `modes` (any order), see sfamd_embed_modes."""
    dev = sigma.device
    out = torch.empty([D] * (2 * n if mixed else n), dtype=sigma.dtype, device=dev)
    k = len(modes)
    _lib.call(
        "sfamd_embed_modes",
        _lib.ptr(rest.contiguous()) if rest is not None else None,
        _lib.ptr(sigma.contiguous()),
        _lib.ptr(out),
        n,
        D,
        (ctypes.c_int * k)(*[int(m) for m in modes]),
        k,
        int(mixed),
        _lib.dtype_code(sigma.dtype),
        _lib.stream_ptr(dev),
    )
    return out


def build_gate(kind, p0, p1, D, dtype, device):
    """Gate-table entry of one gate (matrix + derivatives) as a flat device tensor."""
    lib = _lib.load()
    code = _lib.OP_KINDS[kind]
    size = lib.sfamd_gate_table_size(code, D)
    if size < 0:
        raise ValueError("cutoff %d not supported for gate %s" % (D, kind))
    out = torch.empty(max(1, size), dtype=dtype, device=device)
    _lib.call(
        "sfamd_build_gate",
        code,
        float(p0),
        float(p1),
        D,
        _lib.dtype_code(dtype),
        _lib.ptr(out),
        _lib.stream_ptr(torch.device(device)),
    )
    return out


def gate_matrix(kind, p0, p1, D, dtype, device):
    """Dense [D, D] matrix of a single-mode gate (R and K as diagonal matrices)."""
    t = build_gate(kind, p0, p1, D, dtype, device)
    if kind in ("R", "K"):
        return torch.diag(t[:D])
    return t[: D * D].reshape(D, D)


# --------------------------------------------------------------------- fidelity loss
def overlap(a, b):
    """<a|b> over all amplitudes (FP64 accumulation); 0-dim complex128 device tensor."""
    lib = _lib.load()
    n = a.numel()
    part = _scratch(lib.sfamd_overlap_partials(n), torch.float64, a.device)
    out = torch.empty(3, dtype=torch.float64, device=a.device)
    _lib.call(
        "sfamd_overlap",
        _lib.ptr(a.contiguous()),
        _lib.ptr(b.contiguous()),
        n,
        _lib.ptr(part),
        _lib.ptr(out),
        _lib.dtype_code(a.dtype),
        _lib.stream_ptr(a.device),
    )
    return torch.complex(out[0], out[1])


class FidelityLoss(torch.autograd.Function):
    """L = 1 - |<target|psi>|^2 and its cotangent -2 <target|psi> target, in one library call."""

    @staticmethod
    def forward(ctx, psi, target):
        lib = _lib.load()
        psi = psi.detach().contiguous()
        target = target.detach().to(psi.dtype).contiguous()
        n = psi.numel()
        part = _scratch(lib.sfamd_overlap_partials(n), torch.float64, psi.device)
        out = torch.empty(3, dtype=torch.float64, device=psi.device)
        g = torch.empty_like(psi)
        _lib.call(
            "sfamd_fidelity_loss",
            _lib.ptr(target),
            _lib.ptr(psi),
            n,
            _lib.ptr(part),
            _lib.ptr(out),
            _lib.ptr(g),
            _lib.dtype_code(psi.dtype),
            _lib.stream_ptr(psi.device),
        )
        ctx.save_for_backward(g)
        return out[2]

    @staticmethod
    def backward(ctx, gl):
        (g,) = ctx.saved_tensors
        return g * gl.to(g.real.dtype), None


def fidelity_loss(psi, target):
    return FidelityLoss.apply(psi, target)


class GradEvaluator:
    """One captured gradient evaluation of L = 1 - |<target|psi(params)>|^2.

    All buffers (parameters, every step input, cotangents, gradients) are
    allocated once; the gate-table build, the fused forward, the loss and the
    adjoint sweep are recorded into one HIP graph on a private stream and
    replayed per call.  Parameters are copied into the static buffer before
    each replay.  Requires the whole plan's step inputs to fit in memory.
    """

    def __init__(self, cc, state_in, target, use_graph=True, forward_only=False):
        lib = _lib.load()
        self.cc = cc
        dev = cc.device
        self.stream = torch.cuda.Stream(device=dev)
        self.params = torch.zeros((cc.nops, 2), dtype=torch.float64, device=dev)
        self.state_in = state_in.detach().to(cc.dtype).contiguous().clone()
        self.target = target.detach().to(cc.dtype).contiguous().clone().reshape(-1)
        self.saved = [self.state_in] + [cc.new_state(i) for i in range(1, cc.nsteps)]
        self.psi = cc.new_state(cc.nsteps)
        self.g_psi = torch.empty_like(self.psi)
        self.g_in = cc.new_state(0)
        self.grads = torch.zeros(cc.nops * 2, dtype=torch.float64, device=dev)
        self.out = torch.zeros(3, dtype=torch.float64, device=dev)
        self.part = torch.empty(max(1, lib.sfamd_overlap_partials(self.psi.numel())), dtype=torch.float64, device=dev)
        self.graph = None
        self.forward_only = forward_only
        torch.cuda.synchronize(dev)
        with torch.cuda.stream(self.stream):
            self._enqueue()  # eager run: warms the kernels, checks every call
        self.stream.synchronize()
        if use_graph:
            sp = ctypes.c_void_p(self.stream.cuda_stream)
            _lib.call("sfamd_graph_begin", sp)
            try:
                with torch.cuda.stream(self.stream):
                    self._enqueue()
            finally:
                g = ctypes.c_void_p()
                _lib.call("sfamd_graph_end", sp, ctypes.byref(g))
            self.graph = g
        self.stream.synchronize()

    def _enqueue(self):
        cc = self.cc
        cc.build_table(self.params)
        if self.forward_only:
            cc.run(self.state_in, out=self.psi)
        else:
            cc.forward(0, cc.nsteps, self.state_in, out=self.psi, saved=self.saved[: cc.nsteps])
        _lib.call(
            "sfamd_fidelity_loss",
            _lib.ptr(self.target),
            _lib.ptr(self.psi),
            self.psi.numel(),
            _lib.ptr(self.part),
            _lib.ptr(self.out),
            None if self.forward_only else _lib.ptr(self.g_psi),
            cc.code,
            _lib.stream_ptr(cc.device),
        )
        if not self.forward_only:
            cc.adjoint(0, cc.nsteps, self.saved[: cc.nsteps], self.g_psi, self.g_in, self.grads)

    def __call__(self, params):
        """Returns (loss, grads [nops, 2]) as device tensors valid until the next call."""
        cur = torch.cuda.current_stream(self.cc.device)
        self.stream.wait_stream(cur)
        with torch.cuda.stream(self.stream):
            self.params.copy_(params.detach().reshape(self.cc.nops, 2))
            if self.graph is not None:
                _lib.call("sfamd_graph_launch", self.graph, ctypes.c_void_p(self.stream.cuda_stream))
            else:
                self._enqueue()
        # the replay rewrote the shared gate table: a pending autograd backward
        # of the same plan must rebuild it from its own parameters
        self.cc._built = None
        cur.wait_stream(self.stream)
        return self.out[2], self.grads.reshape(self.cc.nops, 2)

    def __del__(self):
        g = getattr(self, "graph", None)
        if g is not None:
            try:
                _lib.load().sfamd_graph_destroy(g)
            except Exception:
                pass
            self.graph = None


# --------------------------------------------------------------------- autotuning
# counts the changes of what a number of local modes means to the planner: a
# choice stored under another number was measured on other kernels
PLAN_REVISION = 2


def _structure_key(ops, n, D, mixed, dtype, forward_only=False):
    import hashlib

    h = hashlib.sha1(repr([(name, tuple(m)) for name, m in ops]).encode()).hexdigest()[:16]
    what = "f" if forward_only else "g"
    return "v%d%s:%d:%d:%d:%s:%s" % (PLAN_REVISION, what, n, D, int(mixed), str(dtype).split(".")[-1], h)


class Autotuner:
    """Measures the stage tile (local modes K per fused stage, 0 = one kernel
    per gate) for a circuit structure and caches the fastest.

    Candidates are the K with plans of their own (a K without stage kernels for
    the cutoff falls back to another plan); each is timed with HIP events on
    random parameters, over a forward + adjoint sweep or, for circuits that are
    only run, over the run.  The choice is cached in memory and, when `path` is
    set (default $SFAMD_AUTOTUNE_CACHE), in a JSON file keyed by the planner's
    revision, what was timed, (modes, cutoff, mixed, dtype, structure hash).
    """

    def __init__(self, path=None, reps=3):
        import json
        import os

        self.path = path if path is not None else os.environ.get("SFAMD_AUTOTUNE_CACHE")
        self.reps = reps
        self.cache = {}
        if self.path and os.path.exists(self.path):
            try:
                with open(self.path) as f:
                    self.cache = json.load(f)
            except (OSError, ValueError):
                self.cache = {}

    def _save(self):
        import json

        if self.path:
            try:
                with open(self.path, "w") as f:
                    json.dump(self.cache, f, indent=0, sort_keys=True)
            except OSError:
                pass

    def _time(self, run, dev):
        run()
        torch.cuda.synchronize(dev)
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(self.reps):
            run()
        e1.record()
        torch.cuda.synchronize(dev)
        return e0.elapsed_time(e1) * 1e3 / self.reps

    @staticmethod
    def candidates(n, D, mixed):
        if n < 2 or not 2 <= D <= 20:
            return [0]
        # stages of more than three modes have tiles of at most 4096 amplitudes; on a density matrix
        # a stage of two modes has the tile of three axes
        return [0] + [K for K in range(3 if mixed else 2, 7) if (mixed or K <= n) and (K <= 3 or D**K <= 4096)]

    def best(self, ops, n, D, mixed, dtype, device, forward_only=False):
        key = _structure_key(ops, n, D, mixed, dtype, forward_only)
        if key in self.cache:
            return self.cache[key]["fuse"]
        cands = self.candidates(n, D, mixed)
        if len(cands) == 1:
            self.cache[key] = {"fuse": cands[0], "us": {}}
            return cands[0]
        dev = torch.device(device)
        gen = torch.Generator(device="cpu").manual_seed(0)
        params = (torch.rand((len(ops), 2), generator=gen, dtype=torch.float64) * 0.3).to(dev)
        st = torch.zeros([D] * (2 * n if mixed else n), dtype=dtype, device=dev)
        st.view(-1)[0] = 1.0
        times = {}
        plans = []
        for K in cands:
            cc = CompiledCircuit(ops, n, D, mixed, dtype, dev, fuse=K)
            kinds = cc.step_kinds(forward_only)
            if "vector" not in kinds and "matrix" not in kinds:
                plan = None  # one kernel per gate
            else:
                plan = K if forward_only else (kinds, cc.step_ops)
            if plan in plans:
                continue  # timed under a smaller K
            plans.append(plan)
            cc.build_table(params)
            if forward_only:
                out = cc.new_state(cc.nsteps)
                times[K] = self._time(lambda: cc.run(st, out=out), dev)
                continue
            saved = [st] + [cc.new_state(i) for i in range(1, cc.nsteps)]
            out = cc.new_state(cc.nsteps)
            lam = torch.randn_like(out)
            gin = cc.new_state(0)
            grads = torch.zeros(2 * len(ops), dtype=torch.float64, device=dev)

            def run():
                cc.forward(0, cc.nsteps, st, out=out, saved=saved)
                cc.adjoint(0, cc.nsteps, saved, lam, gin, grads)

            times[K] = self._time(run, dev)
        best = min(times, key=times.get)
        self.cache[key] = {"fuse": best, "us": {str(k): round(v, 2) for k, v in times.items()}}
        self._save()
        return best


# --------------------------------------------------------------------- batches
def deal_by_work(works, nbranches):
    """Items dealt to `nbranches` branches so that the branches end together:
    largest first, each to the branch with the least work so far (ties to the
    lowest branch).  Returns the item indices of each branch, in dealing order."""
    order = sorted(range(len(works)), key=lambda i: (-works[i], i))
    load = [0.0] * nbranches
    out = [[] for _ in range(nbranches)]
    for k in order:
        b = min(range(nbranches), key=lambda j: (load[j], j))
        out[b].append(k)
        load[b] += works[k]
    return out


class BatchEvaluator:
    """Gradient of the total mean photon number of many independent pure-state
    circuits, replayed from ONE captured HIP graph.

    Each circuit is planned with the autotuned stage tile and owns its buffers
    (every step input, cotangents, gradients).  The capture forks the circuits
    over `nstreams` streams (independent graph branches the GPU runs
    concurrently, so small circuits fill the compute units left idle by large
    ones) and joins them before the graph ends.  Most circuits of a mixed batch
    are small and bound by per-launch latency, so many branches pay: on the
    256-circuit workload 8 streams give 5.3 batches/s, 32 give 9.5 and 64 give
    9.8.  A call copies every circuit's parameters into its static buffer and
    launches the graph once.
    """

    def __init__(self, circuits, dtype=torch.complex64, device="cuda", nstreams=64, tuner=None, use_graph=True):
        lib = _lib.load()
        dev = torch.device(device)
        self.device = dev
        self.tuner = tuner if tuner is not None else Autotuner()
        self.items = []
        offset = 0
        for c in circuits:
            ops = [(o[0], tuple(o[1])) for o in c["ops"]]
            n, D = c["n"], c["D"]
            K = self.tuner.best(ops, n, D, False, dtype, dev)
            cc = CompiledCircuit(ops, n, D, False, dtype, dev, fuse=K)
            st = torch.zeros([D] * n, dtype=dtype, device=dev)
            st.view(-1)[0] = 1.0
            it = {
                "cc": cc,
                "n": n,
                "D": D,
                "off": offset,
                "params": torch.zeros((len(ops), 2), dtype=torch.float64, device=dev),
                "saved": [st] + [cc.new_state(i) for i in range(1, cc.nsteps)],
                "psi": cc.new_state(cc.nsteps),
                "g_in": cc.new_state(0),
                "grads": torch.zeros(2 * len(ops), dtype=torch.float64, device=dev),
                "part": torch.empty(max(1, lib.sfamd_reduce_partials(n, D, 0)), dtype=torch.float64, device=dev),
            }
            it["g_psi"] = torch.empty_like(it["psi"])
            offset += len(ops)
            self.items.append(it)
        self.nparams_rows = offset
        self.losses = torch.zeros(len(self.items), dtype=torch.float64, device=dev)
        self.main = torch.cuda.Stream(device=dev)
        self.streams = [torch.cuda.Stream(device=dev) for _ in range(nstreams)]
        self.assign = deal_by_work([self._work(it) for it in self.items], nstreams)
        self.graph = None
        torch.cuda.synchronize(dev)
        self._enqueue_all()
        torch.cuda.synchronize(dev)
        if use_graph:
            sp = ctypes.c_void_p(self.main.cuda_stream)
            _lib.call("sfamd_graph_begin", sp)
            try:
                self._enqueue_all()
            finally:
                g = ctypes.c_void_p()
                _lib.call("sfamd_graph_end", sp, ctypes.byref(g))
            self.graph = g
        torch.cuda.synchronize(dev)

    @staticmethod
    def _work(it):
        # per step: a fixed launch and latency cost (about that of streaming
        # 2^18 amplitudes) plus the state's size
        return max(1, it["cc"].nsteps) * (1.0 + it["psi"].numel() / float(1 << 18))

    def _enqueue_one(self, it, k):
        cc = it["cc"]
        cc.build_table(it["params"])
        cc.forward(0, cc.nsteps, it["saved"][0], out=it["psi"], saved=it["saved"][: cc.nsteps])
        _lib.call(
            "sfamd_number_loss",
            _lib.ptr(it["psi"]),
            _lib.ptr(it["g_psi"]),
            it["n"],
            it["D"],
            _lib.ptr(it["part"]),
            _lib.ptr(self.losses[k : k + 1]),
            cc.code,
            _lib.stream_ptr(cc.device),
        )
        cc.adjoint(0, cc.nsteps, it["saved"][: cc.nsteps], it["g_psi"], it["g_in"], it["grads"])

    def _enqueue_all(self):
        fork = torch.cuda.Event()
        fork.record(self.main)
        joins = []
        for si, s in enumerate(self.streams):
            s.wait_event(fork)
            with torch.cuda.stream(s):
                for k in self.assign[si]:
                    self._enqueue_one(self.items[k], k)
            ev = torch.cuda.Event()
            ev.record(s)
            joins.append(ev)
        for ev in joins:
            self.main.wait_event(ev)

    def __call__(self, params_list):
        """params_list: one float64 [nops, 2] tensor per circuit. Returns
        (losses [ncircuits], list of gradient tensors [nops, 2]) on the device."""
        cur = torch.cuda.current_stream(self.device)
        self.main.wait_stream(cur)
        with torch.cuda.stream(self.main):
            for it, p in zip(self.items, params_list):
                it["params"].copy_(p.detach().reshape(it["params"].shape))
            if self.graph is not None:
                _lib.call("sfamd_graph_launch", self.graph, ctypes.c_void_p(self.main.cuda_stream))
            else:
                self._enqueue_all()
        for it in self.items:  # gate tables rewritten (see GradEvaluator.__call__)
            it["cc"]._built = None
        cur.wait_stream(self.main)
        return self.losses, [it["grads"].reshape(-1, 2) for it in self.items]

    def __del__(self):
        g = getattr(self, "graph", None)
        if g is not None:
            try:
                _lib.load().sfamd_graph_destroy(g)
            except Exception:
                pass
            self.graph = None
