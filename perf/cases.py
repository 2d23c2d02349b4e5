"""Performance cases of the engine: whole calls through its public Python
entry points, over the sizes, solver options and call styles it is used with.

The engine refuses a process whose HIP runtime another library brought
(torch's wheel bundles one under the same soname), and a program that uses
both keeps them in processes of their own.  So the cases run the engine in one
worker process that never imports torch: ``prepare`` builds the problem and
the context there, ``run`` asks it for one pass, and outputs come back in
memory that both processes map.  Every entry point used here returns when its
work is done.
"""
import gc
import json
import math
import mmap
import os
import socket
import subprocess
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# The step size a run starts with here.  Nearly all steps of a cycle
# simulation are interseismic ones of 1e5 s and more, with two to three
# V-cycles a solve; from the default 1e-3 s a run spends its first 20 steps
# growing the step instead.
INI_DT = 1.0e4


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest production grid: every launch of a V-cycle is short, so
        # latency and launch counts decide
        dict(name="cycle_129", kind="cycle", problem="bp1", ni=129, nk=129, levels=4,
             solver="fast64", start="plain", tune=True, steps=20),
        # the usual run: the basin problem at 1025^2, FP64, 1e-10 relative
        dict(name="cycle_1025", kind="cycle", problem="basin", ni=1025, nk=1025, levels=7,
             solver="fast64", start="plain", tune=True, steps=40),
        # the same run with the projection start of its stage solves
        dict(name="cycle_1025_projection", kind="cycle", problem="basin", ni=1025, nk=1025,
             levels=7, solver="fast64", start="projection", tune=True, steps=40),
        # the largest grid: FP32 V-cycles in FP64 refinement at 2049^2
        dict(name="cycle_2049_ir", kind="cycle", problem="basin", ni=2049, nk=2049, levels=8,
             solver="fast32", start="plain", tune=True, steps=10),
        # a grid of another size in the reference's medium, wider than deep,
        # with the tile shapes a context has without the tuner
        dict(name="cycle_801x481", kind="cycle", problem="reference", ni=801, nk=481, levels=6,
             solver="fast64", start="plain", tune=False, steps=20),
        # the parity run: the reference's own V-cycle (32 sweeps, absolute
        # stop rule) on the small problem
        dict(name="reference_129", kind="cycle", problem="bp1", ni=129, nk=129, levels=4,
             solver="reference", start="plain", tune=False, steps=6),
        # the reference's own problem with its own V-cycle
        dict(name="reference_801", kind="cycle", problem="reference", ni=801, nk=801, levels=6,
             solver="reference", start="plain", tune=False, steps=3),
        # a small ensemble of uneven grids stepped together, FP32 refinement
        dict(name="ensemble_6", kind="ensemble", sizes="257 513 257 1025 257 513",
             solver="fast32", steps=10),
        # the drop-in functions of one RK stage, called one by one on the
        # caller's host arrays, at the usual size ...
        dict(name="stage_1025", kind="stage", ni=1025, nk=1025, levels=7, solver="fast64"),
        # ... and with the default configuration on a small grid
        dict(name="stage_257_reference", kind="stage", ni=257, nk=257, levels=5,
             solver="reference"),
        # training of the learned start on pairs harvested from a run
        dict(name="train_513", kind="train", nk=513, pairs=480, batch=160, epochs=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """(n, levels): n = m 2^(levels-1) + 1 nodes, m odd or even in 8..20."""
    m = rng.randint(8, 20)
    levels = max(2, int(round(math.log2(_log_int(rng, lo, hi) / m))) + 1)
    while m * 2 ** (levels - 1) + 1 > hi:
        levels -= 1
    return m * 2 ** (levels - 1) + 1, levels


def draw(rng):
    kind = rng.choice(["cycle", "cycle", "cycle", "reference", "ensemble", "stage", "train"])
    if kind == "cycle":
        n, levels = _grid(rng, 65, 2049)
        solver = rng.choice(["fast64", "fast64", "fast32"])
        problem = rng.choice(["bp1", "basin", "reference"])
        nk = n
        if problem == "reference":  # not square: another m on the same levels
            nk = max(8, min(20, (n - 1) // 2 ** (levels - 1) + rng.randint(-5, 5))) \
                * 2 ** (levels - 1) + 1
        if nk > 2049:
            nk = n
        start = "projection" if solver == "fast64" and n <= 1025 and rng.random() < 0.3 \
            else "plain"
        steps = max(6, min(40, int(4.0e7 / (n * nk)) + rng.randint(0, 4)))
        return dict(kind="cycle", problem=problem, ni=n, nk=nk, levels=levels, solver=solver,
                    start=start, tune=rng.random() < 0.7, steps=steps)
    if kind == "reference":
        n, levels = _grid(rng, 65, 641)
        return dict(kind="cycle", problem=rng.choice(["bp1", "basin"]), ni=n, nk=n,
                    levels=levels, solver="reference", start="plain", tune=False,
                    steps=2 + rng.randint(0, 2))
    if kind == "ensemble":
        sizes = [rng.choice([129, 257, 257, 513]) for _ in range(rng.randint(2, 6))]
        return dict(kind="ensemble", sizes=" ".join(map(str, sizes)),
                    solver=rng.choice(["fast64", "fast32"]), steps=rng.randint(5, 10))
    if kind == "stage":
        if rng.random() < 0.5:
            n, levels = _grid(rng, 65, 1281)
            return dict(kind="stage", ni=n, nk=n, levels=levels, solver="fast64")
        n, levels = _grid(rng, 65, 321)
        return dict(kind="stage", ni=n, nk=n, levels=levels, solver="reference")
    return dict(kind="train", nk=rng.choice([129, 257, 385, 513]),
                pairs=rng.randint(100, 400), batch=rng.choice([50, 128, 200]),
                epochs=rng.randint(4, 10))


def work(case):
    """What a pass cannot do without: a V-cycle reads each level's unknowns,
    right-hand side and face coefficients once and writes its unknowns and the
    coarse right-hand side once; 11 operations per point and sweep, 12 per
    residual, 6 for the transfers."""
    if case["kind"] == "train":
        nk, H = case["nk"], 512
        nout = ((nk - 1) // 4 + 1) ** 2
        params = 64 + 2 * (nk - 1) * H + 2 * H * H + nout * H
        steps = case["epochs"] * -(-case["pairs"] // case["batch"])
        return {"bytes": 24.0 * params * steps + 4.0 * case["epochs"] * case["pairs"] * (nk + nout),
                "flops": 6.0 * params * case["epochs"] * case["pairs"]}
    if case["kind"] == "ensemble":
        points = sum(int(s) ** 2 for s in case["sizes"].split())
    else:
        points = case["ni"] * case["nk"]
    word = 4.0 if case["solver"] == "fast32" else 8.0
    sweeps = 64 if case["solver"] == "reference" else 4
    if case["kind"] == "stage":
        vcycles = 2 * 2.0
        host = 8.0 * points * 2
    else:
        per_solve = 1.5 if case.get("start") == "projection" else 2.2
        vcycles = per_solve * (6 * case["steps"] + 1)
        host = 8.0 * points * 2
    # level 0 has no right-hand side (FP64) or gets one from the FP64 residual
    level0 = 4.0 * word if word == 8.0 else 5.0 * word + 5 * 8.0
    return {"bytes": vcycles * points * (level0 + 6.0 * word / 3.0) + host,
            "flops": vcycles * points * (4.0 / 3.0) * (11.0 * sweeps + 2 * 12.0 + 6.0)}


# ---------------------------------------------------------------------------
# The caller's side
# ---------------------------------------------------------------------------

class _Worker:
    """The engine's process and the calls to it."""

    def __init__(self):
        here, there = socket.socketpair()
        self.proc = subprocess.Popen(
            [sys.executable, "-u", os.path.abspath(__file__), str(there.fileno())],
            cwd=ROOT, stdin=subprocess.DEVNULL, stdout=sys.stderr, pass_fds=[there.fileno()])
        there.close()
        self.sock = here
        self.owner = os.getpid()

    def call(self, **msg):
        _send(self.sock, msg)
        reply, fds = _receive(self.sock)
        if reply is None:
            raise RuntimeError("the engine's process ended (%s)" % self.proc.poll())
        if "error" in reply:
            raise RuntimeError(reply["error"])
        return reply, fds


class _State:
    """A prepared case: its number in the worker and the mapped outputs."""

    def __init__(self, worker, case, seed):
        self.worker = worker
        reply, fds = worker.call(do="new", case=case, seed=seed)
        self.id = reply["id"]
        with os.fdopen(fds[0], "rb") as f:
            self.map = mmap.mmap(f.fileno(), reply["size"], prot=mmap.PROT_READ)
        self.arrays = _views(self.map, reply["arrays"])

    def __del__(self):
        try:
            if self.worker.owner == os.getpid() and self.worker.proc.poll() is None:
                self.worker.call(do="drop", id=self.id)
        except Exception:
            pass


_worker = None


def prepare(case, seed):
    global _worker
    if _worker is None or _worker.proc.poll() is not None or _worker.owner != os.getpid():
        _worker = _Worker()
    return _State(_worker, {k: v for k, v in case.items() if k != "name"}, seed)


def run(state):
    reply, _ = state.worker.call(do="run", id=state.id)
    return {**reply["values"], **state.arrays}


# ---------------------------------------------------------------------------
# Both sides: messages and the shared output block
# ---------------------------------------------------------------------------

def _send(sock, msg, fds=()):
    data = json.dumps(msg).encode()
    data = len(data).to_bytes(8, "little") + data
    if fds:
        n = socket.send_fds(sock, [data], list(fds))
        data = data[n:]
    if data:
        sock.sendall(data)


def _receive(sock):
    data, fds = b"", []
    need = 8
    while len(data) < need:
        more, got, _, _ = socket.recv_fds(sock, 1 << 16, 4)
        if not more:
            return None, []
        fds += got
        data += more
        if need == 8 and len(data) >= 8:
            need = 8 + int.from_bytes(data[:8], "little")
    return json.loads(data[8:need]), fds


def _layout(arrays):
    """[name, dtype, shape, offset] of each array in one block, and its size."""
    out, at = [], 0
    for name, dtype, shape in arrays:
        out.append([name, dtype, list(shape), at])
        at += -(-int(np.prod(shape)) * np.dtype(dtype).itemsize // 4096) * 4096
    return out, max(at, 4096)


def _views(block, layout):
    return {name: np.frombuffer(block, dtype, int(np.prod(shape)), at).reshape(shape)
            for name, dtype, shape, at in layout}


# ---------------------------------------------------------------------------
# Inputs (the same from the same seed, wherever they are made)
# ---------------------------------------------------------------------------

def _problem(case, seed):
    """A case's problem with the seed's friction: Dc log-uniform in
    [4, 16] mm, normal stress uniform in [25, 75] MPa, b uniform in
    [0.013, 0.018] (the reference problem keeps its own stress and b profile
    but for a factor)."""
    import dataclasses

    from qdeqcycle_fdm_amd import config

    rng = np.random.default_rng([seed, 11])
    Dc = float(math.exp(rng.uniform(math.log(0.004), math.log(0.016))))
    sigma_n, b = float(rng.uniform(25.0, 75.0)), float(rng.uniform(0.013, 0.018))
    problem = case.get("problem", "bp1")
    if problem == "reference":
        pb = config.make_reference_problem(case["ni"], case["nk"], 24000.0 / (case["ni"] - 1))
        pb = dataclasses.replace(pb, b=pb.b * (b / 0.0155))
    else:
        pb = config.make_bp1_problem(case["ni"], basin=problem == "basin", Dc=Dc,
                                     sigma_n=sigma_n, b_seis=b)
    params = dataclasses.replace(pb.params, n_levels=case["levels"], L=Dc, ini_dt=INI_DT)
    return dataclasses.replace(pb, params=params)


_SOLVERS = {
    # the engine's production cycle, FP64 and FP32 in FP64 refinement
    "fast64": dict(cycle=1, precision=0, n_pre=1, n_post=3, n_coarse=0, relax=1.15, tol_mode=1,
                   tol=1e-10),
    "fast32": dict(cycle=1, precision=1, n_pre=1, n_post=3, n_coarse=0, relax=1.15, tol_mode=1,
                   tol=1e-10),
    # the reference's cycle and stop rule (the defaults)
    "reference": dict(),
}


def _stage_inputs(case, seed):
    """Fault data of two successive stages around a smooth slip profile, and
    the friction inputs of the fault update, length nz."""
    pb = _problem(dict(case, problem="bp1"), seed)
    rng = np.random.default_rng([seed, 12])
    nk, nz = case["nk"], case["nk"] + 2
    z = np.zeros(nz)
    z[1:nk + 1] = np.linspace(0.0, 1.0, nk)
    base = pb.U0[:, 1] * 2.0
    slips = []
    for amp in (0.10, 0.11):
        s = np.zeros(nz)
        for m in range(1, 6):
            s += rng.normal() / m * np.cos(math.pi * m * z)
        s[1:nk + 1] = base[1:nk + 1] + amp * s[1:nk + 1]
        s[0] = s[-1] = 0.0
        slips.append(s)
    p = pb.params
    psi = np.zeros(nz)
    psi[1:nk + 1] = p.f0 + pb.b[1:nk + 1] * math.log(p.V0 / p.Vini) \
        + 0.01 * rng.normal(size=nk)
    V = np.zeros(nz)
    V[1:nk + 1] = 1e-9
    shift = np.ascontiguousarray(pb.U0[:, case["ni"]])
    return pb, slips, shift, psi, V


# ---------------------------------------------------------------------------
# The engine's side: one object per prepared case
# ---------------------------------------------------------------------------

_STATE_KEYS = ("slip", "psi", "V", "dpsi", "Ts")


def _state_arrays(prefix, pb):
    p = pb.params
    return [(prefix + "U", "f8", (p.nz, p.nx))] + \
        [(prefix + k, "f8", (p.nz,)) for k in _STATE_KEYS] + \
        [(prefix + "times", "f8", (2,)), (prefix + "counts", "i8", (3,))]


def _write_state(out, prefix, st):
    for k in ("U",) + _STATE_KEYS:
        np.copyto(out[prefix + k], st[k])
    info = st["info"]
    out[prefix + "times"][:] = info["t"], info["dt"]
    out[prefix + "counts"][:] = info["it"], info["vcycles"], info["solves"]


class _Cycle:
    """A simulation of its own: set up, stepped, its state read."""

    def __init__(self, case, seed):
        from qdeqcycle_fdm_amd import lib
        self.pb = _problem(case, seed)
        self.steps = case["steps"]
        kw = dict(_SOLVERS[case["solver"]])
        if case["start"] == "projection":
            kw["tol"] = 1e-11
        self.eng = lib.Engine(self.pb, **kw)
        if case["tune"]:
            self.eng.autotune_tiles()
        if case["start"] == "projection":
            self.eng.projection_enable(8)
        self.arrays = _state_arrays("", self.pb)

    def run(self, out):
        self.eng.rk43_setup()
        self.eng.rk43_step(self.steps)
        _write_state(out, "", self.eng.state())
        return {}


class _Ensemble:
    """Independent simulations stepped together from one thread."""

    def __init__(self, case, seed):
        from qdeqcycle_fdm_amd import lib
        self.steps, self.eng, self.arrays = case["steps"], [], []
        shapes = {}
        for m, n in enumerate(int(s) for s in case["sizes"].split()):
            levels = int(round(math.log2((n - 1) / 16))) + 1
            pb = _problem(dict(problem="basin", ni=n, nk=n, levels=levels), 1000 * seed + m)
            eng = lib.Engine(pb, **_SOLVERS[case["solver"]])
            if n in shapes:
                eng.set_tile_shapes(shapes[n])
            else:
                shapes[n] = eng.autotune_tiles()
            self.eng.append(eng)
            self.arrays += _state_arrays("m%d_" % m, pb)

    def run(self, out):
        from qdeqcycle_fdm_amd import lib
        for eng in self.eng:
            eng.rk43_setup()
        lib.ensemble_step(self.eng, self.steps)
        for m, eng in enumerate(self.eng):
            _write_state(out, "m%d_" % m, eng.state())
        return {}


class _Stage:
    """The functions of an RK stage called one by one, twice in turn, on the
    caller's host arrays; U is solved in place, warm from the last stage."""

    def __init__(self, case, seed):
        from qdeqcycle_fdm_amd import lib
        self.pb, self.slips, self.shift, self.psi, self.V = _stage_inputs(case, seed)
        self.eng = lib.Engine(self.pb, **_SOLVERS[case["solver"]])
        p = self.pb.params
        self.arrays = [("U", "f8", (p.nz, p.nx))] + \
            [(k, "f8", (p.nz,)) for k in ("Ts", "Tn", "V", "dpsi")]

    def start(self, out):
        np.copyto(out["U"], self.pb.U0)

    def run(self, out):
        pb, eng, U = self.pb, self.eng, out["U"]
        vcycles = 0
        for slip in self.slips:
            eng.setBoundary(U, slip, self.shift, 1.0e7, 0.5, 1.0e6)
            vcycles += eng.ode_solve(U)[0]
            Ts, Tn = eng.eval_stress_on_fault(U, pb.mu, pb.tau_n0)
            V = eng.NRsearch(Ts, Tn, self.psi, pb.a, pb.eta, self.V)
            dpsi = eng.cal_dpsi(self.psi, V, pb.b)
        for k, v in (("Ts", Ts), ("Tn", Tn), ("V", V), ("dpsi", dpsi)):
            np.copyto(out[k], v)
        return {}


class _Train:
    """Further epochs of training on the pairs a run has left."""

    def __init__(self, case, seed):
        from qdeqcycle_fdm_amd import lib
        nk = case["nk"]
        levels = 1
        while (nk - 1) % 2 ** levels == 0 and (nk - 1) >> levels >= 8:
            levels += 1
        pb = _problem(dict(problem="basin", ni=nk, nk=nk, levels=levels), seed)
        self.guess = lib.Guess(nk, capacity=case["pairs"], seed=seed)
        self.opts = dict(epochs=case["epochs"], batch=case["batch"])
        with lib.Engine(pb, **_SOLVERS["fast64"]) as eng:
            eng.rk43_setup()
            eng.attach_guess(self.guess, lib.GUESS_HARVEST)
            while self.guess.pairs < case["pairs"]:
                eng.rk43_step(10)
            eng.attach_guess(None, lib.GUESS_OFF)
        self.arrays = [("params", "f4", (self.guess.num_params,))]

    def run(self, out):
        loss = self.guess.train(**self.opts)
        np.copyto(out["params"], self.guess.get_params())
        return {"loss": loss}


_KINDS = {"cycle": _Cycle, "ensemble": _Ensemble, "stage": _Stage, "train": _Train}


def _serve(fd):
    sys.path.insert(0, ROOT)
    sock = socket.socket(fileno=fd)
    held, last = {}, 0
    while True:
        msg, _ = _receive(sock)
        if msg is None:
            return
        try:
            if msg["do"] == "new":
                obj = _KINDS[msg["case"]["kind"]](msg["case"], msg["seed"])
                layout, size = _layout(obj.arrays)
                block = os.memfd_create("cases")
                os.ftruncate(block, size)
                out = _views(mmap.mmap(block, size), layout)
                for a in out.values():
                    a[...] = 0
                if hasattr(obj, "start"):
                    obj.start(out)
                last += 1
                held[last] = (obj, out)
                _send(sock, {"id": last, "size": size, "arrays": layout}, [block])
                os.close(block)
            elif msg["do"] == "run":
                obj, out = held[msg["id"]]
                _send(sock, {"values": obj.run(out)})
            else:
                held.pop(msg["id"], None)
                obj = out = None
                gc.collect()
                _send(sock, {})
        except Exception as e:
            _send(sock, {"error": "%s: %s" % (type(e).__name__, e)})


# ---------------------------------------------------------------------------
# What the outputs are in exact arithmetic
# ---------------------------------------------------------------------------

def exact(case, seed):
    """The stage functions on the uniform medium, where the five-point system
    separates: cosines in depth (mirrored rows at both ends), hyperbolic sines
    in x.  A cycle's steps follow the controller's history and a training run
    its own roundings; neither has a value of its own."""
    if case["kind"] != "stage":
        return None
    pb, slips, shift, psi, V0 = _stage_inputs(case, seed)
    p = pb.params
    N, K, h = p.nk, p.ni, p.dh
    left = slips[-1][1:N + 1] / 2.0
    right = p.Vini * (1.0e7 + 0.5 * 1.0e6) / 2.0 + shift[1:N + 1]
    j = np.arange(N)
    w = np.ones(N)
    w[0] = w[-1] = 0.5
    C = np.cos(math.pi * np.outer(j, j) / (N - 1))            # C[row, mode]
    norm = (w[:, None] * C * C).sum(axis=0)
    modes = [(C * w[:, None]).T @ c / norm for c in (left, right)]
    # u_{k-1} + u_{k+1} = 2 cosh(theta) u_k for each cosine mode
    th = np.arccosh(2.0 - np.cos(math.pi * j / (N - 1)))
    k = np.arange(K)
    with np.errstate(divide="ignore", invalid="ignore"):
        def ratio(s):  # sinh(theta s) / sinh(theta (K - 1))
            r = np.exp(np.outer(th, s - (K - 1))) * np.expm1(-2.0 * np.outer(th, s)) \
                / np.expm1(-2.0 * th * (K - 1))[:, None]
            r[0] = s / (K - 1.0)
            return r
        coef = modes[0][:, None] * ratio(K - 1.0 - k) + modes[1][:, None] * ratio(k + 0.0)
    u = C @ coef
    U = np.zeros((p.nz, p.nx))
    U[1:N + 1, 1:K + 1] = u
    U[:, 0] = 2.0 * U[:, 1] - U[:, 2]
    U[:, -1] = 2.0 * U[:, -2] - U[:, -3]
    U[0], U[-1] = U[2], U[-3]
    Ts, Tn, V, dpsi = (np.zeros(p.nz) for _ in range(4))
    du = (-24.0 / 17.0 * u[:, 0] + 59.0 / 34.0 * u[:, 1] - 4.0 / 17.0 * u[:, 2]
          - 3.0 / 34.0 * u[:, 3]) / h
    i = slice(1, N + 1)
    Ts[i], Tn[i] = pb.mu[i, 1] * du * 1e3, pb.tau_n0[i]
    # |Ts| = -Tn a asinh(V / (2 V0) exp(psi / a)) + eta V, by bisection on
    # the friction angle y = asinh(...)
    a, eta, ps = pb.a[i], pb.eta[i], psi[i]
    t = np.abs(Ts[i])
    lo, hi = np.zeros(N), t / (-Tn[i] * a)  # t = fa y + eta rate(y) has y >= 0 here

    def rate(y):
        return p.V0 * (np.exp(y - ps / a) - np.exp(-y - ps / a))

    for _ in range(200):
        y = 0.5 * (lo + hi)
        over = -Tn[i] * a * y + eta * rate(y) > t
        hi, lo = np.where(over, y, hi), np.where(over, lo, y)
    V[i] = np.sign(Ts[i]) * rate(0.5 * (lo + hi))
    dpsi[i] = pb.b[i] * p.V0 / p.L * (np.exp((p.f0 - ps) / pb.b[i]) - V[i] / p.V0)
    return {"U": U, "Ts": Ts, "Tn": Tn, "V": V, "dpsi": dpsi}


if __name__ == "__main__":
    _serve(int(sys.argv[1]))
