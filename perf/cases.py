"""Performance cases: what users of the framework run, each through the
Python binding of the C-ABI (atus2_amd.hip), with the library's default
kernel choices, as the drivers take them.

Every case names its workload in "kind" and carries its sizes:

  line     rt_solver in 1D: freeprop blocks, norm and energy after every block
  plane    rt_solver in 2D (double slit): freeprop blocks, norm after every block
  bragg    the two-component Bragg pulse in 3D, Rabi populations after every block
  scan     a parameter scan over runs of several grids: one graph launch a block
  batch    independent Bragg runs of one grid: eager blocks, Rabi populations
  ground   sobmin / sobmin_2: the Sobolev minimiser from its start state
  states   three-state steps: double_bragg, the numerical Bragg step, raman
  species  two species: bragg_ds and its free propagation
  observe  what ana_expval and the drivers read from a state
  train    the warm-start network: Adam steps on its training set

A pass starts from the state that prepare() left (a device snapshot, as
the chirp scan restores it) and ends with the final state on the host (the
drivers' .bin output) and the observables of every block.
"""
import math

import numpy as np
import torch

from atus2_amd import hip
from atus2_amd.scan import RABI_THRESHOLD, ScanRun
from atus2_amd.workloads import axis_coords, grid_spacings


def listed():
    return [
        # the 1D configuration: 4096 points, harmonic trap, 1000 steps
        {"name": "line_4096", "kind": "line", "n": 4096, "nk": 100, "blocks": 10},
        # the 2D configuration: double slit on 2048^2
        {"name": "plane_2048", "kind": "plane", "n0": 2048, "n1": 2048, "nk": 100, "blocks": 3},
        # the headline configuration: Bragg pulse on 256^3
        {"name": "bragg_256", "kind": "bragg", "n0": 256, "n1": 256, "n2": 256, "nk": 100, "blocks": 3, "dk": False},
        # a small 3D run, where launches and latency count
        {"name": "bragg_32x64x32", "kind": "bragg", "n0": 32, "n1": 64, "n2": 32, "nk": 100, "blocks": 2, "dk": True},
        # the parameter scan, an eighth of its 512 runs, all its grid shapes
        {"name": "scan_64", "kind": "scan", "n1d": 48, "n2d": 16, "nk": 100, "blocks": 3},
        # one 1D shape group of that scan run eagerly
        {"name": "batch_77x2048", "kind": "batch", "n0": 2048, "n1": 1, "runs": 77, "nk": 100, "blocks": 10},
        # the ground-state configuration: 128^3, anisotropic trap
        {"name": "ground_128", "kind": "ground", "n0": 128, "n1": 128, "n2": 128, "nw": 1, "its": 200},
        # the training set's ground states: 4096 of them on 32^3
        {"name": "ground_32", "kind": "ground", "n0": 32, "n1": 32, "n2": 32, "nw": 1, "its": 500},
        # double Bragg diffraction of three momentum states in 2D
        {"name": "states_512", "kind": "states", "step": "double", "nc": 3, "n0": 512, "n1": 512, "n2": 1, "nk": 100,
         "blocks": 2},
        # two-species interferometer in 3D
        {"name": "species_64", "kind": "species", "step": "bragg_ds", "nc": 4, "n0": 64, "n1": 64, "n2": 64, "nk": 100,
         "blocks": 2},
        # analysis of one saved 3D state
        {"name": "observe_256", "kind": "observe", "nc": 1, "n0": 256, "n1": 256, "n2": 256},
        # training of the warm-start network
        {"name": "train_256", "kind": "train", "batch": 256, "n_out": 32768, "steps": 40},
    ]


def _p2(rng, lo, hi):
    """A power of two in [lo, hi] (the lengths an axis can have)."""
    return 2 ** rng.randint(lo.bit_length() - 1, hi.bit_length() - 1)


def _axes(rng, dim, lo, hi, most):
    while True:
        n = [_p2(rng, lo, hi) if a < dim else 1 for a in range(3)]
        if math.prod(n) <= most:
            return {"n0": n[0], "n1": n[1], "n2": n[2]}


def draw(rng):
    kind = rng.choice(["line", "plane", "bragg", "scan", "batch", "ground", "states", "species", "observe", "train"])
    nk = rng.randint(20, 100)
    if kind == "line":
        return {"kind": kind, "n": _p2(rng, 256, 65536), "nk": nk, "blocks": rng.randint(2, 10)}
    if kind == "plane":
        return {"kind": kind, "n0": _p2(rng, 128, 2048), "n1": _p2(rng, 128, 2048), "nk": nk,
                "blocks": rng.randint(1, 3)}
    if kind == "bragg":
        return {"kind": kind, **_axes(rng, 3, 16, 256, 1 << 23), "nk": nk, "blocks": rng.randint(1, 3),
                "dk": rng.random() < 0.5}
    if kind == "scan":
        return {"kind": kind, "n1d": rng.randint(4, 48), "n2d": rng.randint(0, 12), "nk": nk,
                "blocks": rng.randint(1, 3)}
    if kind == "batch":
        two = rng.random() < 0.4
        return {"kind": kind, "n0": _p2(rng, 64, 512) if two else _p2(rng, 256, 16384),
                "n1": _p2(rng, 64, 512) if two else 1, "runs": rng.randint(1, 16 if two else 100), "nk": nk,
                "blocks": rng.randint(1, 6)}
    if kind == "ground":
        dim = rng.choice([1, 2, 3, 3])
        lo, hi = ((256, 4096), (64, 1024), (16, 128))[dim - 1]
        return {"kind": kind, **_axes(rng, dim, lo, hi, 1 << 21), "nw": rng.choice([1, 2]),
                "its": rng.randint(20, 200)}
    if kind == "states":
        step, nc = rng.choice([("double", 3), ("bragg", 2), ("bragg", 3), ("raman", 3), ("raman", 4)])
        dim = rng.choice([1, 2, 2, 3])
        lo, hi = ((256, 4096), (64, 512), (16, 64))[dim - 1]
        return {"kind": kind, "step": step, "nc": nc, **_axes(rng, dim, lo, hi, 1 << 18), "nk": nk,
                "blocks": rng.randint(1, 3)}
    if kind == "species":
        step, nc = rng.choice([("bragg_ds", 4), ("freeprop", 2), ("freeprop", 4)])
        dim = rng.choice([1, 2, 3])
        lo, hi = ((256, 4096), (64, 1024), (16, 128))[dim - 1]
        return {"kind": kind, "step": step, "nc": nc, **_axes(rng, dim, lo, hi, 1 << 20), "nk": nk,
                "blocks": rng.randint(1, 2)}
    if kind == "observe":
        dim = rng.choice([1, 2, 3])
        lo, hi = ((1024, 65536), (128, 4096), (32, 256))[dim - 1]
        return {"kind": kind, "nc": rng.choice([1, 2]), **_axes(rng, dim, lo, hi, 1 << 23)}
    return {"kind": kind, "batch": rng.randint(32, 256), "n_out": rng.choice([4096, 32768]),
            "steps": rng.randint(10, 40)}


# ------------------------------------------------------------ inputs

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _shape(case):
    if case["kind"] == "line":
        return (case["n"],)
    n = [case["n0"], case["n1"], case.get("n2", 1)]
    while n[-1] == 1:
        n.pop()
    return tuple(n)


def _coords(shape, L):
    """Per-axis coordinates, broadcastable over the grid."""
    out = []
    for a, n in enumerate(shape):
        x = torch.from_numpy(axis_coords(n, L[a])).to(_dev())
        out.append(x.reshape([n if b == a else 1 for b in range(len(shape))]))
    return out


def _packets(shape, L, widths, weights, seed, noise=1e-3, shift=0.0, kick=None):
    """One Gaussian packet per weight plus complex noise, normalised to the
    weight: a list of complex128 tensors."""
    g = torch.Generator(device=_dev()).manual_seed(int(seed))
    xs = _coords(shape, L)
    dx, _ = grid_spacings(shape, L)
    env = torch.ones(shape, dtype=torch.float64, device=_dev())
    ph = torch.zeros(shape, dtype=torch.float64, device=_dev())
    for a, x in enumerate(xs):
        env = env * torch.exp(-((x - shift * (a + 1)) / widths[a]) ** 2 / 2)
        if kick:
            ph = ph + kick[a] * x
    out = []
    for w in weights:
        r = torch.empty((2,) + tuple(shape), dtype=torch.float64, device=_dev()).normal_(generator=g)
        p = torch.complex(env + noise * r[0], noise * r[1])
        if kick:
            p = p * torch.exp(1j * ph)
        out.append(p * math.sqrt(w / (math.prod(dx) * float((p.real ** 2 + p.imag ** 2).sum()))))
    return out


def _inputs(case, seed):
    """Everything a pass depends on, as plain values and tensors: shared by
    prepare() and exact()."""
    rng = np.random.default_rng(int(seed))
    k = case["kind"]
    if k == "line":
        L = [80.0]
        p = _packets((case["n"],), L, [1.0], [1.0], seed)
        x = _coords((case["n"],), L)[0]
        return {"shape": (case["n"],), "L": L, "psi": p, "V": 0.5 * x ** 2, "gs": [float(rng.uniform(5, 15))], "dt": 1e-3}
    if k == "plane":
        shape, L = _shape(case), [128.0, 128.0]
        x, y = _coords(shape, L)

        def rect(v, lo, hi):
            return ((v >= lo) & (v < hi)).double()
        V = 1e3 * rect(x, -0.5, 0.5) * (1.0 - rect(y, -5.0, -3.0) - rect(y, 3.0, 5.0))
        p = _packets(shape, L, [4.0, 4.0], [1.0], seed, noise=1e-4, kick=[float(rng.uniform(2, 4)), 0.0])
        return {"shape": shape, "L": L, "psi": p, "V": V, "gs": [1.0], "dt": 5e-4}
    if k == "bragg":
        shape, L = _shape(case), [64.0] * 3
        p = _packets(shape, L, [6.0, 4.0, 4.0], [1.0, 0.02], seed, noise=1e-4)
        g = float(rng.uniform(50, 150))
        las = dict(amp0=float(rng.uniform(3, 7)), laser_k=4.0, laser_domh=float(rng.uniform(6, 10)),
                   laser_dk=0.05 if case["dk"] else 0.0, deltaL=(0.0, 0.0))
        return {"shape": shape, "L": L, "psi": p, "gs": [g, 0.95 * g, 0.95 * g, g], "las": las, "dt": 2e-4,
                "t0": 0.3, "sigma": 0.5}
    if k in ("scan", "batch"):
        if k == "batch":
            shapes = [_shape(case)] * case["runs"]
        else:
            shapes = [(1024 << (i % 5),) for i in range(case["n1d"])]
            shapes += [(256 << (i % 3),) * 2 for i in range(case["n2d"])]
        return {"runs": [ScanRun(shape=s, amp0=float(rng.uniform(1, 10)), sigma=float(rng.uniform(0.2, 1)),
                                 laser_domh=float(8 + rng.uniform(-2, 2)), g=float(rng.uniform(1, 200)))
                         for s in shapes], "dt": 2e-4, "seed": int(seed)}
    if k == "ground":
        shape = _shape(case)
        d, nw = len(shape), case["nw"]
        L = [32.0 if n >= 64 else 16.0 for n in shape]
        w = rng.uniform(0.5, 2.0, 3)[:d]
        g = float(np.exp(rng.uniform(math.log(10.0), math.log(2000.0))))
        xs = _coords(shape, L)
        V = 0.5 * sum((float(w[a]) * xs[a]) ** 2 for a in range(d)) + torch.zeros(shape, dtype=torch.float64, device=_dev())
        gs = [g] if nw == 1 else [g, 0.9 * g, 0.9 * g, 1.1 * g]
        p = [q.real + 0j for q in _packets(shape, L, [1.5] * d, [1.0] * nw, seed, noise=1e-5)]
        if nw == 2:
            p[1] = torch.roll(p[1], 1, 0)
        peak = max(float((q.real ** 2).max()) for q in p)
        return {"shape": shape, "L": L, "psi": p, "V": V, "gs": gs, "step": 1.0 / (float(V.max()) + 3 * sum(gs[:nw]) * peak + 1)}
    if k in ("states", "species"):
        shape, nc = _shape(case), case["nc"]
        d = len(shape)
        L = [40.0, 32.0, 36.0][:d]
        p = _packets(shape, L, [2.0, 3.0, 4.0], [1.0, 0.5, 0.3, 0.2][:nc], seed)
        gs = [float(v) for v in rng.uniform(5.0, 30.0, nc * nc)]
        if k == "states":
            las = dict(amp0=float(rng.uniform(4, 6)), amp1=float(rng.uniform(2, 4)), laser_k=1.1, laser_domh=0.6,
                       phase0=0.3, beta=[0.03, -0.02, 0.01][:d] + [0.0] * (3 - d))
            if case["step"] != "raman":
                las["chirp_rate0"] = 0.2
            las["deltaL"] = (0.0, -0.7, 0.0, 0.0) if case["step"] == "double" else (0.1, -0.7, 0.4, 0.3)
            return {"shape": shape, "L": L, "psi": p, "gs": gs, "las": las, "dt": 1e-3}
        l1 = dict(beta0=0.01, deltaL=(0.0, 0.4, 0.1, -0.3), amp0=float(rng.uniform(4, 6)),
                  laser_k=6 * math.pi / L[0], laser_domh=8.0, laser_dk=0.05, chirp_rate0=0.2, phase0=0.3)
        l2 = dict(beta0=-0.02, amp0=float(rng.uniform(3, 4)), laser_k=4 * math.pi / L[0], laser_domh=6.0, laser_dk=0.03,
                  chirp_rate0=-0.1, phase0=0.7)
        return {"shape": shape, "L": L, "psi": p, "gs": gs, "las": l1, "las2": l2, "dt": 1e-3,
                "durations": (1e3, 1.5 * case["nk"] * 1e-3)}
    if k == "observe":
        shape, nc = _shape(case), case["nc"]
        d = len(shape)
        L = [64.0] * d
        p = _packets(shape, L, [6.0, 4.0, 4.0], [1.0, 0.5][:nc], seed, shift=0.7, kick=[float(v) for v in rng.uniform(0.3, 0.9, 3)])
        gs = [100.0] if nc == 1 else [100.0, 95.0, 95.0, 100.0]
        xs = _coords(shape, L)
        V = 0.05 * sum(x ** 2 for x in xs) + torch.zeros(shape, dtype=torch.float64, device=_dev())
        return {"shape": shape, "L": L, "psi": p, "V": V, "gs": gs,
                "k0": [[0.0] * d, [5.0] + [0.0] * (d - 1), [-5.0] + [0.0] * (d - 1)]}
    # train: features of (w, g), targets the Gaussian ground states of the
    # traps on a box of +-4.5 lengths, on an n^3 grid
    dims = (4, 256, 256, 64, case["n_out"])
    x = rng.uniform(-1, 1, (case["batch"], 4)).astype(np.float32)
    n = round(case["n_out"] ** (1 / 3))
    s = (np.arange(n) - n // 2) / (n / 2) * 4.5
    e = [np.exp(-s[None, :] ** 2 / 2 * (1.2 + 0.5 * x[:, a:a + 1] + 0.2 * x[:, 3:4])) for a in range(3)]
    t = np.einsum("bi,bj,bk->bijk", *e).reshape(case["batch"], -1).astype(np.float32)
    par = []
    for i, o in zip(dims[:-1], dims[1:]):
        a = math.sqrt(6.0 / (i + o))
        par += [rng.uniform(-a, a, i * o), np.zeros(o)]
    return {"dims": dims, "x": x, "t": t, "par": np.concatenate(par).astype(np.float32), "lr": 2e-3}


# ------------------------------------------------------------ prepare

def _context(q, nc):
    dx, dk = grid_spacings(q["shape"], q["L"])
    ctx = hip.Context(q["shape"], dx, dk, nc)
    for c in range(nc):
        ctx.upload(c, q["psi"][c].cpu().numpy())
    ctx.set_g(q["gs"])
    ctx.set_alpha([0.5] * len(q["shape"]))
    if "V" in q:
        for c in range(nc):
            ctx.set_potential(c, q["V"].cpu().numpy())
    return ctx


def _batches(runs):
    """One batch context per grid shape, loaded with its runs."""
    groups = {}
    for i, r in enumerate(runs):
        groups.setdefault(r.shape, []).append(i)
    out = []
    for shape, idx in sorted(groups.items()):
        rs = [runs[i] for i in idx]
        dx, dk = grid_spacings(shape, rs[0].L)
        B = hip.BatchContext(shape, dx, dk, len(rs))
        p1, p2 = rs[0].initial_state()
        for j in range(len(rs)):
            B.upload(2 * j, p1)
            B.upload(2 * j + 1, p2)
        B.set_alpha([0.5] * len(shape))
        B.set_runs([r.gs for r in rs], [r.laser() for r in rs])
        B.snapshot_save(0)
        out.append((B, rs))
    return out


def prepare(case, seed):
    q = _inputs(case, seed)
    s = {"case": case, "q": q}
    k = case["kind"]
    if k in ("scan", "batch"):
        s["groups"] = _batches(q["runs"])
        s["k0"] = q["runs"][0].rabi_k0()
        if k == "scan":
            s["graph"] = hip.ScanGraph([B for B, _ in s["groups"]], hip.STEP_BRAGG_AD, q["dt"], case["nk"], s["k0"],
                                       RABI_THRESHOLD)
        return s
    if k == "train":
        s["net"] = hip.Net(q["dims"], max_batch=case["batch"], seed=1)
        s["net"].set_data(q["x"], q["t"])
        return s
    nc = len(q["psi"])
    s["ctx"] = ctx = _context(q, nc)
    if k == "ground":
        ctx.sob_setup([0.5] * nc, q["step"])
    if k == "species":
        ctx.set_alpha2([0.35] * len(q["shape"]))
    if k in ("bragg", "states", "species"):
        s["las"] = hip.laser(**q["las"])
    if k == "species":
        s["las2"] = hip.laser(**q["las2"])
    if k == "bragg":
        s["amp"] = lambda t: math.exp(-0.5 * ((t - q["t0"]) / q["sigma"]) ** 2)
        s["k0"] = _bragg_k0(q)
    if k == "states":
        s["amp"] = lambda t: math.exp(-0.5 * ((t - 0.1) / 0.2) ** 2)
    if k != "observe":
        ctx.snapshot_save(0)
    del q["psi"]
    return s


def _bragg_k0(q):
    k = 2 * q["las"]["laser_k"]
    return [(0.0, 0.0, 0.0), (k, 0.0, 0.0), (-k, 0.0, 0.0)]


def _amplitudes(B, rs, t, dt, nk):
    t1 = np.array(B.step_times(t, dt, nk))[:, None]
    sig = np.array([r.sigma for r in rs])[None, :]
    t0 = np.array([r.t0 for r in rs])[None, :]
    return np.exp(-0.5 * ((t1 - t0) / sig) ** 2)


def _state(ctx):
    return [ctx.download(c) for c in range(ctx.ncomp)]


# ------------------------------------------------------------ run

def run(s):
    case, q = s["case"], s["q"]
    k, nk = case["kind"], case.get("nk")
    if k == "line":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        t, norm, energy = 0.0, [], []
        for _ in range(case["blocks"]):
            t = ctx.run_block(hip.STEP_FREEPROP, q["dt"], nk, t)
            norm.append(ctx.particle_number(0))
            energy.append(ctx.energy())
        return {"psi": _state(ctx), "norm": np.array(norm), "energy": np.array(energy)}
    if k == "plane":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        t, norm = 0.0, []
        for _ in range(case["blocks"]):
            t = ctx.run_block(hip.STEP_FREEPROP, q["dt"], nk, t)
            norm.append(ctx.particle_number(0))
        return {"psi": _state(ctx), "norm": np.array(norm)}
    if k == "bragg":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        t, rabi = 0.0, []
        for _ in range(case["blocks"]):
            t = ctx.run_block(hip.STEP_BRAGG_AD, q["dt"], nk, t, s["las"], s["amp"])
            rabi.append(ctx.rabi_integrals(0, s["k0"], RABI_THRESHOLD))
        return {"psi": _state(ctx), "rabi": np.array(rabi)}
    if k == "scan":
        for B, _ in s["groups"]:
            B.snapshot_restore(0)
        t, rabi = 0.0, [[] for _ in s["groups"]]
        for _ in range(case["blocks"]):
            F = [_amplitudes(B, rs, t, q["dt"], nk) for B, rs in s["groups"]]
            t, got, _ = s["graph"].launch(t, F)
            for g, r in zip(rabi, got):
                g.append(r)
        return {"rabi": [np.array(g) for g in rabi]}
    if k == "batch":
        B, rs = s["groups"][0]
        B.snapshot_restore(0)
        t, rabi = 0.0, []
        for _ in range(case["blocks"]):
            t = B.run_batch_block(hip.STEP_BRAGG_AD, q["dt"], nk, t, _amplitudes(B, rs, t, q["dt"], nk))
            rabi.append(B.batch_rabi_integrals(0, s["k0"], RABI_THRESHOLD))
        return {"psi": np.stack(_state(B)), "rabi": np.array(rabi), "norm": B.particle_numbers()}
    if k == "ground":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        ctx.sob_renormalize()
        its, res = ctx.sob_run(1e-10, case["its"])
        return {"psi": _state(ctx), "its": its, "res": res, "mu": ctx.sob_mu()}
    if k == "states":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        step = {"double": hip.STEP_DOUBLE_BRAGG, "bragg": hip.STEP_NUM_BRAGG, "raman": hip.STEP_RAMAN}[case["step"]]
        t = 0.0
        for _ in range(case["blocks"]):
            t = ctx.run_block(step, q["dt"], nk, t, s["las"], s["amp"])
        return {"psi": _state(ctx), "norm": np.array([ctx.particle_number(c) for c in range(ctx.ncomp)])}
    if k == "species":
        ctx = s["ctx"]
        ctx.snapshot_restore(0)
        step = hip.STEP_BRAGG_AD if case["step"] == "bragg_ds" else hip.STEP_FREEPROP_IF
        t = 0.0
        for _ in range(case["blocks"]):
            t = ctx.run_block_ds(step, q["dt"], nk, t, s["las"], s["las2"], 0.0, q["durations"])
        return {"psi": _state(ctx), "norm": np.array([ctx.particle_number(c) for c in range(ctx.ncomp)])}
    if k == "observe":
        ctx = s["ctx"]
        out = {"energy": ctx.energy()}
        for c in range(ctx.ncomp):
            m = ctx.moments(c)
            out["c%d" % c] = {"N": ctx.particle_number(c), "x": ctx.expval_x(c), "k": ctx.expval_k(c),
                              "rabi": ctx.rabi_integrals(c, q["k0"], RABI_THRESHOLD),
                              "moments": np.array([m["N"]] + m["x"] + m["x2"] + m["k"] + m["k2"] + [m["phase"]])}
        return out
    net = s["net"]
    net.set_params(q["par"])
    losses = net.train(case["steps"], case["batch"], q["lr"], q["lr"] * 0.02, seed=5)
    return {"losses": losses, "params": net.get_params()}


# ------------------------------------------------------------ work

def work(case):
    """Bytes: the state read and written once per step (a step couples every
    point with every other, so none but a run that fits one compute unit can
    skip that), a 1D run of up to 4096 points once per block; the potential
    and the observables' reads beside it.  Flops: 5 N log2 N per transform,
    two per step and component, and the pointwise step."""
    k = case["kind"]
    if k == "train":
        d = (4, 256, 256, 64, case["n_out"])
        w = sum(a * b for a, b in zip(d[:-1], d[1:]))
        act = case["batch"] * sum(d)
        return {"bytes": case["steps"] * (4.0 * (7 * w + act + case["batch"] * case["n_out"])),
                "flops": case["steps"] * 6.0 * case["batch"] * w}

    def evolve(shape, nc, steps, blocks, point, pot=0):
        n = math.prod(shape)
        resident = len(shape) == 1 and n <= 4096
        return (n * nc * (32.0 + pot) * (blocks if resident else steps),
                steps * n * nc * (10.0 * math.log2(n) + point))
    if k in ("scan", "batch"):
        steps = case["nk"] * case["blocks"]
        shapes = [_shape(case)] * case["runs"] if k == "batch" else \
            [(1024 << (i % 5),) for i in range(case["n1d"])] + [(256 << (i % 3),) * 2 for i in range(case["n2d"])]
        parts = [evolve(sh, 2, steps, case["blocks"], 60) for sh in shapes]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    shape = _shape(case)
    n, d = math.prod(shape), len(shape)
    if k == "observe":
        # the state and the potential read once for the sums in x space, the
        # state once per axis for those in k space
        nc = case["nc"]
        return {"bytes": n * nc * (16.0 * (1 + d) + 8), "flops": n * nc * (5 * math.log2(n) + 60.0)}
    if k == "ground":
        # an iteration reads and writes the state, reads the potential; two
        # forward transforms (state, nonlinear term), one back
        return {"bytes": case["its"] * n * case["nw"] * 40.0, "flops": case["its"] * n * case["nw"] * (15 * math.log2(n) + 40)}
    nc = {"line": 1, "plane": 1, "bragg": 2}.get(k) or case["nc"]
    b, f = evolve(shape, nc, case["nk"] * case["blocks"], case["blocks"], 60, 8 if k in ("line", "plane") else 0)
    return {"bytes": b + 16.0 * n * nc, "flops": f}


# ------------------------------------------------------------ exact

def _kvec(n, L):
    return 2 * math.pi / L * ((torch.arange(n, device=_dev(), dtype=torch.float64) + n // 2) % n - n // 2)


def _k2(shape, L, alpha):
    out = 0.0
    for a, n in enumerate(shape):
        out = out + alpha * _kvec(n, L[a]).reshape([n if b == a else 1 for b in range(len(shape))]) ** 2
    return out


def _expm(H, dt, psi):
    """exp(-i dt H) psi by its series, H a dict of the nonzero elements."""
    big = dt * sum(float(h.abs().max()) if torch.is_tensor(h) else abs(h) for h in H.values())
    out, term = list(psi), list(psi)
    n, size = 0, 1.0
    while size > 1e-18 and n < 60:
        n += 1
        size *= big / n
        new = [0.0] * len(psi)
        for (i, j), h in H.items():
            new[i] = new[i] + h * term[j]
        term = [(-1j * dt / n) * v for v in new]
        out = [o + v for o, v in zip(out, term)]
    return out


def _diag(psi, gs, extra):
    nc = len(psi)
    den = [p.real ** 2 + p.imag ** 2 for p in psi]
    return [sum(gs[j + nc * i] * den[j] for j in range(nc)) + extra[i] for i in range(nc)]


class _Split:
    """Strang blocks of a list of components over their last d axes."""

    def __init__(self, psi, L, dt, alphas):
        self.psi, self.dt = list(psi), dt
        d = len(L)
        self.axes = tuple(range(-d, 0))
        shape = tuple(psi[0].shape[-d:])
        self.half = [torch.exp(-0.5j * dt * _k2(shape, L, a)) for a in alphas]

    def kinetic(self, full):
        for c, e in enumerate(self.half):
            f = torch.fft.fftn(self.psi[c], dim=self.axes)
            self.psi[c] = torch.fft.ifftn(f * (e * e if full else e), dim=self.axes)

    def block(self, nk, t, vstep):
        """vstep(psi, t, t1): one potential step; t: the time before it."""
        self.kinetic(False)
        t += 0.5 * self.dt
        for m in range(1, nk + 1):
            self.psi = vstep(self.psi, t, t + 0.5 * self.dt)
            self.kinetic(m < nk)
            t += self.dt if m < nk else 0.5 * self.dt
        return t


def _norm(psi, dx):
    return math.prod(dx) * float((psi.real ** 2 + psi.imag ** 2).sum())


def _spectrum(psi, dx):
    """|psi^|^2 with the transform's factor dx / sqrt(2 pi) per axis."""
    f = torch.fft.fftn(psi)
    return (f.real ** 2 + f.imag ** 2) * (math.prod(dx) / (2 * math.pi) ** (0.5 * len(dx))) ** 2


def _rabi(psi, L, k0, axes_from=0):
    """Populations of the balls around k0; leading axes are runs."""
    shape = tuple(psi.shape[axes_from:])
    d = len(shape)
    dx, dk = grid_spacings(shape, L)
    f = torch.fft.fftn(psi, dim=tuple(range(-d, 0)))
    den = (f.real ** 2 + f.imag ** 2) * (math.prod(dx) / (2 * math.pi) ** (0.5 * d)) ** 2
    out = []
    for k in k0:
        r = 0.0
        for a, n in enumerate(shape):
            r = r + (_kvec(n, L[a]).reshape([n if b == a else 1 for b in range(d)]) - k[a]) ** 2
        out.append((den * (torch.sqrt(r) < RABI_THRESHOLD)).sum(dim=tuple(range(-d, 0))) * math.prod(dk))
    return torch.stack(out, dim=-1).cpu().numpy()


def _energy(psi, q):
    dx, dk = grid_spacings(q["shape"], q["L"])
    nc = len(psi)
    k2 = _k2(q["shape"], q["L"], 0.5)
    e = sum(float((k2 * _spectrum(p, dx)).sum()) for p in psi) * math.prod(dk)
    den = [p.real ** 2 + p.imag ** 2 for p in psi]
    for i in range(nc):
        e += math.prod(dx) * float(((q["V"] + 0.5 * sum(q["gs"][j + nc * i] * den[j] for j in range(nc))) * den[i]).sum())
    return e


def _bragg_v(gs, amp0, lk, domh, dk, F, x, dt):
    """The Bragg potential step; every parameter a number or a tensor over
    the leading run axis, F a function of t1."""
    def v(psi, t, t1):
        Om = F(t1) * amp0 * torch.cos(lk * x - domh * t1)
        D = _diag(psi, gs, [0.0, 0.0])
        eta = torch.exp(-0.5j * dk * x)
        return _expm({(0, 0): D[0], (1, 1): D[1], (0, 1): Om * eta, (1, 0): Om * eta.conj()}, dt, psi)
    return v


def _exact_runs(case, q):
    groups = {}
    for r in q["runs"]:
        groups.setdefault(r.shape, []).append(r)
    out = []
    for shape, rs in sorted(groups.items()):
        d = len(shape)

        def col(f):
            return torch.tensor([f(r) for r in rs], dtype=torch.float64, device=_dev()).reshape([-1] + [1] * d)
        L = [rs[0].L] * d
        x = _coords(shape, L)[0]
        p1 = torch.from_numpy(rs[0].initial_state()[0]).to(_dev())
        S = _Split([p1.repeat([len(rs)] + [1] * d), torch.zeros([len(rs)] + list(shape), dtype=p1.dtype, device=_dev())],
                   L, q["dt"], [0.5, 0.5])
        g, sig, t0 = col(lambda r: r.g), col(lambda r: r.sigma), col(lambda r: r.t0)
        v = _bragg_v([g, 0.95 * g, 0.95 * g, g], col(lambda r: r.amp0), rs[0].laser_k, col(lambda r: r.laser_domh), 0.0,
                     lambda t: torch.exp(-0.5 * ((t - t0) / sig) ** 2), x, q["dt"])
        t, rabi = 0.0, []
        for _ in range(case["blocks"]):
            t = S.block(case["nk"], t, v)
            rabi.append(_rabi(S.psi[0], L, rs[0].rabi_k0(), 1))
        out.append((S.psi, np.array(rabi), grid_spacings(shape, L)[0]))
    return out


def exact(case, seed):
    q = _inputs(case, seed)
    k, nk, dt = case["kind"], case.get("nk"), q.get("dt")
    if k in ("scan", "batch"):
        got = _exact_runs(case, q)
        if k == "scan":
            return {"rabi": [r for _, r, _ in got]}
        psi, rabi, dx = got[0]
        both = torch.stack(psi, dim=1)
        d = len(_shape(case))
        norm = math.prod(dx) * (both.real ** 2 + both.imag ** 2).sum(dim=tuple(range(-d, 0)))
        return {"psi": both.reshape((-1,) + tuple(both.shape[2:])).cpu().numpy(), "rabi": rabi, "norm": norm.cpu().numpy()}
    if k == "train":
        return _exact_train(case, q)
    shape, L, psi = q["shape"], q["L"], q["psi"]
    dx, dk = grid_spacings(shape, L)
    xs = _coords(shape, L)
    nc = len(psi)
    if k in ("line", "plane"):
        S = _Split(psi, L, dt, [0.5])
        t, norm, energy = 0.0, [], []

        def v(p, t, t1):
            return [p[0] * torch.exp(-1j * dt * _diag(p, q["gs"], [q["V"]])[0])]
        for _ in range(case["blocks"]):
            t = S.block(nk, t, v)
            norm.append(_norm(S.psi[0], dx))
            if k == "line":
                energy.append(_energy(S.psi, q))
        out = {"psi": [p.cpu().numpy() for p in S.psi], "norm": np.array(norm)}
        return dict(out, energy=np.array(energy)) if k == "line" else out
    if k == "bragg":
        las = q["las"]
        S = _Split(psi, L, dt, [0.5, 0.5])
        v = _bragg_v(q["gs"], las["amp0"], las["laser_k"], las["laser_domh"], las["laser_dk"],
                     lambda t: math.exp(-0.5 * ((t - q["t0"]) / q["sigma"]) ** 2), xs[0], dt)
        t, rabi = 0.0, []
        for _ in range(case["blocks"]):
            t = S.block(nk, t, v)
            rabi.append(_rabi(S.psi[0], L, _bragg_k0(q)))
        return {"psi": [p.cpu().numpy() for p in S.psi], "rabi": np.array(rabi)}
    if k == "states":
        las = q["las"]
        bx = sum(las["beta"][a] * xs[a] for a in range(len(shape)))
        x, lk, dl, ph, cr = xs[0], las["laser_k"], las["deltaL"], las["phase0"], las.get("chirp_rate0", 0.0)

        def v(p, t, t1):
            D = _diag(p, q["gs"], [bx - dl[i] for i in range(nc)])
            H = {(i, i): D[i] for i in range(nc)}
            if case["step"] == "double":
                # states 1 and 2 share the diagonal of state 1
                F = max(0.0, math.exp(-0.5 * ((t1 - 0.1) / 0.2) ** 2))
                H[0, 0] = D[0] + dl[0]
                H[2, 2] = D[1]
                for i, s in ((1, 1), (2, -1)):
                    dw = las["laser_domh"] + s * cr * t1
                    H[0, i] = H[i, 0] = F * las["amp0"] * torch.cos(s * lk * x - dw * t1 - ph / 2)
            elif case["step"] == "bragg":
                for i in range(nc - 1):
                    s = 1 if i == 0 else -1
                    a = (-las["laser_domh"] + s * cr * t) * t + s * lk * x - 0.5 * ph
                    e = 0.5 * (las["amp0"] * torch.exp(1j * a) + las["amp1"] * torch.exp(-1j * a))
                    H[i + 1, 0], H[0, i + 1] = e, e.conj()
            else:
                H[2, 2] = D[2] + las["laser_domh"]
                e = torch.exp(1j * lk * x)
                H[0, 2], H[2, 0] = las["amp0"] / 2 * e, las["amp0"] / 2 * e.conj()
                H[1, 2], H[2, 1] = las["amp1"] / 2 * e.conj(), las["amp1"] / 2 * e
            return _expm(H, dt, p)
        S, t = _Split(psi, L, dt, [0.5] * nc), 0.0
        for _ in range(case["blocks"]):
            t = S.block(nk, t, v)
        return {"psi": [p.cpu().numpy() for p in S.psi], "norm": np.array([_norm(p, dx) for p in S.psi])}
    if k == "species":
        x, lasers = xs[0], (q["las"], q["las2"])
        dl = q["las"]["deltaL"]

        def v(p, t, t1):
            D = _diag(p, q["gs"], [lasers[i >= nc // 2]["beta0"] * x - dl[i] for i in range(nc)])
            H = {(i, i): D[i] for i in range(nc)}
            if case["step"] == "bragg_ds":
                for s, las in enumerate(lasers):
                    on = 0.0 if t1 > q["durations"][s] else 1.0
                    Om = on * las["amp0"] * torch.cos(las["laser_k"] * x - (las["laser_domh"] + las["chirp_rate0"] * t1) * t1
                                                      + las["phase0"] / 2)
                    e = torch.exp(-0.5j * (las["laser_dk"] * x + las["phase0"]))
                    H[2 * s, 2 * s + 1], H[2 * s + 1, 2 * s] = Om * e, Om * e.conj()
            return _expm(H, dt, p)
        S, t = _Split(psi, L, dt, [0.5] * (nc // 2) + [0.35] * (nc // 2)), 0.0
        for _ in range(case["blocks"]):
            t = S.block(nk, t, v)
        return {"psi": [p.cpu().numpy() for p in S.psi], "norm": np.array([_norm(p, dx) for p in S.psi])}
    if k == "ground":
        return _exact_ground(case, q)
    out = {"energy": _energy(psi, q)}
    for c in range(nc):
        den = psi[c].real ** 2 + psi[c].imag ** 2
        sp = _spectrum(psi[c], dx)
        N = math.prod(dx) * float(den.sum())
        ks = [_kvec(n, L[a]).reshape([n if b == a else 1 for b in range(len(shape))]) for a, n in enumerate(shape)]
        X = [math.prod(dx) * float((x * den).sum()) for x in xs]
        K = [math.prod(dk) * float((kk * sp).sum()) for kk in ks]
        x2 = [math.prod(dx) * float(((x - m / N) ** 2 * den).sum()) / N for x, m in zip(xs, X)]
        k2 = [math.prod(dk) * float(((kk - m / N) ** 2 * sp).sum()) / N for kk, m in zip(ks, K)]
        ph = float((torch.atan2(psi[c].imag, psi[c].real) * den).sum() / den.sum())
        out["c%d" % c] = {"N": N, "x": np.array(X), "k": np.array(K), "rabi": _rabi(psi[c], L, q["k0"]),
                          "moments": np.array([N] + [v / N for v in X] + x2 + [v / N for v in K] + k2 + [ph])}
    return out


def _exact_ground(case, q):
    """CSOB_Base::run: the Sobolev gradient, its projection, the update."""
    shape, L, nw, step = q["shape"], q["L"], case["nw"], q["step"]
    dx, _ = grid_spacings(shape, L)
    ar, k2 = math.prod(dx), _k2(shape, L, 0.5)
    psi = [p / math.sqrt(_norm(p, dx)) for p in q["psi"]]

    def dot(a, b):
        return float((a.real * b.real + a.imag * b.imag).sum())

    its, res = 0, 0.0
    while its < case["its"]:
        N = [_norm(p, dx) for p in psi]
        f = [1.0 / math.sqrt(n) for n in N] if any(abs(n - 1) > 1e-5 for n in N) else [1.0] * nw
        W = _diag(psi, q["gs"], [q["V"]] * nw)
        new, res = [], 0.0
        for i, p in enumerate(psi):
            F = torch.fft.fftn(p)
            sob = torch.fft.ifftn(F / (1 + k2))
            grad = torch.fft.ifftn((k2 * F + torch.fft.fftn(W[i] * p)) / (1 + k2))
            d = grad - dot(p, grad) / dot(p, sob) * sob
            res += (ar * dot(d, d)) ** 2
            new.append(f[i] * p - step * d)
        psi, its, res = new, its + 1, math.sqrt(res)
        if res <= 1e-10:
            break
    W = _diag(psi, q["gs"], [q["V"]] * nw)
    mu = [ar * (dot(p, torch.fft.ifftn(k2 * torch.fft.fftn(p))) + float((W[i] * (p.real ** 2 + p.imag ** 2)).sum()))
          for i, p in enumerate(psi)]
    return {"psi": [p.cpu().numpy() for p in psi], "its": None, "res": res, "mu": np.array(mu)}


def _exact_train(case, q):
    """Adam on the whole training set (every batch is a permutation of it),
    the learning rate on a cosine from lr to lr / 50."""
    dims, lr = q["dims"], q["lr"]
    x = torch.from_numpy(q["x"]).double().to(_dev())
    t = torch.from_numpy(q["t"]).double().to(_dev())
    par, off = torch.from_numpy(q["par"]).double().to(_dev()), 0
    p = []
    for i, o in zip(dims[:-1], dims[1:]):
        p += [par[off:off + i * o].reshape(i, o).clone(), par[off + i * o:off + i * o + o].clone()]
        off += i * o + o
    m, v = [torch.zeros_like(a) for a in p], [torch.zeros_like(a) for a in p]
    losses = []
    for it in range(case["steps"]):
        acts = [x]
        for l in range(4):
            z = acts[-1] @ p[2 * l] + p[2 * l + 1]
            acts.append(torch.tanh(z) if l < 3 else z)
        diff = acts[-1] - t
        losses.append(float((diff ** 2).mean()))
        d, g = 2.0 * diff / diff.numel(), [None] * 8
        for l in range(3, -1, -1):
            if l < 3:
                d = d * (1 - acts[l + 1] ** 2)
            g[2 * l], g[2 * l + 1] = acts[l].t().contiguous() @ d, d.sum(0)
            d = d @ p[2 * l].t().contiguous()
        rate = lr * 0.02 + (lr - lr * 0.02) * 0.5 * (1 + math.cos(math.pi * it / case["steps"]))
        for a, b, mm, vv in zip(p, g, m, v):
            mm.mul_(0.9).add_(0.1 * b)
            vv.mul_(0.999).add_(0.001 * b * b)
            a.sub_(rate * (mm / (1 - 0.9 ** (it + 1))) / (torch.sqrt(vv / (1 - 0.999 ** (it + 1))) + 1e-8))
    return {"losses": np.array(losses), "params": torch.cat([a.reshape(-1) for a in p]).cpu().numpy()}
