"""Timing cases of the explicit GeoFLAC step: what a user of this framework has it do.

Each case is one pass of a user's program through the public entry points: a stretch
of the time loop on a model that is already on the device, then the fields the program
looks at brought back to its host arrays (an output interval, made short).  Listed are
the driver's own loop on the smallest box, single models from 60x20 elements to the
2 million elements of half the benchmark box, each precision mode, the stress
boundaries, the surface processes, parameter sweeps in one batch, the learned
viscosity, and the gradient that trains its network.  `draw` gives other sizes and
options of the same ranges.

Model states are the framework's own new starts (model.build_box) of the two decks in
geoflac_amd/configs on meshes of other sizes.  The host state of a mesh is built once
per process; a seed then gives each model its own cohesion factors, thermal anomaly,
friction, and pulling velocity.
"""
import functools
import math
import os

import numpy as np
import torch

from geoflac_amd import abi, gpu, inp, model, sweep, train_surrogate

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CONFIGS = os.path.join(ROOT, "geoflac_amd", "configs")

PRECISION = {"fp64": abi.PREC_FP64, "mixed": abi.PREC_MIXED, "storage": abi.PREC_MIXED_STORAGE}
# what a program looks at after a stretch of steps: mesh, velocity, temperature,
# stress, plastic strain and viscosity
FIELDS = ("cord", "vel", "temp", "stress0", "aps", "visn")

BASE = {"kind": "step", "deck": "box60x20", "nelx": 60, "nelz": 20, "precision": "fp64", "steps": 100,
        "option": "plain"}


def listed():
    c = lambda name, **kw: dict(BASE, name=name, **kw)  # noqa: E731
    return [
        # the reference driver's loop with the drop-in `flac`: one call per step, the
        # remeshing test every ntest_rem = 10 steps; the smallest deck, launches and latency
        c("driver_60x20", kind="driver", steps=20),
        # a small model with erosion and sedimentation on its surface
        c("topo_60x20", option="topo", steps=200),
        # odd sizes; hydrostatic side walls, a stress on part of the surface, Winkler base
        c("stressbc_151x47", option="stressbc", nelx=151, nelz=47, steps=300),
        # an ordinary regional model, drop-in precision, four layers
        c("layers_400x100", deck="layers4000x1000", nelx=400, nelz=100, steps=400),
        # a fine regional model on the two-layer box, odd in both directions
        c("box_901x301", nelx=901, nelz=301, steps=400),
        # the largest: half the benchmark box's elements, the same rows
        c("layers_2000x1000", deck="layers4000x1000", nelx=2000, nelz=1000, steps=400),
        # the FP32 modes on models of the sizes they are used at
        c("mixed_1000x250", deck="layers4000x1000", nelx=1000, nelz=250, precision="mixed", steps=500),
        c("storage_1200x500", deck="layers4000x1000", nelx=1200, nelz=500, precision="storage", steps=300),
        # the learned viscosity in the FP32-arithmetic step, with its audits
        c("learned_1000x250", deck="layers4000x1000", nelx=1000, nelz=250, precision="mixed", option="learned",
          steps=300),
        # parameter sweeps: many small models per launch, meshes of 100-600 x 40-150 in FP32
        # arithmetic, and smaller ones in drop-in precision
        {"name": "sweep_24_mixed", "kind": "sweep", "models": 24, "nx_lo": 100, "nx_hi": 600, "nz_lo": 40, "nz_hi": 150,
         "mesh_seed": 0, "precision": "mixed", "steps": 300},
        {"name": "sweep_12_fp64", "kind": "sweep", "models": 12, "nx_lo": 60, "nx_hi": 240, "nz_lo": 20, "nz_hi": 80,
         "mesh_seed": 1, "precision": "fp64", "steps": 200},
        # training the viscosity network: the gradient over a large minibatch on the device
        {"name": "mlp_grad_65536", "kind": "mlp_grad", "n": 65536},
    ]


def draw(rng):
    logint = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    kind = rng.choice(["step"] * 6 + ["driver", "sweep", "mlp_grad"])
    if kind == "mlp_grad":
        return {"kind": kind, "n": logint(1000, 400000)}
    if kind == "sweep":
        lo, hi = rng.choice([(100, 600), (60, 240), (80, 300)])
        return {"kind": kind, "models": rng.randint(3, 16), "nx_lo": lo, "nx_hi": hi, "nz_lo": max(20, lo // 3),
                "nz_hi": hi // 4, "mesh_seed": rng.randint(2, 1 << 20), "precision": rng.choice(["mixed", "fp64", "storage"]),
                "steps": 100}
    if kind == "driver":
        return dict(BASE, kind=kind, nelx=logint(30, 200), nelz=logint(12, 60), steps=20)
    nelx = logint(40, 1500)
    nelz = max(12, min(700, int(nelx * rng.uniform(0.2, 0.6))))
    deck = rng.choice(["box60x20", "layers4000x1000"])
    option = rng.choice(["plain", "plain", "plain", "topo", "stressbc"]) if deck == "box60x20" else "plain"
    precision = rng.choice(["fp64", "fp64", "mixed", "storage"]) if option == "plain" else "fp64"
    if option == "topo":  # (the marker arrays are allocated to their capacity)
        nelx, nelz = min(nelx, 400), min(nelz, 100)
    return dict(BASE, deck=deck, nelx=nelx, nelz=nelz, precision=precision, option=option, steps=10 * rng.randint(8, 25))


# ---------------------------------------------------------------- preparing a model
def _params(deck, nelx, nelz, option):
    p = sweep.variant(inp.read_inp(os.path.join(CONFIGS, deck + ".inp")), nelx, nelz)
    if option == "topo":
        # diffusion of the surface with resurfacing, and a weak block for the extension to localise in
        p["topo_kappa"] = 1e-3
        mid = nelx // 2
        p["inhom"], p["inhoms"] = 1, [dict(ix1=max(1, mid - 1), ix2=mid + 2, iy1=1, iy2=max(2, nelz * 2 // 5),
                                           inphase=-1, igeom=0, xinitaps=0.5)]
    elif option == "stressbc":
        # the surface 1 km under the sea, walls in hydrostatic equilibrium, -5 MPa on a third
        # of the surface, a Winkler base in place of the bottom's velocity condition
        p["z0"] = -1000.0
        p["nystressbc"], p["nydrsides"], p["nyhydro"] = 1, 1, 2
        p["bcs"] = [b for b in p["bcs"] if b["nofside"] in (1, 3)]
        p["bcs"].append(dict(p["bcs"][0], nofside=4, nbc1=1 + nelx // 3, nbc2=1 + 2 * nelx // 3, nbc=20, bca=-5.0e6))
        p["nofbc"] = len(p["bcs"])
    return p


@functools.lru_cache(maxsize=64)
def _built(deck, nelx, nelz, option):
    """The new-start host state of one mesh (kept: a seed only changes a copy of it)."""
    # (interfaces moved by up to 2 km per column, as the benchmark's box)
    return model.build_box(_params(deck, nelx, nelz, option), interface_noise=2.0 if option == "plain" else 0.0, seed=0)


def _new_model(deck, nelx, nelz, option, precision, rng):
    gp0, st0 = _built(deck, nelx, nelz, option)
    gp, st = type(gp0).from_buffer_copy(gp0), st0.copy()
    ez, ex = nelz, nelx
    st.coh_scale = np.asfortranarray((1.0 + 0.01 * rng.uniform(-1.0, 1.0, size=(ez, ex))).astype(np.float32))
    # a smooth thermal anomaly of some kelvin between the fixed surface and base
    x, z = np.linspace(0.0, math.pi, nelx + 1)[None, :], np.linspace(0.0, math.pi, nelz + 1)[:, None]
    for k in (1, 2, 3, 5):
        st.temp[1:-1, :] += (rng.uniform(-10.0, 10.0) / k * np.cos(k * x + rng.uniform(0.0, 3.0)) * np.sin(k * z))[1:-1]
    st.temp0[...] = st.temp
    f = 1.0 + 0.1 * float(rng.uniform(-1.0, 1.0))
    st.bc *= f
    gp.vbc = gp.vbc * f
    fric, coh = float(rng.uniform(20.0, 32.0)), float(rng.uniform(2.0e7, 5.0e7))
    for k in range(gp.nphase):
        gp.fric1[k], gp.cohesion1[k] = fric, coh
    m = gpu.Model(gp, st, precision=PRECISION[precision])
    model.device_setup(m)
    if option == "learned":
        w, cfg, _ = train_surrogate.load(os.path.join(ROOT, "geoflac_amd", "weights", "visc_mlp_layers4000x1000.npz"))
        m.surrogate_weights(w, cfg)
        m.surrogate_enable(True, tol=0.5, audit_stride=64)
    return m


class _Sweep:
    """A batch and its models, given back in the order the library asks for."""

    def __init__(self, models):
        self.models = models
        self.batch = sweep.Batch(models)
        self.batch.set_graph(True)

    def __del__(self):
        if hasattr(self, "batch"):
            self.batch.close()


def _mlp_inputs(case, seed):
    """Normalised samples of the viscosity network and weights of its initialisation's
    scale, from the seed, in 32 bits."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["n"], 8)).astype(np.float32)
    x[:, 3:7] = rng.dirichlet(np.ones(4), case["n"]).astype(np.float32)
    x[:, 7] = np.tanh(x[:, 0] + 0.5 * x[:, 1] - 0.3 * x[:, 2]) + 0.05 * x[:, 7]
    b = lambda n, fan: rng.uniform(-1, 1, n) / math.sqrt(fan)  # noqa: E731
    w = np.concatenate([b(64 * 7, 7), b(64, 7), b(64 * 64, 64), b(64, 64), b(64, 64), b(1, 64)]).astype(np.float32)
    return x, w


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp_grad":
        x, w = _mlp_inputs(case, seed)
        return {"case": case, "x": torch.from_numpy(x).cuda(), "w": torch.from_numpy(w).cuda(),
                "grad": torch.empty(gpu.MLP_NPARAM + 1, dtype=torch.float32, device="cuda")}
    rng = np.random.default_rng(seed)
    if kind == "sweep":
        mesh = np.random.default_rng(case["mesh_seed"])
        models = []
        for _ in range(case["models"]):
            nelx = int(mesh.integers(case["nx_lo"], case["nx_hi"] + 1))
            nelz = int(mesh.integers(case["nz_lo"], case["nz_hi"] + 1))
            models.append(_new_model("box60x20", nelx, nelz, "plain", case["precision"], rng))
        return {"case": case, "sweep": _Sweep(models)}
    return {"case": case,
            "model": _new_model(case["deck"], case["nelx"], case["nelz"], case["option"], case["precision"], rng)}


# ---------------------------------------------------------------- one pass
def _fields(m, names=FIELDS):
    m.download(sum(abi.FIELD_BIT[n] for n in names))
    return {n: getattr(m.state, n) for n in names}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mlp_grad":
        rc = gpu.lib().gf_mlp_grad_noalloc(state["x"].data_ptr(), case["n"], state["w"].data_ptr(),
                                           state["grad"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("gf_mlp_grad_noalloc: %d" % rc)
        return state["grad"]
    if kind == "sweep":
        sw = state["sweep"]
        sw.batch.step(case["steps"])
        # (a sweep looks at the velocities and plastic strain of each model)
        return [_fields(m, ("vel", "aps")) for m in sw.models]
    m = state["model"]
    if kind == "driver":
        # the reference driver's inner loop around the drop-in (src/par.f90:81-95)
        c = m.state.clock
        tests = []
        for _ in range(case["steps"] // 10):
            for _ in range(10):
                m.call("flac")
                c.nloop += 1
                c.time += c.dt
            tests.append(m.itest_mesh(3, 1.3, 11.0))
        return dict(_fields(m), tests=tests)
    m.step(case["steps"])
    out = _fields(m)
    if case["option"] == "topo":
        m.download(abi.GF_TOPO)
        out["dtopo"], out["dhacc"] = m.state.dtopo, m.state.dhacc
    return out


# ---------------------------------------------------------------- what a pass needs
def _step_bytes(E, N, precision):
    """State that one step reads and writes once.  Per element: the stress (16 values),
    strain, plastic strain, averaged strain rate and heat in and out; viscosity,
    source and phase in.  Per node: coordinates, velocity and temperature in and out;
    both masses and the boundary values and codes in."""
    sv = 8 if precision == "fp64" else 4
    return E * (2 * (16 * sv + 24 + 8 + 24 + 8) + 8 + 8 + 4) + N * (2 * (16 + 2 * sv + 8) + 16 + 16 + 8)


STEP_FLOPS = 1200  # per element: four triangles of strain rate, rotation and stress update, the gather, diffusion


def work(case):
    if case["kind"] == "mlp_grad":
        n = case["n"]
        return {"bytes": 32.0 * n + 8.0 * gpu.MLP_NPARAM, "flops": 6.0 * gpu.MLP_NPARAM * n}
    if case["kind"] == "sweep":
        mesh = np.random.default_rng(case["mesh_seed"])
        E = N = 0
        for _ in range(case["models"]):
            nelx = int(mesh.integers(case["nx_lo"], case["nx_hi"] + 1))
            nelz = int(mesh.integers(case["nz_lo"], case["nz_hi"] + 1))
            E, N = E + nelx * nelz, N + (nelx + 1) * (nelz + 1)
    else:
        E, N = case["nelx"] * case["nelz"], (case["nelx"] + 1) * (case["nelz"] + 1)
    return {"bytes": float(case["steps"]) * _step_bytes(E, N, case["precision"]),
            "flops": float(case["steps"]) * STEP_FLOPS * E}


def exact(case, seed):
    """The network's gradient and summed squared error in 64 bits.  The stretches of the
    step have none: hundreds of steps of a serial in-place sweep and of a discontinuous
    choice per element, over 20 seconds in plain numpy."""
    if case["kind"] != "mlp_grad":
        return None
    x, w = (torch.from_numpy(a).double() for a in _mlp_inputs(case, seed))
    W1, b1 = w[:448].view(64, 7).requires_grad_(), w[448:512].clone().requires_grad_()
    W2, b2 = w[512:4608].view(64, 64).clone().requires_grad_(), w[4608:4672].clone().requires_grad_()
    W3, b3 = w[4672:4736].clone().requires_grad_(), w[4736:4737].clone().requires_grad_()
    h = torch.nn.functional.silu(x[:, :7] @ W1.t() + b1)
    h = torch.nn.functional.silu(h @ W2.t() + b2)
    sse = ((h @ W3 + b3 - x[:, 7]) ** 2).sum()
    (sse / case["n"]).backward()
    return torch.cat([t.grad.reshape(-1) for t in (W1, b1, W2, b2, W3, b3)] + [sse.detach().reshape(1)])
