"""Performance cases of the EVP-FFT solver: the work its users have it do, through the public Python API.

Kinds of case (``kind``):

* ``increments`` -- a loading path in progress: a solver opened on a polycrystal (FCC copper, x3
  tension at 1e-3 1/s with stress-free lateral faces, 0.01% strain per increment, Err 2e-5), already a
  few increments in, so that the texture rotates.  One pass advances it by ``increments`` converged
  increments, then reads the macroscopic response and the stress, deformation and orientation fields,
  as a run that writes its fields every few increments does.
* ``dump`` -- the fields of one output step (the set the reference writes at a PrintControl step).
* ``fft`` -- the transform entry points on host arrays: half-spectrum forward and its inverse.
* ``ensemble`` -- a batch of small independent polycrystals from deck files to their final reports.
* ``train`` -- training of the learned Newton start on recorded-like samples.

A mixed-precision run's fields carry FP32 transforms, and its users keep them as float32 arrays; FP64
runs keep float64.
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

import srx_amd
from srx_amd import inputs

NSTEPS = 1 << 20          # more increments than any measurement takes
WARM_INCREMENTS = 4       # increments before the measured ones (the texture rotates from the fourth)


def listed() -> list:
    inc = dict(kind="increments", gnd=0, warm_start=0)
    return [
        # the smallest RVE in use (the 16^3 deck of the tests): latency and launches of one increment
        dict(inc, name="increments_16_fp64", n0=16, n1=16, n2=16, grains=8, precision="fp64", increments=4),
        # extents that are no powers of two and differ per axis
        dict(inc, name="increments_45x60x50_fp64", n0=45, n1=60, n2=50, grains=30, precision="fp64", increments=3),
        # the in-plane grid of the reference's own deck, 256 x 256 x 1
        dict(inc, name="increments_256x256x1_fp64", n0=256, n1=256, n2=1, grains=60, precision="fp64", increments=3),
        # the drop-in check configuration: 64^3, 125 grains
        dict(inc, name="increments_64_mixed", n0=64, n1=64, n2=64, grains=125, precision="mixed", increments=4),
        # the same RVE with geometrically necessary dislocations
        dict(inc, name="increments_64_gnd_fp64", n0=64, n1=64, n2=64, grains=125, precision="fp64", increments=4,
             gnd=1),
        # an ensemble member's size, with the extrapolated Newton start
        dict(inc, name="increments_96_mixed_ws1", n0=96, n1=96, n2=96, grains=300, precision="mixed", increments=4,
             warm_start=1),
        # the headline workload, 128^3 and 1000 grains, in both precisions
        dict(inc, name="increments_128_mixed", n0=128, n1=128, n2=128, grains=1000, precision="mixed", increments=6),
        dict(inc, name="increments_128_fp64", n0=128, n1=128, n2=128, grains=1000, precision="fp64", increments=6),
        # one output step's fields
        dict(kind="dump", name="dump_64_fp64", n0=64, n1=64, n2=64, grains=125, precision="fp64"),
        # six tensor components through the transforms
        dict(kind="fft", name="fft_6x60x64x75_fp64", comps=6, n0=60, n1=64, n2=75, precision="fp64"),
        # a batch of uneven small RVEs, three increments each
        dict(kind="ensemble", name="ensemble_8x16to40", members=8, nmin=16, nmax=40, steps=3, concurrency=4),
        # training of the learned start, default batch
        dict(kind="train", name="train_64k", samples=65536, epochs=4, batch=4096),
    ]


SMOOTH = sorted({2 ** a * 3 ** b * 5 ** c for a in range(8) for b in range(5) for c in range(4)
                 if 12 <= 2 ** a * 3 ** b * 5 ** c <= 128})


def _extent(rng, lo: int, hi: int) -> int:
    """A supported extent, spread over the logarithm of [lo, hi]."""
    x = lo * (hi / lo) ** rng.random()
    return min((s for s in SMOOTH if lo <= s <= hi), key=lambda s: abs(s - x))


def draw(rng) -> dict:
    u = rng.random()
    if u < 0.70:
        while True:
            n = [_extent(rng, 12, 120) for _ in range(3)]
            if rng.random() < 0.1:
                n[2] = 1
                n[0] = rng.choice((96, 120, 128, 160, 200, 256))
                n[1] = rng.choice((96, 120, 128, 160, 200, 256))
            if 1500 <= n[0] * n[1] * n[2] <= 900000:
                break
        gnd = 1 if rng.random() < 0.15 else 0
        return dict(kind="increments", n0=n[0], n1=n[1], n2=n[2], grains=rng.randint(8, 200),
                    precision=rng.choice(("fp64", "mixed")), increments=rng.randint(1, 3), gnd=gnd,
                    warm_start=0 if gnd else rng.choice((0, 0, 1)))
    if u < 0.80:
        n = [_extent(rng, 16, 72) for _ in range(3)]
        return dict(kind="dump", n0=n[0], n1=n[1], n2=n[2], grains=rng.randint(8, 100),
                    precision=rng.choice(("fp64", "mixed")))
    if u < 0.90:
        n = [_extent(rng, 12, 80) for _ in range(3)]
        return dict(kind="fft", comps=rng.randint(1, 9), n0=n[0], n1=n[1], n2=n[2],
                    precision=rng.choice(("fp64", "mixed")))
    if u < 0.95:
        return dict(kind="ensemble", members=rng.randint(3, 8), nmin=12, nmax=rng.choice((24, 30, 36, 40)),
                    steps=rng.randint(2, 3), concurrency=rng.choice((0, 2, 4)))
    return dict(kind="train", samples=rng.randint(8000, 65536), epochs=rng.randint(1, 4),
                batch=rng.choice((1024, 4096)))


def _precision(case) -> int:
    return srx_amd.PREC_MIXED if case["precision"] == "mixed" else srx_amd.PREC_FP64


def _write_case(folder: str, n, grains: int, seed: int, nsteps: int) -> str:
    """Deck, slip file and mesh of a periodic Voronoi polycrystal with uniform random orientations
    (as inputs.make_case writes them, the voxels assigned to their nearest seed on the GPU)."""
    os.makedirs(folder, exist_ok=True)
    rng = np.random.default_rng(seed)
    box = torch.tensor([float(x) for x in n], device="cuda")
    pts = torch.from_numpy(rng.random((grains, 3)).astype(np.float32)).cuda() * box
    N = n[0] * n[1] * n[2]
    owner = np.empty(N, np.int64)
    step = 1 << 17
    for s in range(0, N, step):
        v = torch.arange(s, min(N, s + step), device="cuda")
        d2 = torch.zeros((len(v), grains), device="cuda")
        for a, c in enumerate((v // (n[1] * n[2]), (v // n[2]) % n[1], v % n[2])):
            d = (c.float()[:, None] + 0.5 - pts[None, :, a]).abs()
            d = torch.minimum(d, box[a] - d)
            d2 += d * d
        owner[s:s + len(v)] = d2.argmin(1).cpu().numpy() + 1
    rot = inputs.random_rotations(rng, grains)
    eul = inputs.matrix_to_bunge(np.transpose(rot, (0, 2, 1)))
    inputs.write_sx(os.path.join(folder, "Cu_p.sx"))
    inputs.write_mesh_grains(os.path.join(folder, "mesh.txt"), n, eul, owner)
    deck = os.path.join(folder, "deck.in")
    inputs.write_deck(deck, n=n, nsteps=nsteps, timestep=0.1)
    return deck


def _open(case, seed: int):
    with tempfile.TemporaryDirectory(prefix="srx_perf_") as folder:
        deck = _write_case(folder, (case["n0"], case["n1"], case["n2"]), case["grains"], seed, NSTEPS)
        s = srx_amd.Solver(deck, precision=_precision(case), gnd=case.get("gnd", 0),
                           warm_start=case.get("warm_start", 0))
    for _ in range(WARM_INCREMENTS):
        s.step()
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("increments", "dump"):
        return {"case": case, "solver": _open(case, seed)}
    if kind == "fft":
        g = torch.Generator(device="cuda").manual_seed(seed)
        shape = (case["comps"], case["n0"], case["n1"], case["n2"])
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
        y = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
        return {"case": case, "x": x.cpu().numpy(), "spectrum": np.fft.rfftn(y.cpu().numpy(), axes=(1, 2, 3))}
    if kind == "ensemble":
        rng = np.random.default_rng(seed)
        folder = tempfile.TemporaryDirectory(prefix="srx_perf_")
        sizes = [s for s in SMOOTH if case["nmin"] <= s <= case["nmax"]] or [case["nmin"]]
        decks = []
        for k in range(case["members"]):   # evenly spread sizes, the largest first
            e = sizes[(len(sizes) - 1) * (case["members"] - 1 - k) // max(case["members"] - 1, 1)]
            decks.append(_write_case(os.path.join(folder.name, "rve%02d" % k), (e, e, e), int(rng.integers(10, 60)),
                                     seed + k, case["steps"]))
        return {"case": case, "folder": folder, "decks": decks}
    # recorded-like samples: a unit quaternion, a unit direction, the stress / 100 MPa, the bounded
    # forcing, a log ratio and a log density; targets a smooth function of them plus noise
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = case["samples"]
    x = torch.randn((n, 24), generator=g, device="cuda")
    x[:, 0:4] /= x[:, 0:4].norm(dim=1, keepdim=True)
    x[:, 4:10] /= x[:, 4:10].norm(dim=1, keepdim=True)
    x[:, 16:22] /= 1.0 + x[:, 16:22].norm(dim=1, keepdim=True)
    x[:, 22] = -3.0 + 0.5 * x[:, 22]
    x[:, 23] *= 0.05
    w = torch.randn((24, 6), generator=g, device="cuda") / 5.0
    t = torch.tanh(x @ w) + 0.05 * torch.randn((n, 6), generator=g, device="cuda")
    return {"case": case, "x": x.cpu().numpy(), "t": t.cpu().numpy()}


REPORT = ("time_tot", "e_vm", "evmp", "d_vm", "dvmp", "s_vm", "s_vm1", "rho_F_avg", "rho_P_avg", "rho_s_avg",
          "rho_m_avg", "rho_g_avg", "rho_forest_avg", "rho_inplane_avg")
AVERAGES = ("sig_avg", "eps_avg", "edot_avg", "disgrad_avg_actual", "velgrad_avg")


def _report(rep: dict) -> dict:
    out = {"scalars": np.array([rep[k] for k in REPORT])}
    out.update({k: np.array(rep[k]) for k in AVERAGES})
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "increments":
        s = state["solver"]
        for _ in range(case["increments"]):
            rep = s.step()
        out = _report(rep)
        out.update({k: s.field(k) for k in ("sig", "disgrad", "tranmat")})
    elif kind == "dump":
        s = state["solver"]
        out = {k: s.field(k) for k in ("sig", "eps", "disgrad", "tranmat", "rho_s", "trial_gam_acum")}
    elif kind == "fft":
        prec = _precision(case)
        scale = 1.0 / (case["n0"] * case["n1"] * case["n2"])
        return {"forward": srx_amd.fft_forward(state["x"], prec),
                "inverse": srx_amd.fft_inverse(state["spectrum"], case["n2"], prec, scale)}
    elif kind == "ensemble":
        res = srx_amd.run_ensemble(state["decks"], concurrency=case["concurrency"])
        return [_report(r["last"]) for r in res]
    else:
        blob, hist = srx_amd.mlp_train(state["x"], state["t"], epochs=case["epochs"], batch=case["batch"])
        return {"weights": blob, "loss": hist}
    if case["precision"] == "mixed":   # kept in single precision
        out = {k: torch.from_numpy(v).to(torch.float32) for k, v in out.items()}
    return out


def exact(case, seed):
    """The transforms in 64 bits by numpy.  The solver's fixed point, the ensemble's reports and a
    training run have no value outside this repository."""
    if case["kind"] != "fft":
        return None
    st = prepare(case, seed)
    n = (case["n0"], case["n1"], case["n2"])
    return {"forward": np.fft.rfftn(st["x"], axes=(1, 2, 3)),
            "inverse": np.fft.irfftn(st["spectrum"], s=n, axes=(1, 2, 3))}


OUTER_ITERS = 57.0        # outer iterations of an increment of this loading (50-increment average)
NEWTON_ITERS = 3.3        # Newton iterations per voxel and outer iteration
NEWTON_FLOPS = 2300.0     # algorithmic flops of one Newton iteration of one voxel


def _increment_work(N: float, gnd: int) -> tuple:
    """Bytes and flops of one increment of N voxels: per outer iteration the stress and the strain (6
    components each) read and written, 6 + 6 real transforms and the Newton solve; per increment
    the dislocation state (12 systems, 7 arrays), orientation and strain read and written."""
    it_bytes = 4 * 6 * 8.0 * N
    it_flops = NEWTON_FLOPS * NEWTON_ITERS * N + 12 * 2.5 * N * math.log2(max(N, 2.0))
    state = 2 * (7 * 12 + 9 + 9 + 5 + (48 if gnd else 0)) * 8.0 * N
    return OUTER_ITERS * it_bytes + state, OUTER_ITERS * it_flops


def work(case) -> dict:
    kind = case["kind"]
    if kind == "ensemble":
        sizes = [s for s in SMOOTH if case["nmin"] <= s <= case["nmax"]] or [case["nmin"]]
        b = f = 0.0
        for k in range(case["members"]):
            e = sizes[(len(sizes) - 1) * (case["members"] - 1 - k) // max(case["members"] - 1, 1)]
            bb, ff = _increment_work(float(e ** 3), 0)
            b += case["steps"] * bb + 59.0 * e ** 3
            f += case["steps"] * ff
        return {"bytes": b, "flops": f}
    if kind == "train":
        params = 24 * 64 + 64 * 64 + 64 * 6
        return {"bytes": 4.0 * 30 * case["samples"] * case["epochs"], "flops": 6.0 * params * case["samples"] * case["epochs"]}
    N = float(case["n0"] * case["n1"] * case["n2"])
    if kind == "increments":
        b, f = _increment_work(N, case["gnd"])
        return {"bytes": case["increments"] * b + (6 + 9 + 9 + 27) * 8.0 * N, "flops": case["increments"] * f}
    if kind == "dump":
        return {"bytes": 2 * (4 * 9 + 2 * 12) * 8.0 * N, "flops": 0.0}
    return {"bytes": 4 * case["comps"] * 8.0 * N, "flops": 2 * case["comps"] * 2.5 * N * math.log2(N)}
