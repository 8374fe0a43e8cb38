"""The workloads that the framework is timed on, through its public entry points.

Three kinds of case:

* ``deck``: a whole tea.in deck through ``run_deck`` (read the deck, set the
  chunk up, run its timesteps to the end), then u and energy1 copied off the
  engine into the caller's device tensors.  The layout is drawn from the seed.
* ``abi``: one timestep through the kernel layer's own entry points, called
  one by one as the Fortran driver calls them: CG, one call per kernel, the
  recurrence on the host.
* ``train``: the loss and the gradient of the warm-start network for one
  batch of training crops.

``exact`` solves the same timesteps (or differentiates the same network) in
64 bits with plain torch.
"""
from __future__ import annotations

import ctypes
import math
import tempfile
from pathlib import Path

import numpy as np
import torch  # before the engine library: torch's HIP runtime is then the process's one

import tealeaf_cuda_amd as tl
from tealeaf_cuda_amd import runtime as rt
from tealeaf_cuda_amd import warmstart as ws

EXTENT = 10.0          # the mesh is [0, 10]^2, as in every deck of the reference
DT = 0.004
MARGIN = 6             # cells at a crop's edge that the training loss leaves out


def _deck(name, solver, prec, nx, ny, steps, eps, halo=1, precision="none", warm="none"):
    return {"name": name, "kind": "deck", "solver": solver, "prec": prec, "nx": nx, "ny": ny, "steps": steps,
            "eps": eps, "halo": halo, "precision": precision, "warm": warm}


def listed():
    return [
        # the smallest benchmark deck of the reference: ten timesteps of about ten CG iterations on 100 cells;
        # a first run, a regression suite, a parameter study on a coarse mesh
        _deck("cg_10", "cg", "none", 10, 10, 10, 1e-15),
        # the reference's 250^2 benchmark (CG, no preconditioner, eps 1e-15), two of its timesteps
        _deck("cg_250", "cg", "none", 250, 250, 2, 1e-15),
        # the reference's single-core 1000^2 benchmark, one timestep
        _deck("cg_1000", "cg", "none", 1000, 1000, 1, 1e-15),
        # the reference's 4000^2 benchmark mesh with the diagonal preconditioner, to the stop of the production decks
        _deck("cg_diag_4000", "cg", "jac_diag", 4000, 4000, 1, 1e-10),
        # Chebyshev on a ragged mesh that is no multiple of any tile
        _deck("cheby_1533x1021", "chebyshev", "none", 1533, 1021, 1, 1e-10),
        # PPCG on a small mesh, the reference's stop: many short timesteps
        _deck("ppcg_block_512", "ppcg", "jac_block", 512, 512, 5, 1e-10),
        # an ordinary ragged PPCG run to the true-residual stop
        _deck("ppcg_diag_1531x997", "ppcg", "jac_diag", 1531, 997, 2, 1e-10, halo=2, precision="fp64"),
        # plain FP64 PPCG at the production size: the baseline that a user compares with
        _deck("ppcg_block_4096", "ppcg", "jac_block", 4096, 4096, 1, 1e-10),
        # FP32 inner solver with FP64 refinement, warm start from the previous steps only
        _deck("fp32_history_2048", "ppcg", "jac_block", 2048, 2048, 4, 1e-10, precision="fp32", warm="extrapolate"),
        # the production configuration: FP32 refinement with the learned warm start
        _deck("learned_4096", "ppcg", "jac_block", 4096, 4096, 3, 1e-10, precision="fp32", warm="network"),
        # the kernel layer under a Fortran-style driver: one launch and one scalar per call
        {"name": "abi_cg_diag_640x480", "kind": "abi", "prec": "jac_diag", "nx": 640, "ny": 480, "eps": 1e-10},
        # one training batch at the trainer's default shape
        {"name": "train_32x128", "kind": "train", "batch": 32, "height": 128, "width": 128, "loss": "energy"},
    ]


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "ppcg", "ppcg", "ppcg", "refined", "refined", "chebyshev", "abi", "train"])
    if kind == "train":
        return {"kind": "train", "batch": rng.choice([8, 16, 24, 32]), "height": 4 * rng.randint(16, 32),
                "width": rng.choice([64, 128]), "loss": rng.choice(["energy", "mse"])}
    top = {"cg": 2400, "ppcg": 3000, "refined": 4096, "chebyshev": 2000, "abi": 1200}[kind]
    low = 10 if kind == "cg" else 64

    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    nx = side(low, top)
    ny = max(low, min(top, side(max(low, nx // 2), min(top, 2 * nx))))
    cells = nx * ny
    if kind == "abi":
        return {"kind": "abi", "prec": rng.choice(["none", "jac_diag", "jac_block"]), "nx": nx, "ny": ny, "eps": 1e-10}
    prec = rng.choice(["none", "jac_diag", "jac_block"])
    eps = rng.choice([1e-10, 1e-12, 1e-15]) if kind == "cg" and cells < 1000 * 1000 else 1e-10
    steps = rng.randint(2, 6) if cells < 1024 * 1024 else (rng.randint(1, 2) if cells < 2200 * 2200 else 1)
    c = _deck("", kind, prec, nx, ny, steps, eps)
    if kind == "cg":
        c["precision"] = rng.choice(["none", "none", "fp64", "fp32"])
        if c["precision"] != "none":
            c["eps"] = 1e-10       # the true residual reaches no 1e-15
    elif kind == "ppcg":
        c["prec"] = rng.choice(["none", "jac_diag", "jac_block", "jac_block"])
        c["halo"] = 1 if c["prec"] == "jac_block" else rng.choice([1, 2, 4])
        c["precision"] = rng.choice(["none", "fp64"])
    elif kind == "refined":
        c["solver"], c["prec"], c["precision"] = "ppcg", "jac_block", "fp32"
        c["steps"] = max(2, steps) if cells < 3600 * 3600 else 2
        c["warm"] = rng.choice(["none", "extrapolate", "network"])
        if c["warm"] == "network":
            c["nx"], c["ny"] = max(64, nx // 64 * 64), max(64, ny // 4 * 4)
    del c["name"]
    return c


# ----------------------------------------------------------------------------- inputs

def _layout(case, seed):
    return tl.random_layout(seed, cells=min(case["nx"], case["ny"]))


def _write_deck(case, states, folder):
    kw = {}
    if case["kind"] == "abi":
        solver, halo, steps = "cg", 1, 1
    else:
        solver, halo, steps = case["solver"], case["halo"], case["steps"]
        if solver in ("chebyshev", "ppcg"):
            kw["ch_cg_presteps"] = 20
        if solver == "ppcg":
            kw["ppcg_inner_steps"] = 10
        if case["precision"] != "none":
            kw["inner_precision"] = case["precision"]
        if case["warm"] == "network":
            kw["warm_start"] = str(ws.default_weights(4096 if case["nx"] > 2048 else 1024))
        elif case["warm"] != "none":
            kw["warm_start"] = case["warm"]
    deck = tl.Deck(x_cells=case["nx"], y_cells=case["ny"], xmax=EXTENT, ymax=EXTENT, initial_timestep=DT,
                   end_step=steps, solver=solver, preconditioner=case["prec"], eps=case["eps"], max_iters=10000,
                   halo_depth=halo, summary_frequency=0, states=states, **kw)
    return deck.write(Path(folder) / "tea.in")


def prepare(case, seed):
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    folder = tempfile.TemporaryDirectory()
    states = _layout(case, seed)
    state = {"case": case, "folder": folder, "deck": _write_deck(case, states, folder.name), "lib": ws.library()}
    for key in ("u", "energy"):
        state[key] = torch.empty((case["ny"], case["nx"]), dtype=torch.float64, device="cuda")
    if case["kind"] == "abi":
        eng = rt.Engine()
        eng.initialise(state["deck"], case["nx"], case["ny"])
        dx, dy = EXTENT / case["nx"], EXTENT / case["ny"]
        eng.initialise_chunk(0.0, 0.0, dx, dy)
        state["engine"] = eng
        # the states as the driver hands them over: extents pulled in by 1/100 of a cell
        rects = [(s.density, s.energy, s.xmin + dx / 100.0, s.xmax - dx / 100.0, s.ymin + dy / 100.0,
                  s.ymax - dy / 100.0, 0.0, rt.G_RECT) for s in states]
        state["states"] = [list(v) for v in zip(*rects)]
    return state


def _planes(case, seed):
    """A batch of training crops as the data generator makes them: density and
    face coefficients of a rectangle layout, smooth step differences of unit
    RMS, and a small smooth target."""
    b, h, w = case["batch"], case["height"], case["width"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def uniform(*shape):
        return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)

    y = torch.arange(h, device="cuda", dtype=torch.float64)[None, :, None]
    x = torch.arange(w, device="cuda", dtype=torch.float64)[None, None, :]
    rho = torch.full((b, h, w), 2.0, device="cuda", dtype=torch.float64)   # log10 density
    for _ in range(4):
        ends = uniform(b, 4)
        x0, x1 = torch.minimum(ends[:, 0], ends[:, 1]) * w, torch.maximum(ends[:, 0], ends[:, 1]) * w
        y0, y1 = torch.minimum(ends[:, 2], ends[:, 3]) * h, torch.maximum(ends[:, 2], ends[:, 3]) * h
        inside = ((x >= x0[:, None, None]) & (x < x1[:, None, None]) &
                  (y >= y0[:, None, None]) & (y < y1[:, None, None]))
        rho = torch.where(inside, (3.0 * uniform(b) - 1.0)[:, None, None], rho)

    def smooth(rms):
        f = torch.zeros((b, h, w), device="cuda", dtype=torch.float64)
        for _ in range(6):
            a = uniform(b, 4)[:, :, None, None]
            f += (a[:, 0] - 0.5) * torch.sin(2 * math.pi * (3 * a[:, 1] * x / w + 3 * a[:, 2] * y / h + a[:, 3]))
        return rms * f / f.square().mean(dim=(1, 2), keepdim=True).sqrt()

    d = 10.0 ** rho
    face = DT / (EXTENT / 1024) ** 2
    kx, ky = torch.zeros_like(d), torch.zeros_like(d)
    kx[:, :, 1:] = face * (d[:, :, :-1] + d[:, :, 1:]) / (2.0 * d[:, :, :-1] * d[:, :, 1:])
    ky[:, 1:, :] = face * (d[:, :-1, :] + d[:, 1:, :]) / (2.0 * d[:, :-1, :] * d[:, 1:, :])
    planes = [(rho - 0.5) / 1.5, smooth(1.0), smooth(1.0), smooth(0.1), kx, ky]
    return torch.stack(planes, dim=1).float().contiguous()


def _prepare_train(case, seed):
    trainer = ws.Trainer(case["batch"], case["height"], case["width"], margin=MARGIN, loss=case["loss"])
    trainer.set_params(ws.load_weights(ws.default_weights(1024)))
    return {"case": case, "trainer": trainer, "samples": _planes(case, seed)}


# ----------------------------------------------------------------------------- one pass

def _copy_out(state):
    for fid, key in ((rt.FIELD_U, "u"), (rt.FIELD_ENERGY1, "energy")):
        if state["lib"].tea_engine_copy_field(fid, ctypes.c_void_p(state[key].data_ptr())) != 0:
            raise tl.TeaError("tea_engine_copy_field failed")


def _run_abi(state):
    """One timestep of tea_solve.f90's CG, kernel by kernel."""
    eng, case = state["engine"], state["case"]
    eng.generate_chunk(*state["states"])
    eng.set_field_kernel()
    eng.common_init(rt.CONDUCTIVITY, DT)
    eng.calc_residual()
    initial = math.sqrt(eng.calc_2norm(1))
    rro = eng.cg_init()
    for _ in range(10000):
        alpha = rro / eng.cg_calc_w()
        rrn = eng.cg_calc_ur(alpha)
        eng.cg_calc_p(rrn / rro)
        rro = rrn
        if math.sqrt(abs(rrn)) < case["eps"] * initial:
            break
    eng.finalise()
    summary = eng.field_summary()
    _copy_out(state)
    return {"u": state["u"], "energy": state["energy"], "summary": list(summary)}


def run(state):
    kind = state["case"]["kind"]
    if kind == "train":
        loss, grad = state["trainer"].gradient(state["samples"])
        return {"loss": loss, "gradient": grad}
    if kind == "abi":
        return _run_abi(state)
    final = tl.run_deck(state["deck"]).final
    _copy_out(state)
    return {"u": state["u"], "energy": state["energy"],
            "summary": [final.volume, final.mass, final.energy, final.u]}


def work(case):
    """Bytes: each timestep reads density and energy and writes u and energy
    (a training batch: its planes, parameters and gradient).  Operations: the
    five-point products, updates and sums of the iterations that the solve
    needs, after the usual bound sqrt(kappa)/2 ln(2/eps) with the mesh's
    coupling, and for the network 2 per multiply-add, forward and backward."""
    if case["kind"] == "train":
        cells = case["batch"] * case["height"] * case["width"]
        macs = 27 * 32 + 4 * 9 * 32 * 32 + 9 * 32
        return {"bytes": 4.0 * (6 * cells + 2 * ws.param_count()), "flops": 6.0 * macs * cells}
    cells = case["nx"] * case["ny"]
    steps = case.get("steps", 1)
    coupling = DT * ((case["nx"] / EXTENT) ** 2 + (case["ny"] / EXTENT) ** 2)
    kappa = 1.0 + 4.0 * coupling * (1.0 if case["prec"] != "none" else 4.0)
    iterations = max(5.0, 0.5 * math.sqrt(kappa) * math.log(2.0 / case["eps"]) * 0.25)
    return {"bytes": 32.0 * cells * steps, "flops": 20.0 * cells * steps * iterations}


# ----------------------------------------------------------------------------- 64-bit values

def _fields(case, seed):
    """density and energy of the layout on the mesh (generate_chunk's rectangles)."""
    nx, ny = case["nx"], case["ny"]
    dx, dy = EXTENT / nx, EXTENT / ny
    vx = dx * torch.arange(nx + 1, device="cuda", dtype=torch.float64)
    vy = dy * torch.arange(ny + 1, device="cuda", dtype=torch.float64)
    states = _layout(case, seed)
    rho = torch.full((ny, nx), states[0].density, device="cuda", dtype=torch.float64)
    energy = torch.full((ny, nx), states[0].energy, device="cuda", dtype=torch.float64)
    for s in states[1:]:
        in_x = (vx[1:] >= s.xmin + dx / 100.0) & (vx[:-1] < s.xmax - dx / 100.0)
        in_y = (vy[1:] >= s.ymin + dy / 100.0) & (vy[:-1] < s.ymax - dy / 100.0)
        inside = in_y[:, None] & in_x[None, :]
        rho = torch.where(inside, s.density, rho)
        energy = torch.where(inside, s.energy, energy)
    return rho, energy


def _solve(kx, ky, b, tol=1e-15):
    """A x = b by Jacobi-preconditioned CG from x = b, restarted on the true residual."""
    diag = torch.ones_like(b)
    diag[:, 1:] += kx
    diag[:, :-1] += kx
    diag[1:, :] += ky
    diag[:-1, :] += ky

    def apply(x):
        fx, fy = kx * (x[:, 1:] - x[:, :-1]), ky * (x[1:, :] - x[:-1, :])
        y = x.clone()
        y[:, 1:] += fx
        y[:, :-1] -= fx
        y[1:, :] += fy
        y[:-1, :] -= fy
        return y

    x = b.clone()
    floor = tol * float(torch.linalg.vector_norm(b))
    last = math.inf
    for _ in range(4):
        r = b - apply(x)
        size = float(torch.linalg.vector_norm(r))
        if size <= floor or size > 0.5 * last:
            break
        last = size
        z = r / diag
        p = z.clone()
        rz = torch.sum(r * z)
        d = torch.zeros_like(b)
        target = max(1e-9 * size, 0.1 * floor)
        for k in range(1, 20001):
            q = apply(p)
            alpha = rz / torch.sum(p * q)
            d.add_(alpha * p)
            r.sub_(alpha * q)
            if k % 25 == 0 and float(torch.linalg.vector_norm(r)) <= target:
                break
            z = r / diag
            new = torch.sum(r * z)
            p = z + (new / rz) * p
            rz = new
        x = x + torch.where(torch.isfinite(d), d, torch.zeros_like(d))
    return x


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    rho, energy = _fields(case, seed)
    dx, dy = EXTENT / case["nx"], EXTENT / case["ny"]
    kx = DT / (dx * dx) * (rho[:, :-1] + rho[:, 1:]) / (2.0 * rho[:, :-1] * rho[:, 1:])
    ky = DT / (dy * dy) * (rho[:-1, :] + rho[1:, :]) / (2.0 * rho[:-1, :] * rho[1:, :])
    u = None
    for _ in range(case.get("steps", 1)):
        u = _solve(kx, ky, energy * rho)
        energy = u / rho
    v = dx * dy
    summary = [v * rho.numel(), float(v * rho.sum()), float(v * (rho * energy).sum()), float(v * (rho * u).sum())]
    return {"u": u, "energy": energy, "summary": summary}


def _exact_train(case, seed):
    """Loss and gradient of the six-layer network in 64 bits: each layer as
    nine shifted products, differentiated by autograd."""
    planes = _planes(case, seed).double()
    flat = torch.from_numpy(ws.load_weights(ws.default_weights(1024))).to("cuda").double().requires_grad_(True)
    b, h, w = case["batch"], case["height"], case["width"]
    at = 0

    def take(*shape):
        nonlocal at
        n = int(np.prod(shape))
        part = flat[at:at + n].reshape(shape)
        at += n
        return part

    def conv(a, weight, bias):
        padded = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        out = bias
        for tap in range(9):
            dy, dx = divmod(tap, 3)
            rows = padded[:, dy:dy + h, dx:dx + w].reshape(b * h * w, a.shape[3])
            out = out + rows @ weight[tap]
        return out.reshape(b, h, w, weight.shape[2])

    a = planes[:, :3].permute(0, 2, 3, 1)
    a = torch.relu(conv(a, take(9, 3, 32), take(32)))
    for _ in range(4):
        a = torch.relu(conv(a, take(9, 32, 32), take(32)))
    out = conv(a, take(9, 32, 1), take(1))[..., 0]
    mask = torch.zeros((h, w), device="cuda", dtype=torch.float64)
    mask[MARGIN:h - MARGIN, MARGIN:w - MARGIN] = 1.0
    e = (out - planes[:, 3]) * mask
    total = e.square().sum()
    if case["loss"] == "energy":
        fx, fy = mask[:, 1:] * mask[:, :-1], mask[1:, :] * mask[:-1, :]
        total = total + (planes[:, 4, :, 1:] * fx * (e[:, :, 1:] - e[:, :, :-1]).square()).sum()
        total = total + (planes[:, 5, 1:, :] * fy * (e[:, 1:, :] - e[:, :-1, :]).square()).sum()
    loss = total / (b * float(mask.sum()))
    loss.backward()
    return {"loss": float(loss.detach()), "gradient": flat.grad}
