"""Cases for timing fullmag_amd through its public entry points.

A case is one pass of what a user's program does with a backend it keeps:
time steps with their diagnostics and the state handed over afterwards, a
batched sweep, a differentiable rollout, a multilayer stack, field copies.
`prepare` builds the backend (plan, Newell tensor, magnetisation) and the
buffers a program keeps; `run` makes one pass; `exact` is the same pass in
plain torch / numpy in 64 bits (Newell-Williams-Dunlop tensor, torch.fft
convolution, exchange, Landau-Lifshitz torque, the Runge-Kutta methods).

The state of a double backend is returned as it is (FP64).  Mixed and single
precision carry FP32 fields, so their results are handed over in FP32.
"""

import functools
import math

import numpy as np
import torch
import torch.utils.checkpoint

import fullmag_amd as fa

MU0 = 4.0 * math.pi * 1e-7
GAMMA = 2.211e5


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: the 64x64x1 film of the parity workload, FP64
        # Heun; a step is a handful of launches, so latency is what counts
        dict(name="film_64x64x1_double", kind="step", nx=64, ny=64, nz=1, dx=5.0, dy=5.0, dz=3.0, ms=8e5, a=1.3e-11,
             alpha=0.5, field=10.0, dt=1e-13, integrator="heun", precision="double", m0="random", mask=False, steps=10),
        # muMAG standard problem 4 (500 x 125 x 3 nm) in 1 nm cells: a film
        # whose padded lengths are not powers of two
        dict(name="sp4_500x125x1_mixed", kind="step", nx=500, ny=125, nz=1, dx=1.0, dy=1.0, dz=3.0, ms=8e5, a=1.3e-11,
             alpha=0.02, field=25.0, dt=2e-14, integrator="heun", precision="mixed", m0="smooth", mask=False, steps=10),
        # the headline film: 512x512x8, mixed precision Heun from a random m0
        dict(name="film_512x512x8_mixed", kind="step", nx=512, ny=512, nz=8, dx=4.0, dy=4.0, dz=2.0, ms=8.6e5,
             a=1.3e-11, alpha=0.02, field=30.0, dt=5e-14, integrator="heun", precision="mixed", m0="random",
             mask=False, steps=4),
        # the same film on the FP64 parity path
        dict(name="film_512x512x8_double", kind="step", nx=512, ny=512, nz=8, dx=4.0, dy=4.0, dz=2.0, ms=8.6e5,
             a=1.3e-11, alpha=0.02, field=30.0, dt=5e-14, integrator="heun", precision="double", m0="random",
             mask=False, steps=2),
        # a ragged slab in the reference's single precision
        dict(name="slab_250x150x6_single", kind="step", nx=250, ny=150, nz=6, dx=4.0, dy=4.0, dz=3.0, ms=8e5,
             a=1.3e-11, alpha=0.1, field=20.0, dt=5e-14, integrator="heun", precision="single", m0="smooth",
             mask=True, steps=8),
        # the 3-D block of the DP45 workload
        dict(name="block_256x256x64_dp45_mixed", kind="step", nx=256, ny=256, nz=64, dx=2.0, dy=2.0, dz=2.0, ms=1.4e6,
             a=2.1e-11, alpha=0.01, field=0.0, dt=3e-14, integrator="dp45", precision="mixed", m0="vortex",
             mask=False, steps=2),
        # a cube with an even but not power-of-two edge, RK4 in FP64
        dict(name="cube_100_rk4_double", kind="step", nx=100, ny=100, nz=100, dx=3.0, dy=3.0, dz=3.0, ms=8e5,
             a=1.3e-11, alpha=0.05, field=50.0, dt=5e-14, integrator="rk4", precision="double", m0="vortex",
             mask=False, steps=2),
        # a disc with the sub-cell boundary tier (face links, volume
        # fractions, correction rows)
        dict(name="disc_256x256x4_tier_mixed", kind="tier", nx=256, ny=256, nz=4, dx=4.0, dy=4.0, dz=2.0, ms=8.6e5,
             a=1.3e-11, alpha=0.02, field=10.0, dt=5e-14, tier="volume", precision="mixed", steps=8),
        # a parameter sweep: 32 instances of 16 grids in one graph-captured batch
        dict(name="sweep_32_batch_mixed", kind="batch", sizes="32,64,128,256", layers="1,2,4,8", copies=2,
             precision="mixed", dt=1e-13, steps=20, per_graph=10),
        # the differentiable film: forward and backward through torch.autograd
        dict(name="rollout_128x128x4_double", kind="rollout", nx=128, ny=128, nz=4, dx=5.0, dy=5.0, dz=3.0, a=1.3e-11,
             alpha=0.1, dt=1e-13, precision="double", steps=40, every=10),
        # three coupled films
        dict(name="stack_3x512x512_mixed", kind="stack", nx=512, ny=512, layers=3, gap=1.0, dx=4.0, dy=4.0, dz=1.0,
             precision="mixed", dt=5e-14, steps=4),
        # a program that looks at fields: upload m, refresh, copy H_demag and
        # H_eff to the host, one preview
        dict(name="fields_256x256x8_mixed", kind="fields", nx=256, ny=256, nz=8, dx=4.0, dy=4.0, dz=2.0, ms=8e5,
             a=1.3e-11, field=20.0, precision="mixed", m0="smooth", mask=True, preview=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Films and slabs of 16 to 512 cells by 1 to 8 layers, 3-D blocks of 24
    to 256 by 9 to 64 layers, discs with boundary tiers, sweeps, rollouts,
    stacks and field copies; every precision and integrator that steps them."""
    kind = rng.choice(["film"] * 5 + ["block"] * 3 + ["tier", "batch", "rollout", "stack", "fields"])
    prec = rng.choice(["mixed", "mixed", "double", "single"])
    edge = round(rng.uniform(2.0, 5.0), 2)
    if kind in ("film", "block"):
        if kind == "film":
            nx, ny, nz = _log_int(rng, 16, 512), _log_int(rng, 16, 512), rng.randint(1, 8)
        else:
            nx, ny, nz = _log_int(rng, 24, 256), _log_int(rng, 24, 256), _log_int(rng, 9, 64)
        return dict(kind="step", nx=nx, ny=ny, nz=nz, dx=edge, dy=round(rng.uniform(2.0, 5.0), 2),
                    dz=round(rng.uniform(2.0, 4.0), 2), ms=8e5, a=1.3e-11, alpha=round(rng.uniform(0.01, 0.5), 3),
                    field=round(rng.uniform(5.0, 50.0), 1), dt=2e-14,
                    integrator=rng.choice(["heun", "heun", "heun", "rk4", "rk23", "dp45"]), precision=prec,
                    m0=rng.choice(["random", "smooth", "vortex"]), mask=rng.random() < 0.3,
                    steps=2 if nx * ny * nz > 500_000 else 6)
    if kind == "tier":
        return dict(kind="tier", nx=rng.randint(48, 256), ny=rng.randint(48, 256), nz=rng.randint(1, 4), dx=edge,
                    dy=edge, dz=2.0, ms=8e5, a=1.3e-11, alpha=0.05, field=10.0, dt=2e-14,
                    tier=rng.choice(["volume", "full"]), precision=rng.choice(["mixed", "double"]), steps=6)
    if kind == "batch":
        sizes = sorted({_log_int(rng, 24, 200) for _ in range(3)})
        return dict(kind="batch", sizes=",".join(map(str, sizes)), layers=rng.choice(["1", "1,2", "1,4", "2,5,8"]),
                    copies=rng.randint(1, 4), precision=rng.choice(["mixed", "double"]), dt=5e-14, steps=12,
                    per_graph=rng.choice([3, 6, 12]))
    if kind == "rollout":
        return dict(kind="rollout", nx=_log_int(rng, 24, 128), ny=_log_int(rng, 24, 128), nz=rng.randint(1, 4), dx=edge,
                    dy=edge, dz=3.0, a=1.3e-11, alpha=0.1, dt=5e-14, precision=rng.choice(["mixed", "double"]),
                    steps=rng.randint(12, 40), every=rng.randint(4, 10))
    if kind == "stack":
        return dict(kind="stack", nx=_log_int(rng, 48, 512), ny=_log_int(rng, 48, 512), layers=rng.randint(2, 5),
                    gap=round(rng.uniform(0.5, 3.0), 2), dx=edge, dy=edge, dz=1.0,
                    precision=rng.choice(["mixed", "double"]), dt=2e-14, steps=4)
    return dict(kind="fields", nx=_log_int(rng, 32, 400), ny=_log_int(rng, 32, 400), nz=rng.randint(1, 8), dx=edge,
                dy=edge, dz=2.0, ms=8e5, a=1.3e-11, field=20.0, precision=prec, m0=rng.choice(["smooth", "vortex"]),
                mask=rng.random() < 0.5, preview=rng.choice([16, 32]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _unit(v):
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _m0(kind, nx, ny, nz, rng):
    """Initial magnetisation (cells, 3), x fastest: random on the sphere, a
    smooth in-plane modulation, or a vortex, the last two with 1% noise."""
    n = nx * ny * nz
    if kind == "random":
        return _unit(rng.standard_normal((n, 3)))
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    if kind == "smooth":
        th = 0.4 * np.sin(2 * np.pi * x / nx + rng.uniform(0, 6)) + 0.2 * np.cos(2 * np.pi * y / ny)
        v = np.stack([np.cos(th), np.sin(th), np.full(th.shape, 0.1)], -1)
    else:
        v = np.stack([-(y - (ny - 1) / 2), x - (nx - 1) / 2, np.full(x.shape, 0.1 * max(nx, ny))], -1)
    v = _unit(v)
    v = np.broadcast_to(v[None], (nz, ny, nx, 3)).reshape(-1, 3)
    return _unit(v + 0.01 * rng.standard_normal(v.shape))


def _disc(nx, ny, nz):
    y, x = np.meshgrid(np.arange(ny) + 0.5, np.arange(nx) + 0.5, indexing="ij")
    one = ((2 * x / nx - 1) ** 2 + (2 * y / ny - 1) ** 2 <= 1.0).astype(np.uint8)
    return np.broadcast_to(one[None], (nz, ny, nx)).reshape(-1).copy()


def _field(mt, rng):
    d = _unit(rng.standard_normal(3))
    return tuple(float(v) for v in mt * 1e-3 / MU0 * d)


def _cell(case):
    return tuple(case[k] * 1e-9 for k in ("dx", "dy", "dz"))


def _step_inputs(case, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    m0 = _m0(case.get("m0", "random"), nx, ny, nz, rng)
    mask = _disc(nx, ny, nz) if case.get("mask") else None
    h = _field(case["field"], rng) if case["field"] > 0 else None
    return m0, mask, h


def _step_plan(case, m0, mask, h, **kw):
    return fa.FdmPlan(cells=(case["nx"], case["ny"], case["nz"]), cell_size=_cell(case), initial_magnetization=m0,
                      saturation_magnetisation=case["ms"], exchange_stiffness=case["a"],
                      damping=case.get("alpha", 0.1), precision=case["precision"],
                      integrator=case.get("integrator", "heun"), external_field=h, active_mask=mask,
                      demag_kernel="device", **kw)


@functools.lru_cache(maxsize=4)
def _disc_geometry(nx, ny, nz, dx, dy, dz, delta):
    from fullmag_amd import boundary

    radius = 0.42 * min(nx * dx, ny * dy)
    return boundary.compute_boundary_geometry(boundary.cylinder_sdf(radius, nx * dx / 2, ny * dy / 2), nx, ny, nz, dx,
                                              dy, dz, delta)


def _sweep_members(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["copies"]):
        for s in (int(v) for v in case["sizes"].split(",")):
            for l in (int(v) for v in case["layers"].split(",")):
                out.append(dict(nx=s, ny=s, nz=l, dx=5.0, dy=5.0, dz=3.0, ms=float(rng.uniform(4e5, 1.4e6)),
                                a=float(rng.uniform(5e-12, 2e-11)), alpha=float(rng.uniform(0.005, 0.5)),
                                precision=case["precision"], m=_m0("random", s, s, l, rng),
                                h=_field(100.0 * rng.uniform(), rng)))
    return out


def _rollout_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["nx"] * case["ny"] * case["nz"]
    m0 = _m0("smooth", case["nx"], case["ny"], case["nz"], rng)
    ms = rng.uniform(6e5, 9e5, n)
    h = np.array([20.0, 5.0, 0.0]) * 1e-3 / MU0
    w = rng.standard_normal((n, 3)) / n
    return m0, ms, h, w


def _stack_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["nx"] * case["ny"]
    layers = [dict(m=_m0("random", case["nx"], case["ny"], 1, rng), ms=8e5 if l % 2 == 0 else 6e5,
                   z=l * (case["dz"] + case["gap"]) * 1e-9) for l in range(case["layers"])]
    return layers, (0.01 / MU0, 0.0, 0.0), n


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "tier"):
        m0, mask, h = _step_inputs(case, seed)
        kw = {}
        if kind == "tier":
            g = _disc_geometry(case["nx"], case["ny"], case["nz"], *_cell(case), case["tier"] == "full")
            mask = (g.volume_fraction > 0).astype(np.uint8)
            kw = dict(boundary_correction=case["tier"], boundary_geometry=g)
        b = fa.NativeFdmBackend(_step_plan(case, m0, mask, h, **kw))
        out = torch.empty(3, b.cell_count, dtype=torch.float64, device="cuda") if case["precision"] != "single" else None
        return dict(case=case, backend=b, out=out)
    if kind == "batch":
        members = [fa.NativeFdmBackend(_step_plan(p, p["m"], None, p["h"])) for p in _sweep_members(case, seed)]
        outs = [torch.empty(3, b.cell_count, dtype=torch.float64, device="cuda") for b in members]
        batch = fa.BatchRun(members, [case["dt"]] * len(members), steps_per_graph=case["per_graph"])
        return dict(case=case, members=members, batch=batch, outs=outs)
    if kind == "rollout":
        m0, ms, h, w = _rollout_inputs(case, seed)
        plan = fa.FdmPlan(cells=(case["nx"], case["ny"], case["nz"]), cell_size=_cell(case), initial_magnetization=m0,
                          saturation_magnetisation=8e5, exchange_stiffness=case["a"], damping=case["alpha"],
                          precision=case["precision"], demag_kernel="device")
        dt = torch.float64 if case["precision"] == "double" else torch.float32
        return dict(case=case, plan=plan, m0=m0, ms=torch.tensor(ms, dtype=dt), h=torch.tensor(h, dtype=dt),
                    w=torch.tensor(w, dtype=torch.float64, device="cuda"), dtype=dt)
    if kind == "stack":
        layers, h, n = _stack_inputs(case, seed)
        cell = _cell(case)
        grid = (case["nx"], case["ny"], 1)
        plan = fa.FdmMultilayerPlan(
            common_cells=grid, convolution_cell_size=cell, external_field=h, precision=case["precision"],
            layers=[fa.FdmLayerPlan(magnet_name=f"L{i}", native_grid=grid, native_cell_size=cell,
                                    native_origin=(0.0, 0.0, l["z"]), initial_magnetization=l["m"],
                                    saturation_magnetisation=l["ms"], exchange_stiffness=1.3e-11, damping=0.02)
                    for i, l in enumerate(layers)])
        outs = [torch.empty(3, n, dtype=torch.float64, device="cuda") for _ in layers]
        return dict(case=case, stack=fa.MultilayerStack(plan), outs=outs)
    m0, mask, h = _step_inputs(case, seed)
    new = _step_inputs(case, seed + 7919)[0]
    return dict(case=case, backend=fa.NativeFdmBackend(_step_plan(case, m0, mask, h)), m=new)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _report(stats, double):
    """Energies and maxima of one or several StepStats, one row each."""
    t = np.float64 if double else np.float32
    rows = stats if isinstance(stats, list) else [stats]
    return {"energy": np.array([[s.e_ex, s.e_demag, s.e_ext, s.e_total] for s in rows], dtype=t),
            "h_max": np.array([[s.max_h_eff, s.max_h_demag] for s in rows], dtype=t),
            "rate": np.array([s.max_dm_dt for s in rows], dtype=t)}


def _state(backend, out, double):
    backend.copy_state_device(out.data_ptr())
    return out if double else out.to(torch.float32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    double = case["precision"] == "double"
    if kind in ("step", "tier"):
        b = state["backend"]
        for _ in range(case["steps"]):
            s = b.step(case["dt"])
        if state["out"] is None:
            return {"m": b.copy_field_f32("m"), **_report(s, double)}
        torch.cuda.current_stream().synchronize()  # the buffer's last reader, before the library writes it again
        return {"m": _state(b, state["out"], double), **_report(s, double)}
    if kind == "batch":
        stats = state["batch"].run(case["steps"])
        torch.cuda.current_stream().synchronize()
        return {"m": [_state(b, o, double) for b, o in zip(state["members"], state["outs"])], **_report(stats, double)}
    if kind == "rollout":
        ms = state["ms"].clone().requires_grad_(True)
        h = state["h"].clone().requires_grad_(True)
        m = fa.heun_rollout(state["m0"], ms, h, state["plan"], case["dt"], case["steps"], case["every"])
        loss = (m * state["w"]).sum()
        loss.backward()
        return {"m": m.detach().to(state["dtype"]), "g_ms": ms.grad, "g_h": h.grad}
    if kind == "stack":
        st = state["stack"]
        s = st.step(case["dt"], case["steps"])
        torch.cuda.current_stream().synchronize()
        return {"m": [_state(l, o, double) for l, o in zip(st.layers, state["outs"])], **_report(s, double)}
    b = state["backend"]
    p = case["preview"]
    if double:
        b.upload_magnetization(state["m"])
        b.refresh_observables()
        return {"h_demag": b.copy_field("H_demag"), "h_eff": b.copy_field("H_eff"),
                "preview": b.copy_live_preview_field("m", (min(p, case["nx"]), min(p, case["ny"]), 1))}
    b.upload_magnetization(state["m"])
    b.refresh_observables()
    return {"h_demag": b.copy_field_f32("H_demag"), "h_eff": b.copy_field_f32("H_eff"),
            "preview": b.copy_live_preview_field("m", (min(p, case["nx"]), min(p, case["ny"]), 1), f32=True)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
_EVALS = {"heun": 2, "rk4": 4, "rk23": 3, "dp45": 6}


def _step_work(nx, ny, nz, precision, evals, steps):
    """Per step the state is read and written and the Newell tensor (real,
    one octant of the padded spectrum, six components or four in the film
    plane) is read; per field evaluation six real transforms of the padded
    grid (half-length complex transforms), the tensor product and about 100
    operations per cell for exchange and torque."""
    n = nx * ny * nz
    q = 4 if precision == "single" else 8
    r = 8 if precision == "double" else 4
    pad = 4 * n if nz == 1 else 8 * n
    tensor = (4 if nz == 1 else 6) * (nx + 1) * (ny + 1) * (1 if nz == 1 else nz + 1) * r
    flops = evals * (6 * 2.5 * pad * math.log2(pad) + 0.5 * pad * 30 + 100.0 * n)
    return steps * (2 * 3 * n * q + tensor), steps * flops


def work(case):
    kind = case["kind"]
    if kind in ("step", "tier"):
        b, f = _step_work(case["nx"], case["ny"], case["nz"], case["precision"],
                          _EVALS[case.get("integrator", "heun")], case["steps"])
    elif kind == "batch":
        b = f = 0.0
        for s in (int(v) for v in case["sizes"].split(",")):
            for l in (int(v) for v in case["layers"].split(",")):
                w = _step_work(s, s, l, case["precision"], 2, case["steps"])
                b, f = b + case["copies"] * w[0], f + case["copies"] * w[1]
    elif kind == "rollout":
        # forward, its recomputation, and per backward step four more
        # evaluations with the transposed operators
        b, f = _step_work(case["nx"], case["ny"], case["nz"], case["precision"], 2, case["steps"])
        b, f = 4 * b, 4 * f
    elif kind == "stack":
        b, f = _step_work(case["nx"], case["ny"], 1, case["precision"], 2, case["steps"])
        b, f = case["layers"] * b, case["layers"] * f
    else:
        b, f = _step_work(case["nx"], case["ny"], case["nz"], case["precision"], 1, 1)
        n = case["nx"] * case["ny"] * case["nz"]
        b += 3 * n * (8 + 2 * (8 if case["precision"] == "double" else 4))
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# The same passes in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _newell_f(x, y, z):
    """Newell, Williams and Dunlop (1993), the diagonal integral."""
    x2, y2, z2 = x * x, y * y, z * z
    r = np.sqrt(x2 + y2 + z2)
    with np.errstate(all="ignore"):
        v = (2 * x2 - y2 - z2) * r / 6
        v = v + np.where(x2 + z2 > 0, y * (z2 - x2) / 2 * np.arcsinh(y / np.sqrt(x2 + z2)), 0)
        v = v + np.where(x2 + y2 > 0, z * (y2 - x2) / 2 * np.arcsinh(z / np.sqrt(x2 + y2)), 0)
        v = v - np.where((x != 0) & (r > 0), x * y * z * np.arctan(y * z / (x * r)), 0)
    return v


def _newell_g(x, y, z):
    x2, y2, z2 = x * x, y * y, z * z
    r = np.sqrt(x2 + y2 + z2)
    with np.errstate(all="ignore"):
        v = -x * y * r / 3
        v = v + np.where(x2 + y2 > 0, x * y * z * np.arcsinh(z / np.sqrt(x2 + y2)), 0)
        v = v + np.where(y2 + z2 > 0, y * (3 * z2 - y2) / 6 * np.arcsinh(x / np.sqrt(y2 + z2)), 0)
        v = v + np.where(x2 + z2 > 0, x * (3 * z2 - x2) / 6 * np.arcsinh(y / np.sqrt(x2 + z2)), 0)
        v = v - np.where((z != 0) & (r > 0), z2 * z / 6 * np.arctan(x * y / (z * r)), 0)
        v = v - np.where((y != 0) & (r > 0), y2 * z / 2 * np.arctan(x * z / (y * r)), 0)
        v = v - np.where((x != 0) & (r > 0), x2 * z / 2 * np.arctan(y * z / (x * r)), 0)
    return v


_NEAR = 40  # cells; beyond, the tensor is the point dipole's, as the framework defines it


def _octant(nx, ny, nz, cell, z_off=0.0):
    """Newell tensor xx, yy, zz, xy, xz, yz at the displacements (i, j, k) of
    the non-negative octant (k shifted by z_off), shape (6, nz, ny, nx); near
    cells in extended precision from the 27-point second difference."""
    dx, dy, dz = cell
    ax = [torch.arange(m, dtype=torch.float64, device=_dev()) * d for m, d in zip((nx, ny, nz), cell)]
    ax[2] = ax[2] + z_off
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    r2 = x * x + y * y + z * z
    r2 = torch.where(r2 > 0, r2, torch.ones_like(r2))
    r3 = r2 * r2.sqrt()
    c = dx * dy * dz / (4 * math.pi)
    out = torch.stack([c * (1 / r3 - 3 * x * x / (r3 * r2)), c * (1 / r3 - 3 * y * y / (r3 * r2)),
                       c * (1 / r3 - 3 * z * z / (r3 * r2)), -3 * c * x * y / (r3 * r2), -3 * c * x * z / (r3 * r2),
                       -3 * c * y * z / (r3 * r2)])
    mx, my, mz = (min(m, _NEAR) for m in (nx, ny, nz))
    ld = np.longdouble
    ex, ey = (np.arange(-1, m + 1).astype(ld) * ld(d) for m, d in zip((mx, my), cell))
    ez = np.arange(-1, mz + 1).astype(ld) * ld(dz) + ld(z_off)
    Z, Y, X = np.meshgrid(ez, ey, ex, indexing="ij")
    near = np.zeros((6, mz, my, mx))
    for q, t in enumerate((_newell_f(X, Y, Z), _newell_f(Y, X, Z), _newell_f(Z, Y, X), _newell_g(X, Y, Z),
                           _newell_g(X, Z, Y), _newell_g(Y, Z, X))):
        for axis in range(3):
            lo, mid, hi = (np.take(t, np.arange(s, t.shape[axis] - 2 + s), axis) for s in (0, 1, 2))
            t = 2 * mid - lo - hi
        near[q] = (t / (4 * ld(math.pi) * ld(dx) * ld(dy) * ld(dz))).astype(np.float64)
    k, j, i = np.meshgrid(np.arange(mz), np.arange(my), np.arange(mx), indexing="ij")
    use = torch.tensor(i * i + j * j + k * k < _NEAR * _NEAR, device=_dev())
    part = out[:, :mz, :my, :mx]
    out[:, :mz, :my, :mx] = torch.where(use, torch.tensor(near, device=_dev()), part)
    return out


_ODD = ((0, 0, 0), (0, 0, 0), (0, 0, 0), (1, 1, 0), (1, 0, 1), (0, 1, 1))


class _Demag:
    """H = -N * (Ms m) on one grid by zero-padded FFTs in FP64; z_off != 0
    gives the field of a layer on one that far above it."""

    def __init__(self, nx, ny, nz, cell, z_off=0.0):
        self.n = (nz, ny, nx)
        self.p = (1 if nz == 1 else 2 * nz, 2 * ny, 2 * nx)
        o = _octant(nx, ny, nz, cell, z_off)
        spec = []
        for q in range(6):
            k = torch.zeros(self.p, dtype=torch.float64, device=_dev())
            t = o[q]
            for sz in ((1,) if nz == 1 else (1, -1)):
                for sy in (1, -1):
                    for sx in (1, -1):
                        v, dst = t, []
                        for axis, (s, m, p) in enumerate(zip((sz, sy, sx), self.n, self.p)):
                            if s > 0:
                                dst.append(slice(0, m))
                            else:
                                v = v.flip(axis).narrow(axis, 0, m - 1)
                                dst.append(slice(p - m + 1, p))
                        sign = 1.0
                        for s, odd in zip((sx, sy, sz), _ODD[q]):
                            sign *= s if odd else 1.0
                        k[tuple(dst)] = sign * v
            spec.append(torch.fft.rfftn(k))
        self.k = spec

    def spectrum(self, mag):
        """mag: (3, nz, ny, nx), Ms m."""
        return torch.fft.rfftn(mag, s=self.p, dim=(1, 2, 3))

    def apply(self, s):
        xx, yy, zz, xy, xz, yz = self.k
        return -torch.stack([xx * s[0] + xy * s[1] + xz * s[2], xy * s[0] + yy * s[1] + yz * s[2],
                             xz * s[0] + yz * s[1] + zz * s[2]])

    def back(self, s):
        nz, ny, nx = self.n
        return torch.fft.irfftn(s, s=self.p, dim=(1, 2, 3))[:, :nz, :ny, :nx]

    def field(self, mag):
        return self.back(self.apply(self.spectrum(mag)))


class _Film:
    """One magnet in FP64: fields, torque and diagnostics."""

    def __init__(self, nx, ny, nz, cell, ms, a, alpha, h, mask=None, demag=True):
        self.shape, self.cell, self.ms, self.a, self.alpha = (nz, ny, nx), cell, ms, a, alpha
        self.h = torch.tensor(h if h is not None else (0.0, 0.0, 0.0), dtype=torch.float64, device=_dev())
        self.has_h = h is not None
        self.mask = None if mask is None else torch.tensor(mask.reshape(nz, ny, nx) != 0, device=_dev())
        self.demag = _Demag(nx, ny, nz, cell) if demag else None

    def load(self, m0):
        m = torch.tensor(np.ascontiguousarray(m0.reshape(*self.shape, 3).transpose(3, 0, 1, 2)), device=_dev())
        return m if self.mask is None else m * self.mask

    def exchange(self, m):
        lap = torch.zeros_like(m)
        act = self.mask
        for axis, d in zip((3, 2, 1), self.cell):
            if m.shape[axis] == 1:
                continue
            for s in (1, -1):
                nb = m.roll(s, axis)
                edge = [slice(None)] * 4
                edge[axis] = 0 if s > 0 else m.shape[axis] - 1
                ok = torch.ones(self.shape, dtype=torch.bool, device=m.device)
                ok[tuple(edge[1:])] = False
                if act is not None:
                    ok = ok & act.roll(s, axis - 1)
                lap = lap + torch.where(ok, nb - m, torch.zeros_like(m)) / d**2
        h = 2 * self.a / (MU0 * self.ms) * lap
        return h if act is None else h * act

    def fields(self, m, hd=None):
        hx = self.exchange(m)
        if hd is None:
            hd = self.demag.field(self.ms * m)
        if self.mask is not None:
            hd = hd * self.mask
        he = self.h.view(3, 1, 1, 1).expand_as(m)
        if self.mask is not None:
            he = he * self.mask
        return hx, hd, he

    def torque(self, m, h):
        p = torch.cross(m, h, dim=0)
        return -GAMMA / (1 + self.alpha**2) * (p + self.alpha * torch.cross(m, p, dim=0))

    def rhs(self, m, hd=None):
        return self.torque(m, sum(self.fields(m, hd)))

    def report(self, m, hd=None):
        hx, hd, he = self.fields(m, hd)
        w = MU0 * self.ms * math.prod(self.cell)
        if torch.is_tensor(w):
            w = w.expand(self.shape)
        e = [float((-0.5 * w * (m * hx).sum(0)).sum()), float((-0.5 * w * (m * hd).sum(0)).sum()),
             float((-w * (m * he).sum(0)).sum())]
        h = hx + hd + he
        norm = lambda v: float(v.square().sum(0).max().sqrt())  # noqa: E731
        return e + [sum(e)], [norm(h), norm(hd)], norm(self.torque(m, h))


def _norm(v):
    n = v.square().sum(0, keepdim=True).sqrt()
    return torch.where(n > 0, v / torch.where(n > 0, n, torch.ones_like(n)), torch.zeros_like(v))


# stage points a_ij and weights of the methods, every point renormalised
_TABLE = {
    "heun": ([[1.0]], [0.5, 0.5]),
    "rk4": ([[0.5], [0.0, 0.5], [0.0, 0.0, 1.0]], [1 / 6, 1 / 3, 1 / 3, 1 / 6]),
    "rk23": ([[0.5], [0.0, 0.75]], [2 / 9, 1 / 3, 4 / 9]),
    "dp45": ([[1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
              [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
              [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656]],
             [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]),
}


def _advance(rhs, m, dt, method, steps):
    points, weights = _TABLE[method]
    for _ in range(steps):
        k = [rhs(m)]
        for row in points:
            k.append(rhs(_norm(m + dt * sum(c * v for c, v in zip(row, k) if c))))
        m = _norm(m + dt * sum(c * v for c, v in zip(weights, k) if c))
    return m


def _rows(reports):
    return {"energy": np.array([r[0] for r in reports]), "h_max": np.array([r[1] for r in reports]),
            "rate": np.array([r[2] for r in reports])}


def _aos(m):
    return m.permute(1, 2, 3, 0).reshape(-1, 3)


def exact(case, seed):
    kind = case["kind"]
    if kind == "tier":
        return None  # the planner's sampled geometry has no closed form outside the framework
    if kind == "step":
        m0, mask, h = _step_inputs(case, seed)
        f = _Film(case["nx"], case["ny"], case["nz"], _cell(case), case["ms"], case["a"], case["alpha"], h, mask)
        m = _advance(f.rhs, f.load(m0), case["dt"], case["integrator"], case["steps"])
        rep = _rows([f.report(m)])
        return {"m": _aos(m) if case["precision"] == "single" else m.reshape(3, -1), **rep}
    if kind == "batch":
        ms, reps = [], []
        for p in _sweep_members(case, seed):
            f = _Film(p["nx"], p["ny"], p["nz"], _cell(p), p["ms"], p["a"], p["alpha"], p["h"])
            m = _advance(f.rhs, f.load(p["m"]), case["dt"], "heun", case["steps"])
            ms.append(m.reshape(3, -1))
            reps.append(f.report(m))
        return {"m": ms, **_rows(reps)}
    if kind == "rollout":
        m0, ms, h, w = _rollout_inputs(case, seed)
        shape = (case["nz"], case["ny"], case["nx"])
        f = _Film(case["nx"], case["ny"], case["nz"], _cell(case), 1.0, case["a"], case["alpha"], h)
        ms_t = torch.tensor(ms.reshape(shape), device=_dev(), requires_grad=True)
        h_t = torch.tensor(h, device=_dev(), requires_grad=True)
        f.ms, f.h = ms_t, h_t
        m = f.load(m0)
        step = lambda v, a, b: _advance(f.rhs, v, case["dt"], "heun", 1)  # noqa: E731
        for _ in range(case["steps"]):
            m = torch.utils.checkpoint.checkpoint(step, m, ms_t, h_t, use_reentrant=False)
        out = _aos(m)
        (out * torch.tensor(w, device=_dev())).sum().backward()
        return {"m": out.detach(), "g_ms": ms_t.grad.reshape(-1), "g_h": h_t.grad}
    if kind == "stack":
        layers, h, n = _stack_inputs(case, seed)
        grid = (case["nx"], case["ny"], 1)
        cell = _cell(case)
        fs = [_Film(*grid, cell, l["ms"], 1.3e-11, 0.02, h, demag=False) for l in layers]
        ker = {}
        for a in layers:
            for b in layers:
                d = a["z"] - b["z"]
                if d not in ker:
                    ker[d] = _Demag(*grid, cell, d)

        def coupled(ms):
            s = [ker[0.0].spectrum(f.ms * m) for f, m in zip(fs, ms)]
            return [ker[0.0].back(sum(ker[a["z"] - b["z"]].apply(v) for b, v in zip(layers, s))) for a in layers]

        def rhs(m):
            ms = list(m.unbind(1))
            return torch.stack([f.rhs(v, hd) for f, v, hd in zip(fs, ms, coupled(ms))], 1)

        m = torch.stack([f.load(l["m"]) for f, l in zip(fs, layers)], 1)
        m = _advance(rhs, m, case["dt"], "heun", case["steps"])
        ms = list(m.unbind(1))
        reps = [f.report(v, hd) for f, v, hd in zip(fs, ms, coupled(ms))]
        rep = ([sum(r[0][q] for r in reps) for q in range(4)], [max(r[1][q] for r in reps) for q in range(2)],
               max(r[2] for r in reps))
        return {"m": [v.reshape(3, -1) for v in ms], **_rows([rep])}
    _, mask, h = _step_inputs(case, seed)
    new = _step_inputs(case, seed + 7919)[0]
    f = _Film(case["nx"], case["ny"], case["nz"], _cell(case), case["ms"], case["a"], 0.1, h, mask)
    m = f.load(new)
    parts = f.fields(m)
    p = [min(case["preview"], case[k]) for k in ("nx", "ny")]
    flat = m[:, 0].cpu().numpy()
    edge = lambda n, q: [(b * n // q, max((b + 1) * n // q, b * n // q + 1)) for b in range(q)]  # noqa: E731
    pre = np.array([[flat[:, y0:y1, x0:x1].mean(axis=(1, 2)) for x0, x1 in edge(case["nx"], p[0])]
                    for y0, y1 in edge(case["ny"], p[1])]).reshape(-1, 3)
    return {"h_demag": _aos(parts[1]), "h_eff": _aos(sum(parts)), "preview": pre}
