"""The work that a user of this package has it do, as cases that can be timed.

Four kinds of program are stood for:

  solo    one shot in FP64 through ``capi.Context``, the path that replaces
          the reference's time loop;
  shots   many shots on one mesh in one FP32 batch (``capi.BatchContext``);
  uneven  independent instances of different size and order, packed by order
          (``uneven.PackedBatch``) and advanced as one ``capi.Group``;
  mlp     the learned surrogate's network (``mlp.MLP``): training, gradients
          and inference.

A time-loop case is either ``whole`` (the state is reset, every step is run
and the seismograms are fetched) or a ``chunk`` of a longer run (the next
``chunk`` steps and what has been recorded so far: how the trigger of the PML
and the movie frames divide a run).  The set-up of a mesh is kept for the
process, as a program that solves many shots keeps it; sources, tensors,
velocities, start fields, weights and samples come from the seed.

``exact`` restates the time loop and the network in 64 bits with torch, on the
arrays the set-up hands over; it uses none of this package's kernels.
"""
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nexd-3d_amd"))

from nexd_amd import batch, capi, layout, mesh as meshmod, mlp, problem, sources as srcmod, uneven  # noqa: E402

DEV = "cuda"
ORDERS_POINTS = {1: 4, 2: 10, 3: 20, 4: 35, 5: 56}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _solo(name, n, order, timeint, nt, pml=0, chunk=0):
    nx, ny, nz = n
    return dict(name=name, kind="solo", nx=nx, ny=ny, nz=nz, order=order, timeint=timeint, nt=nt, pml=pml, chunk=chunk)


def _shots(name, n, order, timeint, nt, shots, pml=0, chunk=0, compensated=True, energy=False, own_material=False,
           nrec_side=4):
    nx, ny, nz = n
    return dict(name=name, kind="shots", nx=nx, ny=ny, nz=nz, order=order, timeint=timeint, nt=nt, shots=shots, pml=pml,
                chunk=chunk, compensated=compensated, energy=energy, own_material=own_material, nrec_side=nrec_side)


def _mlp(name, what, hidden, depth, inputs, outputs, rows, steps=0):
    return dict(name=name, kind="mlp", what=what, hidden=hidden, depth=depth, inputs=inputs, outputs=outputs, rows=rows,
                steps=steps)


def listed():
    return [
        # a first small model, and what every unit test and the smoke run do: 162 tets, launch-bound
        _solo("fp64_cube162_n3", (3, 3, 3), 3, 2, 60),
        # the plain homogeneous brick with the low-storage RK4, all of its 1,000 steps
        _solo("fp64_brick3072_n3_rk4", (8, 8, 8), 3, 4, 1000),
        # a ragged box of the highest order, anelastic with PML, third-order Runge-Kutta
        _solo("fp64_box6006_n5_rk3", (13, 11, 7), 5, 3, 60, pml=2),
        # the two-layer anelastic box with NPML at its full size, continued from a wavefield
        _solo("fp64_box192000_n4", (40, 40, 20), 4, 2, 240, pml=10, chunk=8),
        # the same physics as eight shots at once in FP32 with the compensated sum and the energy of every step
        _shots("fp32_box41472_n4_8shots", (24, 24, 12), 4, 2, 320, 8, pml=6, chunk=16, energy=True),
        # a small anelastic box whose waves reach the PML: whole runs of a few shots, plain sum
        _shots("fp32_box3000_n4_4shots", (10, 10, 5), 4, 2, 300, 4, pml=2, compensated=False),
        # low order, where bytes count most; with the energy the PML trigger needs
        _shots("fp32_box24000_n2_6shots", (20, 20, 10), 2, 2, 1200, 6, pml=5, chunk=60, energy=True),
        # the multi-shot workload: 64 shots with perturbed velocities on the brick
        _shots("fp32_brick3072_n3_64shots", (8, 8, 8), 3, 2, 1920, 64, chunk=120, own_material=True,
               nrec_side=2),
        # uneven instances of orders 2 to 5 packed by order
        dict(name="fp32_uneven8", kind="uneven", count=8, n_lo=10, n_hi=15, mesh_seed=4000, nt=1200, chunk=60),
        # an epoch of the surrogate: 9 source parameters to 16 receivers x 3 components x 512 samples
        _mlp("mlp_train_surrogate", "train", 512, 4, 9, 24576, 256, steps=128),
        # its inference on 256 queries
        _mlp("mlp_forward_surrogate", "forward", 512, 4, 9, 24576, 256),
        # a small network's loss and gradients: launches count
        _mlp("mlp_gradients_small", "gradients", 128, 3, 9, 192, 128),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["solo", "solo", "shots", "shots", "shots", "uneven", "mlp", "mlp"])
    if kind == "solo":
        order, pml = rng.randint(2, 5), rng.choice([0, 0, 1, 2])
        n = (log_int(3 + 2 * pml, 14), log_int(3 + 2 * pml, 14), log_int(3 + pml, 9))
        c = _solo("", n, order, rng.choice([2, 2, 3, 4]), rng.randint(40, 160), pml=pml)
    elif kind == "shots":
        order, pml = rng.randint(2, 5), rng.choice([0, 1, 2])
        n = (log_int(3 + 2 * pml, 13), log_int(3 + 2 * pml, 13), log_int(3 + pml, 8))
        nodes = 6 * n[0] * n[1] * n[2] * ORDERS_POINTS[order]
        shots = max(1, min(log_int(1, 64), 600000 // nodes))
        c = _shots("", n, order, rng.choice([2, 2, 3]), rng.randint(60, 200), shots, pml=pml,
                   compensated=rng.random() < 0.6, energy=pml > 0 and rng.random() < 0.6,
                   own_material=pml == 0 and rng.random() < 0.5, nrec_side=rng.randint(1, 4))
    elif kind == "uneven":
        lo = rng.randint(6, 11)
        c = dict(name="", kind="uneven", count=rng.randint(2, 6), n_lo=lo, n_hi=lo + rng.randint(0, 3),
                 mesh_seed=rng.randint(1, 9999), nt=1800, chunk=rng.randint(40, 60))
    else:
        what = rng.choice(["train", "forward", "gradients"])
        c = _mlp("", what, log_int(48, 512), rng.randint(1, 4), rng.randint(4, 80),
                 64 * log_int(1, 256) if what != "forward" else log_int(40, 16384), 64 * rng.randint(1, 4),
                 steps=rng.randint(4, 32) if what == "train" else 0)
    c.pop("name")
    return c


# ---------------------------------------------------------------------------
# set-up
# ---------------------------------------------------------------------------
HSIZE = 500.0


@functools.lru_cache(maxsize=None)
def _box(nx, ny, nz, order, timeint, nt, pml, nrec_side):
    """The mesh with its geometry, materials and receivers.  With PML the
    two-layer anelastic box, without it the homogeneous elastic brick."""
    if pml:
        return problem.layered_box(nx, ny, nz, order=order, nt=nt, hsize=HSIZE, pml_cells=pml, nrec_side=nrec_side,
                                   timeint=timeint, full_source_arrays=False)
    ext = (nx * HSIZE * 2.5, ny * HSIZE * 2.5, nz * HSIZE * 2.5)
    m = meshmod.brick_mesh(nx, ny, nz, ext, material=lambda x, y, z: (4000.0, 2310.0, 2700.0, 9000.0, 9000.0))
    gx, gy = (np.linspace(e / (2 * nrec_side), e - e / (2 * nrec_side), nrec_side) for e in ext[:2])
    src = srcmod.Source(xyz=(ext[0] / 2, ext[1] / 2, ext[2] / 2), kind=1, stf=2, f0=1.0)
    return problem.setup(m, order, dict(timeint=timeint, nt=nt, cfl=0.25), [src], [(x, y, ext[2]) for y in gy for x in gx],
                         name="brick", full_source_arrays=False)


def _base(case):
    return _box(case["nx"], case["ny"], case["nz"], case["order"], case["timeint"], case["nt"], case["pml"],
                case.get("nrec_side", 3))


def _source(base, rng, force):
    """A shallow event below the receivers: a moment tensor, or a point force."""
    g = base.geom
    x, y, z = base.rec_xyz[rng.integers(base.rec_xyz.shape[0])]
    h = HSIZE * (1.0 if base.set_pml else 2.5)
    xyz = (float(np.clip(x + rng.uniform(-0.45, 0.45) * h, g.bounds[0] + 1.0, g.bounds[1] - 1.0)),
           float(np.clip(y + rng.uniform(-0.45, 0.45) * h, g.bounds[2] + 1.0, g.bounds[3] - 1.0)),
           float(z - rng.uniform(0.3, 1.2) * h))
    f0 = 2.0 if base.set_pml else 1.0
    if force:
        return srcmod.Source(xyz=xyz, kind=0, stf=2, f0=f0, factor=1e10, angle_force=tuple(rng.standard_normal(3)))
    return srcmod.Source(xyz=xyz, kind=1, stf=1 if base.set_pml else 2, f0=f0, factor=1.0,
                         M=batch.random_moment_tensor(rng))


def _solo_arrays(case, seed):
    base = _base(case)
    rng = np.random.default_rng(seed)
    src = _source(base, rng, force=not case["pml"])
    loc = srcmod.locate([src.xyz], base.mesh, base.geom, base.order)
    ops = srcmod.prepare_sources([src], loc, base.geom, base.mat, base.order, base.nt, base.dt, True)
    a = layout.reference_arrays(dataclasses.replace(base, sources=[src], src=ops))
    q0 = None
    if case["chunk"]:
        # a wavefield under way: stresses of some 10 kPa, velocities of some cm/s
        g = torch.Generator(device=DEV)
        g.manual_seed(int(seed))
        q0 = torch.randn((9, a["nelem"] * a["np"]), generator=g, device=DEV, dtype=torch.float64)
        q0[:6] *= 1e4
        q0[6:] *= 1e-2
    return a, q0


def _shot_batch(case, seed):
    base = _base(case)
    shots, cen = [], base.mesh.coord[base.mesh.elem].mean(axis=1)
    for k in range(case["shots"]):
        rng = np.random.default_rng([int(seed), k])
        src = _source(base, rng, force=False)
        loc = srcmod.locate([src.xyz], base.mesh, base.geom, base.order)
        mat = base.mat
        if case["own_material"]:
            f = 1 + np.clip(0.025 * batch.correlated_field(cen, 1000.0, rng), -0.05, 0.05)
            mat = problem.physics.materials(base.mesh.vp * f, base.mesh.vs * f, base.mesh.rho.copy(), base.mesh.qp,
                                            base.mesh.qs, base.attenuation, base.par["f0_att"], base.par["fr_att"])
        shots.append(dataclasses.replace(base, mat=mat, sources=[src], src=None, extra={"loc": loc}))
    return batch.finish_shots(base, shots, shared=not case["own_material"])


@functools.lru_cache(maxsize=None)
def _instance_meshes(count, n_lo, n_hi, mesh_seed, nt):
    """Layered elastic cubes of random size and order, with receivers in a
    borehole array around the middle."""
    out = []
    for k in range(count):
        rng = np.random.default_rng([mesh_seed, k])
        n, order = int(rng.integers(n_lo, n_hi + 1)), int(2 + (k + mesh_seed) % 4)
        ext = n * HSIZE
        tops = np.sort(rng.uniform(0.1, 0.9, int(rng.integers(1, 4))))[::-1] * ext
        vps = rng.uniform(2500.0, 6500.0, tops.size + 1)

        def material(x, y, z, tops=tops, vps=vps):
            vp = vps[(z[:, None] < tops[None, :]).sum(axis=1)]
            return vp, vp / math.sqrt(3.0), np.full_like(vp, 2700.0), np.full_like(vp, 9000.0), np.full_like(vp, 9000.0)

        m = meshmod.brick_mesh(n, n, n, (ext,) * 3, material=material)
        src = srcmod.Source(xyz=(0.5 * ext,) * 3, kind=0, stf=2, f0=1.0)
        recs = [(0.5 * ext + 40.0, 0.5 * ext + 60.0, 0.5 * ext + (i - 3.5) * 120.0) for i in range(8)]
        out.append(problem.setup(m, order, dict(timeint=2, nt=nt, cfl=0.25), [src], recs, full_source_arrays=False))
    return out


def _instances(case, seed):
    out = []
    for k, base in enumerate(_instance_meshes(case["count"], case["n_lo"], case["n_hi"], case["mesh_seed"], case["nt"])):
        rng = np.random.default_rng([int(seed), k])
        ext = base.geom.bounds[1]
        src = srcmod.Source(xyz=tuple(float(v) for v in 0.5 * ext + rng.uniform(-400.0, 400.0, 3)), kind=0, stf=2,
                            f0=5.0, factor=1e10, angle_force=tuple(rng.standard_normal(3)))
        loc = srcmod.locate([src.xyz], base.mesh, base.geom, base.order)
        ops = srcmod.prepare_sources([src], loc, base.geom, base.mat, base.order, base.nt, base.dt, False)
        p = dataclasses.replace(base, sources=[src], src=ops)
        out.append(batch.ShotBatch(p, [p], True))
    return out


def _widths(case):
    return [case["inputs"]] + [case["hidden"]] * case["depth"] + [case["outputs"]]


def _mlp_data(case, seed):
    """Weights, standardised inputs and unit-RMS targets smooth in them."""
    rng = np.random.default_rng(seed)
    w = _widths(case)
    params = [(a, (0.05 * rng.standard_normal(b.size)).astype(np.float32)) for a, b in mlp.init_params(w, int(seed))]
    n = case["rows"] if case["what"] == "forward" else 4 * case["rows"]
    x = rng.standard_normal((n, w[0]), dtype=np.float32)
    t = idx = None
    if case["what"] != "forward":
        a = rng.standard_normal((w[0], 24), dtype=np.float32) / math.sqrt(w[0])
        t = (np.sin(2.0 * (x @ a)) @ rng.standard_normal((24, w[-1]), dtype=np.float32)) * math.sqrt(2.0 / 24)
        steps = max(1, case["steps"])
        idx = np.concatenate([rng.permutation(n) for _ in range(steps // 4 + 1)])[:steps * case["rows"]].astype(np.int32)
    return params, x, t, idx


def prepare(case, seed):
    kind, s = case["kind"], {"case": case, "step": 0}
    if kind == "solo":
        a, q0 = _solo_arrays(case, seed)
        s["ctx"] = capi.Context(a, energy=bool(case["pml"]))
        if q0 is not None:
            s["q0"] = q0.cpu().numpy()
            s["ctx"].set_state(0, q=s["q0"])
    elif kind == "shots":
        s["ctx"] = capi.BatchContext(_shot_batch(case, seed), precision=capi.NEXD_FP32, compensated=case["compensated"],
                                     energy=case["energy"])
        s["ctx"].reset()
    elif kind == "uneven":
        s["members"] = [uneven.PackedBatch(p, autotune=False) for p in uneven.pack(_instances(case, seed))]
        s["group"] = _group(s["members"])
    else:
        params, s["x"], t, s["idx"] = _mlp_data(case, seed)
        s["net"] = mlp.MLP(_widths(case), max_batch=case["rows"])
        s["net"].set_params(params)
        s["params"] = params
        if t is not None:
            s["net"].upload_dataset(s["x"], t)
    return s


def _group(members):
    for m in members:
        m.reset()
    return capi.Group(members)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _f32(a):
    """FP32 batches compute in FP32; their getters widen to double."""
    return a.astype(np.float32)


def run(state):
    case = state["case"]
    return {"solo": _run_solo, "shots": _run_shots, "uneven": _run_uneven, "mlp": _run_mlp}[case["kind"]](state, case)


def _next(state, case, rewind):
    """First and last step of this pass; a chunked run starts over at its end."""
    if not case["chunk"] or state["step"] + case["chunk"] > case["nt"]:
        if state["step"] or not case["chunk"]:
            rewind()
        state["step"] = 0
    first = state["step"] + 1
    state["step"] += case["chunk"] or case["nt"]
    return first, state["step"]


def _run_solo(state, case):
    ctx = state["ctx"]
    first, last = _next(state, case, (lambda: ctx.set_state(0, q=state["q0"])) if case["chunk"] else ctx.reset)
    energy = ctx.run(first, last, want_energy=bool(case["pml"]))
    out = {"seismograms": ctx.seismograms()}
    if energy is not None:
        out["energy"] = energy
    return out


def _run_shots(state, case):
    ctx = state["ctx"]
    ctx.run(*_next(state, case, ctx.reset))
    out = {"seismograms": _f32(np.stack([ctx.seismograms(k) for k in range(case["shots"])]))}
    if case["energy"]:
        out["energy"] = _f32(np.stack([ctx.energy(k) for k in range(case["shots"])]) * ENERGY_UNIT)
    return out


# the energies as the reference defines them reach 1e54; this unit brings an
# FP32 run's into the range of the type that it is computed in
ENERGY_UNIT = 1e-50


def _run_uneven(state, case):
    def rewind():
        state["group"].close()
        state["group"] = _group(state["members"])

    first, last = _next(state, case, rewind)
    state["group"].run(first, last)
    return [_f32(s) for m in state["members"] for s in m.seismograms()]


def _run_mlp(state, case):
    net = state["net"]
    if case["what"] == "forward":
        return net.forward(state["x"])
    if case["what"] == "gradients":
        loss = net.gradients(state["idx"])
        return [np.float32(loss), *(v for p in net.grads() for v in p)]
    losses = net.train(state["idx"], case["rows"], lr=LR)
    return [losses, *(v for p in net.params() for v in p)]


LR = 2e-4


# ---------------------------------------------------------------------------
# the least work of one pass
# ---------------------------------------------------------------------------
STAGES = {1: 1, 2: 2, 3: 3, 4: 5}


def _loop_work(nelem, order, timeint, steps, size, att, pml_share, shots, own_material, compensated):
    """Per step and node: the field is read and written at every stage (its
    neighbours read it) and its step-start value once more at the later ones;
    memory variables and PML auxiliaries are read and written once; per stage
    the affine metric, the face frames, the connectivity and the material of
    each element, and the nine PML coefficients of each PML node."""
    np_, npf = ORDERS_POINTS[order], (order + 1) * (order + 2) // 2
    st = STAGES[timeint]
    fields = 9 * (2 if compensated else 1)
    per_node = fields * (3 * st - 1) + (36 if att else 0) + 54 * pml_share
    static = 54 * size + 48
    state = nelem * np_ * size * per_node * shots
    coef = st * nelem * (static * (shots if own_material else 1) + 9 * pml_share * np_ * size)
    cols = 15 if att else 9
    flops = st * nelem * shots * (3 * 2 * np_ * np_ * cols + 2 * np_ * 4 * npf * cols + 4 * npf * 200)
    return steps * (state + coef), steps * flops


def work(case):
    if case["kind"] == "mlp":
        w, rows, steps = _widths(case), case["rows"], max(1, case["steps"])
        mac = sum(a * b for a, b in zip(w[:-1], w[1:]))
        n = mac + sum(w[1:])
        if case["what"] == "forward":
            return {"bytes": 4 * n + 4 * rows * (w[0] + w[-1]), "flops": 2 * rows * mac}
        last = 3 * 2 * rows * mac - 2 * rows * w[0] * w[1]
        if case["what"] == "gradients":
            return {"bytes": 8 * n + 4 * rows * (w[0] + w[-1]), "flops": last}
        # weights and both moments read and written, the batch's rows read
        return {"bytes": steps * (24 * n + 4 * rows * (w[0] + w[-1])), "flops": steps * last}
    if case["kind"] == "uneven":
        b = f = 0
        for p in _instance_meshes(case["count"], case["n_lo"], case["n_hi"], case["mesh_seed"], case["nt"]):
            x, y = _loop_work(p.nelem, p.order, 2, case["chunk"], 4, False, 0.0, 1, False, False)
            b, f = b + x, f + y
        return {"bytes": b, "flops": f}
    nx, ny, nz, p = case["nx"], case["ny"], case["nz"], case["pml"]
    nelem = 6 * nx * ny * nz
    inner = 6 * max(0, nx - 2 * p) * max(0, ny - 2 * p) * max(0, nz - p)
    solo = case["kind"] == "solo"
    b, f = _loop_work(nelem, case["order"], case["timeint"], case["chunk"] or case["nt"], 8 if solo else 4, p > 0,
                      1.0 - inner / nelem if p else 0.0, 1 if solo else case["shots"],
                      not solo and case["own_material"], not solo and case["compensated"])
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _rotation(a, b, c):
    """Stress (xx yy zz xy yz xz) and velocity rows of the 9x9 rotation built
    from the frame vectors a, b, c (..., 3), velocities by the same vectors."""
    z = torch.zeros_like(a[..., 0])
    rows = [[a[..., r] ** 2, b[..., r] ** 2, c[..., r] ** 2, 2 * a[..., r] * b[..., r], 2 * b[..., r] * c[..., r],
             2 * a[..., r] * c[..., r], z, z, z] for r in range(3)]
    for i, k in ((1, 0), (2, 1), (2, 0)):
        rows.append([a[..., i] * a[..., k], b[..., i] * b[..., k], c[..., i] * c[..., k],
                     a[..., i] * b[..., k] + a[..., k] * b[..., i], b[..., i] * c[..., k] + b[..., k] * c[..., i],
                     a[..., i] * c[..., k] + a[..., k] * c[..., i], z, z, z])
    for r in range(3):
        rows.append([z] * 6 + [a[..., r], b[..., r], c[..., r]])
    return torch.stack([torch.stack(r, -1) for r in rows], -2)


class _Loop:
    """The time loop of the discontinuous Galerkin scheme on torch tensors
    [shot][field][element][node]: volume derivatives of the (PML-modified)
    fluxes, the upwind flux through LIFT, memory variables, sources, TVD
    Runge-Kutta or the low-storage RK4."""

    def __init__(self, a, mats, srcs, dt):
        """a: the mesh's arrays; mats: the arrays that hold each shot's
        materials (one: shared); srcs: per shot (element, type, spatial [.., 6,
        Np], stf [.., nt]); dt: the step."""
        t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=DEV)  # noqa: E731
        e, n, npf = a["nelem"], a["np"], a["npf"]
        self.a, self.e, self.n, self.dt, self.shots = a, e, n, dt, len(srcs)
        # D^T of all three operators side by side, so x @ D3 gives the r, s, t derivatives
        self.d3 = t(np.concatenate([np.asarray(a[k]).reshape(n, n) for k in ("dr", "ds", "dt_")], axis=1))
        self.lift = t(np.asarray(a["lift"]).reshape(4 * npf, n))
        self.mass = t(np.asarray(a["mass"]).reshape(n, n))
        self.met = [[t(a[o + x]).view(e, n) for o in "rst"] for x in "xyz"]
        self.fscale = t(a["fscale"]).view(e, 4 * npf)
        self.ibt, self.ibn = t(a["ibt"]).view(-1).long() - 1, t(a["ibn"]).view(-1).long() - 1
        inner = t(a["neighbor"]).view(e, 4) > 0
        self.inner = inner.repeat_interleave(npf, 1).reshape(-1)
        face = t(a["face"]).view(e, 4)
        self.att, self.pml = bool(a["attenuation"]), bool(a["pml"])
        frames = [t(a[k]).view(e, 4, 3) for k in ("nnormal", "stangential", "ttangential")]
        rot = _rotation(*frames)
        back = _rotation(*torch.stack(frames, -2).unbind(-1))
        free = torch.diag(torch.tensor([-2.0, 0, 0, -2, 0, -2, 0, 0, 0], device=DEV, dtype=torch.float64))
        eye = torch.eye(9, device=DEV, dtype=torch.float64)
        is_free = (~inner & (face == -1))[..., None, None]
        # outer faces: dq is the own trace, absorbing ones change the sign
        side = torch.where(is_free, free, torch.where((~inner & (face == -2))[..., None, None], -eye, eye))
        self.flux, self.aflux, self.mat = [], [], []
        for m in mats:
            vp, vs, rho, lam, mu = (t(m[k]) for k in ("vpu", "vsu", "rho", "lambdau", "muu"))
            j = torch.zeros((e, 9, 9), device=DEV, dtype=torch.float64)
            l2m = lam + 2 * mu
            j[:, 0, 0], j[:, 0, 6] = vp, -l2m
            for r in (1, 2):
                j[:, r, 0], j[:, r, 6] = lam * vp / l2m, -lam
            j[:, 3, 3], j[:, 3, 7], j[:, 5, 5], j[:, 5, 8] = vs, -mu, vs, -mu
            for r, c, v in ((6, 0, vp), (7, 3, vs), (8, 5, vs)):
                j[:, r, c], j[:, r, r] = -1 / rho, v
            self.flux.append((rot @ j[:, None] @ side @ back).contiguous())
            if self.att:
                k = torch.zeros((e, 9, 9), device=DEV, dtype=torch.float64)
                k[:, 0, 0], k[:, 0, 6] = 1 / (vp * rho), -1.0
                for r, c in ((3, 7), (5, 8)):
                    k[:, r, r], k[:, r, c] = 1 / (2 * vs * rho), -0.5
                self.aflux.append((rot @ k[:, None] @ side @ back)[..., :6, :].contiguous())
            an = t(m["anelasticvar"]).view(e, -1, 3) if self.att else None
            self.mat.append((-l2m[:, None], -lam[:, None], -mu[:, None], (-1 / rho)[:, None], an))
        self.rho, self.lam_r, self.mu_r = ([t(m[k])[:, None] for m in mats] for k in ("rho", "lambda", "mu"))
        self.srcs = [(np.asarray(s[0]), np.asarray(s[1]), t(s[2]), t(s[3])) for s in srcs]
        if self.pml:
            self.in_pml = (t(a["pmlcheck"]).view(e) != 0)[:, None]
            p = {k: t(a[k]).view(e, n) for k in ("ddx", "ddy", "ddz", "alphax", "alphay", "alphaz", "kx", "ky", "kz")}
            self.alpha = [p["alpha" + x] for x in "xyz"]
            self.dk = [p["dd" + x] / p["k" + x] for x in "xyz"]
            self.k = [p["k" + x] for x in "xyz"]

    def rhs(self, q, th, aux, it, s):
        """Time derivatives of shot s's fields q [9], memory variables th [3][6]
        and PML auxiliaries aux [3][9]."""
        e, n = self.e, self.n
        e0, e1, e2, e3, an = self.mat[s if len(self.mat) > 1 else 0]
        fl = self.flux[s if len(self.flux) > 1 else 0]
        z = torch.zeros_like(q[0])
        f = [torch.stack([e0 * q[6], e1 * q[6], e1 * q[6], e2 * q[7], z, e2 * q[8], e3 * q[0], e3 * q[3], e3 * q[5]]),
             torch.stack([e1 * q[7], e0 * q[7], e1 * q[7], e2 * q[6], e2 * q[8], z, e3 * q[3], e3 * q[1], e3 * q[4]]),
             torch.stack([e1 * q[8], e1 * q[8], e0 * q[8], z, e2 * q[7], e2 * q[6], e3 * q[5], e3 * q[4], e3 * q[2]])]
        daux = None
        if self.pml:
            f = [torch.where(self.in_pml, (aux[d] + f[d]) / self.k[d], f[d]) for d in range(3)]
            # every node takes the last element's fluxes, as the reference does
            daux = torch.stack([-self.alpha[d] * aux[d] - self.dk[d] * (aux[d] + f[d][:, -1:, :]) for d in range(3)])
            daux = torch.where(self.in_pml, daux, torch.zeros_like(daux))
        out = torch.zeros_like(q)
        for d in range(3):
            g = f[d] @ self.d3
            for o in range(3):
                out += self.met[d][o] * g[..., o * n:(o + 1) * n]
        flat = q.reshape(9, -1)
        own = flat[:, self.ibt]
        dq = torch.where(self.inner, flat[:, self.ibn.clamp(min=0)] - own, own).view(9, e, 4, -1)
        jump = dq.permute(1, 2, 0, 3).contiguous()                        # [e][face][9][npf]
        scale = 0.5 * self.fscale.view(e, 4, 1, -1)
        lifted = (scale * (fl @ jump)).permute(2, 0, 1, 3).reshape(9, e, -1) @ self.lift
        dth = None
        if self.att:
            af = self.aflux[s if len(self.aflux) > 1 else 0]
            alift = (scale * (af @ jump)).permute(2, 0, 1, 3).reshape(6, e, -1) @ self.lift
            gv = q[6:] @ self.d3
            dv = [[sum(self.met[x][o] * gv[c][..., o * n:(o + 1) * n] for o in range(3)) for x in range(3)] for c in range(3)]
            ex, ey, ez = dv[0][0], dv[1][1], dv[2][2]
            strain = torch.stack([ex, ey, ez, 0.5 * (dv[1][0] + dv[0][1]), 0.5 * (dv[2][1] + dv[1][2]),
                                  0.5 * (dv[2][0] + dv[0][2])])
            wl = self.a["wl"]
            dth = torch.stack([float(wl[i]) * (alift - strain - th[i]) for i in range(3)])
            for i in range(3):
                a1, a2, a3 = (an[:, i, c][:, None] for c in range(3))
                x, y, zz = th[i][0], th[i][1], th[i][2]
                out[0] += a3 * x + a1 * (y + zz)
                out[1] += a3 * y + a1 * (zz + x)
                out[2] += a3 * zz + a1 * (x + y)
                out[3:6] += a2 * th[i][3:6]
        out += lifted
        el, ty, spatial, stf = self.srcs[s]
        for i in range(len(el)):
            if ty[i] == 0:
                out[6:9, el[i]] += spatial[i, :3] * stf[i, it]
            else:
                out[0:6, el[i]] += spatial[i] * stf[i, it]
        return [out, dth, daux]

    def run(self, nt, steps, q0=None):
        """Seismograms [shot][nrec][9][nt] and energies [shot][steps]."""
        a, e, n = self.a, self.e, self.n
        tiny = float(np.float32(1e-24))
        rec = torch.as_tensor(np.asarray(a["recelem"]).astype(np.int64) - 1, device=DEV)
        wt = torch.as_tensor(np.ascontiguousarray(a["rec_int"]), device=DEV).view(-1, n)
        seis = torch.zeros((self.shots, rec.numel(), 9, nt), device=DEV, dtype=torch.float64)
        energy = torch.zeros((self.shots, steps), device=DEV, dtype=torch.float64)
        third, two_thirds = float(np.float32(1) / np.float32(3)), float(np.float32(2) / np.float32(3))
        for s in range(self.shots):
            mk = lambda *d: torch.full((*d, e, n), tiny, device=DEV, dtype=torch.float64)  # noqa: E731
            y = [mk(9) if q0 is None else q0.reshape(9, e, n).clone(), mk(3, 6) if self.att else None,
                 torch.zeros((3, 9, e, n), device=DEV, dtype=torch.float64) if self.pml else None]
            u, acc = [torch.full((3, rec.numel(), n), tiny, device=DEV, dtype=torch.float64) for _ in range(2)]

            def record(row):
                for c, v in enumerate((u, y[0][6:, rec], acc)):
                    seis[s, :, 3 * c:3 * c + 3, row] = (v * wt).sum(-1).T

            record(0)
            for it in range(steps):
                y, last = self._step(y, it, s, third, two_thirds)
                u += self.dt * y[0][6:, rec]
                acc = last[6:, rec]
                if it + 1 < nt:
                    record(it + 1)
                if self.pml:
                    energy[s, it] = self._energy(y[0], s)
        return seis, energy

    def _step(self, y, it, s, third, two_thirds):
        ti, dt = self.a["timeint"], self.dt
        k = range(3)
        add = lambda v, r: [None if v[i] is None else v[i] + dt * r[i] for i in k]  # noqa: E731
        mix = lambda c, b, d, v: [None if v[i] is None else c * b[i] + d * v[i] for i in k]  # noqa: E731
        if ti == 4:
            ca = [0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
                  -1275806237668 / 842570457699]
            cb = [1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
                  3134564353537 / 4481467310338, 2277821191437 / 14882151754819]
            res = [None if v is None else torch.zeros_like(v) for v in y]
            for x, z in zip(ca, cb):
                r = self.rhs(*y, it, s)
                res = [None if y[i] is None else x * res[i] + dt * r[i] for i in k]
                y = [None if y[i] is None else y[i] + z * res[i] for i in k]
            return y, r[0]
        base = y
        r = self.rhs(*y, it, s)
        y = add(y, r)
        if ti == 2:
            r = self.rhs(*y, it, s)
            y = mix(0.5, base, 0.5, add(y, r))
        elif ti == 3:
            r = self.rhs(*y, it, s)
            y = mix(0.75, base, 0.25, add(y, r))
            r = self.rhs(*y, it, s)
            y = mix(third, base, two_thirds, add(y, r))
        return y, r[0]

    def _energy(self, q, s):
        """The energy as the reference forms it: its normal "strains" are
        stress combinations times 4 mu^2 + 6 mu lambda, the third with q1
        twice."""
        k = s if len(self.rho) > 1 else 0
        rho, lam, mu = self.rho[k], self.lam_r[k], self.mu_r[k]
        c = 4 * mu * mu + 6 * mu * lam
        y = torch.stack([c * (2 * (lam + mu) * q[0] - lam * (q[1] + q[2])), c * (2 * (lam + mu) * q[1] - lam * (q[0] + q[2])),
                         c * (2 * (lam + mu) * q[2] - lam * (q[0] + q[0])), 2 * q[3] / (2 * mu), 2 * q[4] / (2 * mu),
                         2 * q[5] / (2 * mu), rho * q[6], rho * q[7], rho * q[8]])
        j = torch.as_tensor(np.ascontiguousarray(self.a["jac"]), device=DEV).view(self.e, self.n)[:, 0]
        return ((q * (y @ self.mass)).sum((0, 2)) * 0.5 * j).sum()


def _operands(s):
    return s.src.srcelem, s.src.srctype, s.src.spatial, s.src.stf


def _exact_solo(case, seed):
    a, q0 = _solo_arrays(case, seed)
    src = (np.asarray(a["srcelem"]) - 1, a["srctype"], a["src_spatial"], a["src_stf"])
    seis, energy = _Loop(a, [a], [src], a["dt"]).run(case["nt"], case["chunk"] or case["nt"], q0)
    out = {"seismograms": seis[0].cpu().numpy()}
    if case["pml"]:
        out["energy"] = energy[0].cpu().numpy()
    return out


def _exact_shots(case, seed):
    sb = _shot_batch(case, seed)
    a = layout.reference_arrays(sb.base)
    mats = [layout.reference_arrays(s) for s in (sb.shots if case["own_material"] else sb.shots[:1])]
    steps = case["chunk"] or case["nt"]
    seis, energy = _Loop(a, mats, [_operands(s) for s in sb.shots], sb.base.dt).run(case["nt"], steps)
    out = {"seismograms": seis.cpu().numpy()}
    if case["energy"]:
        out["energy"] = np.zeros((case["shots"], case["nt"]))
        out["energy"][:, :steps] = energy.cpu().numpy() * ENERGY_UNIT
    return out


def _exact_uneven(case, seed):
    inst, got = _instances(case, seed), {}
    for k, sb in enumerate(inst):
        a = layout.reference_arrays(sb.base)
        got[k] = _Loop(a, [a], [_operands(sb.base)], sb.base.dt).run(case["nt"], case["chunk"])[0][0].cpu().numpy()
    return [got[k] for k in sorted(got, key=lambda k: (inst[k].base.order, k))]   # packed by order


def _exact_mlp(case, seed):
    params, x, t, idx = _mlp_data(case, seed)
    p = [torch.tensor(v, device=DEV, dtype=torch.float64, requires_grad=True) for q in params for v in q]
    x = torch.tensor(x, device=DEV, dtype=torch.float64)

    def net(h):
        for l in range(len(p) // 2):
            h = h @ p[2 * l].T + p[2 * l + 1]
            if l + 1 < len(p) // 2:
                h = 0.5 * h * (1 + torch.erf(h / math.sqrt(2.0)))
        return h

    if case["what"] == "forward":
        return net(x).detach().cpu().numpy()
    t = torch.tensor(t, device=DEV, dtype=torch.float64)
    rows = torch.tensor(idx, device=DEV, dtype=torch.int64)
    if case["what"] == "gradients":
        loss = ((net(x[rows]) - t[rows]) ** 2).mean()
        return [float(loss.detach()), *(g.cpu().numpy() for g in torch.autograd.grad(loss, p))]
    losses, m, v = [], [torch.zeros_like(w) for w in p], [torch.zeros_like(w) for w in p]
    for s in range(case["steps"]):
        r = rows[s * case["rows"]:(s + 1) * case["rows"]]
        loss = ((net(x[r]) - t[r]) ** 2).mean()
        grads = torch.autograd.grad(loss, p)
        losses.append(float(loss.detach()))
        with torch.no_grad():
            for i, g in enumerate(grads):
                m[i] = 0.9 * m[i] + 0.1 * g
                v[i] = 0.999 * v[i] + 0.001 * g * g
                p[i] -= LR * (m[i] / (1 - 0.9 ** (s + 1))) / (torch.sqrt(v[i] / (1 - 0.999 ** (s + 1))) + 1e-8)
    return [np.array(losses), *(w.detach().cpu().numpy() for w in p)]


def exact(case, seed):
    return {"solo": _exact_solo, "shots": _exact_shots, "uneven": _exact_uneven, "mlp": _exact_mlp}[case["kind"]](case, seed)
