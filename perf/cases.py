"""Performance cases of the simulation step, its projection solve, its adjoint and its renderer.

Every case goes through the entry points a program calls (`dcgrid_amd.Simulation`,
`dcgrid_amd.autograd.rollout`). Kinds of work, by the case's "kind":

  uniform   one or more steps of the dense grid from a given state: set the state (device
            pointers), step, read the state back, as a control or learning loop does
  control   the differentiable rollout of the dense grid, forward and backward (torch autograd)
  dcgrid    a run of an adaptive scene from its start, as a parameter study repeats it: reset,
            seed, steps with topology adaptation, then the fields read back
  frame     the same on 16-bit field storage, then the rendered image (what such a program shows)
  solve     the projection solved to 1e-8 on an adapted (or fully dense) grid
  terrain   steps of the dense moist terrain scene, then the fields read back
  adjoint   the differentiable rollout of the adaptive grid on its frozen topology

The scenes are those of `dcgrid_amd.scenes` (configurations 0 to 4 and the reference's default
scene) at their own sizes and at others; seeds change the initial velocity, the source's noise and
the input fields.
"""
import math

import torch

import dcgrid_amd
from dcgrid_amd import autograd, scenes
from dcgrid_amd._abi import (PROJECT_LOCAL, PROJECT_MULTILEVEL, PROJECT_SOLVE, SOURCE_SPHERE_BUOYANT,
                             STORAGE_BF16, STORAGE_FP16, STORAGE_FP32)

STORAGE = {"fp32": STORAGE_FP32, "fp16": STORAGE_FP16, "bf16": STORAGE_BF16}


def listed():
    return [
        # configuration 0: the small dense plume, 100 Jacobi sweeps a step; launches and latency
        {"name": "uniform64_plume", "kind": "uniform", "gx": 64, "gy": 64, "gz": 64, "mode": "local", "pairs": 50,
         "scene": "plume", "steps": 2},
        # the smallest calls: one step of a small odd-sized domain with the inlet and a solid sphere
        {"name": "uniform_small_odd", "kind": "uniform", "gx": 45, "gy": 37, "gz": 29, "mode": "multilevel", "pairs": 2,
         "scene": "inlet", "steps": 1},
        # a dense grid beyond the caches, multilevel projection, buoyant source
        {"name": "uniform_large", "kind": "uniform", "gx": 320, "gy": 256, "gz": 384, "mode": "multilevel", "pairs": 2,
         "scene": "plume", "steps": 1},
        # configuration 3: differentiable density control, forward and backward
        {"name": "control128", "kind": "control", "gx": 128, "gy": 128, "gz": 128, "steps": 16, "every": 8},
        # configuration 1: the adaptive plume at its benchmark size, reference projection schedule
        {"name": "dcgrid256_plume", "kind": "dcgrid", "scene": "plume", "gx": 256, "gy": 256, "gz": 256, "bw": 8,
         "levels": 3, "budget": 4096, "steps": 20},
        # the reference's default scene: 4^3 blocks, all levels, inlet and solid sphere
        {"name": "dcgrid128_reference", "kind": "dcgrid", "scene": "reference", "gx": 128, "gy": 128, "gz": 128, "bw": 4,
         "levels": 0, "budget": 12000, "steps": 10},
        # configuration 2 as benchmarked: BF16 storage, every projection solved to 1e-8, then a frame
        {"name": "frame512_bf16_solve", "kind": "frame", "gx": 512, "gy": 512, "gz": 512, "levels": 4, "budget": 32768,
         "storage": "bf16", "solve": True, "steps": 8, "width": 256, "height": 256},
        # FP16 storage with the reference schedule, a frame of a mid-sized plume
        {"name": "frame256_fp16", "kind": "frame", "gx": 256, "gy": 256, "gz": 256, "levels": 3, "budget": 4096,
         "storage": "fp16", "solve": False, "steps": 20, "width": 320, "height": 200},
        # one projection of the adapted configuration 2 solved to 1e-8 (FP32 fields)
        {"name": "solve512_adaptive", "kind": "solve", "scene": "plume", "gx": 512, "gy": 512, "gz": 512, "levels": 4,
         "budget": 32768, "warm": 20},
        # one projection of a fully dense grid solved to 1e-8: every level covers the domain
        {"name": "solve256_dense", "kind": "solve", "scene": "dense", "gx": 256, "gy": 128, "gz": 256, "levels": 3,
         "budget": 0, "warm": 0},
        # configuration 4 at full size: the dense moist terrain scene (306.7 M cells), one step
        {"name": "terrain1024", "kind": "terrain", "gx": 1024, "gy": 256, "gz": 1024, "levels": 4, "warm": 1, "steps": 1},
        # differentiable rollout of the adaptive plume on its frozen topology, forward and backward
        {"name": "adjoint256", "kind": "adjoint", "gx": 256, "gy": 256, "gz": 256, "levels": 3, "budget": 4096,
         "warm": 40, "steps": 8, "every": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _block_box(rng, unit, lo, hi):
    """Three extents that are multiples of `unit` in [lo, hi], at most a factor 2 or so apart."""
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [min(hi, max(unit, unit * int(round(base * rng.uniform(0.7, 1.4) / unit)))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "control", "dcgrid", "dcgrid", "frame", "solve", "terrain", "adjoint"])
    if kind == "uniform":
        base = math.exp(rng.uniform(math.log(24), math.log(300)))
        gx, gy, gz = (max(16, int(base * rng.uniform(0.7, 1.4))) for _ in range(3))
        if rng.random() < 0.5:  # sizes that halve a few times (several levels)
            gx, gy, gz = (8 * max(2, v // 8) for v in (gx, gy, gz))
        mode = rng.choice(["local", "multilevel"])
        return {"kind": kind, "gx": gx, "gy": gy, "gz": gz, "mode": mode,
                "pairs": rng.choice([5, 20, 50]) if mode == "local" else 2, "scene": rng.choice(["plume", "inlet"]),
                "steps": rng.choice([1, 2])}
    if kind == "control":
        base = math.exp(rng.uniform(math.log(32), math.log(128)))
        gx, gy, gz = (max(20, int(base * rng.uniform(0.8, 1.2))) for _ in range(3))
        if rng.random() < 0.6:
            gx, gy, gz = (8 * max(3, v // 8) for v in (gx, gy, gz))
        steps = rng.randint(4, 16)
        return {"kind": kind, "gx": gx, "gy": gy, "gz": gz, "steps": steps, "every": rng.choice([1, 4, 8])}
    if kind == "dcgrid" and rng.random() < 0.4:
        gx, gy, gz = _block_box(rng, 32, 64, 160)
        return {"kind": kind, "scene": "reference", "gx": gx, "gy": gy, "gz": gz, "bw": 4, "levels": rng.choice([3, 4]),
                "budget": int(gx * gy * gz / 64 * rng.uniform(0.25, 0.5)), "steps": rng.choice([2, 5, 10])}
    if kind in ("dcgrid", "frame", "solve", "adjoint"):
        levels = rng.choice([3, 4])
        gx, gy, gz = _block_box(rng, 8 << (levels - 1), 96, 512)
        cells = gx * gy * gz
        # level 0's dense block count times a fraction, and room for the dense coarser levels
        budget = int(cells / 512 * rng.uniform(0.1, 0.2)) + 8
        case = {"kind": kind, "scene": "plume", "gx": gx, "gy": gy, "gz": gz, "bw": 8, "levels": levels, "budget": budget,
                "steps": rng.choice([2, 5, 10])}
        if kind == "frame":
            case.update(storage=rng.choice(["fp16", "bf16"]), solve=rng.random() < 0.5, width=_log_int(rng, 100, 320),
                        height=_log_int(rng, 80, 256))
        elif kind == "solve":
            case.pop("steps")
            case["warm"] = rng.choice([10, 30])
            if rng.random() < 0.4:
                case.update(scene="dense", budget=0, warm=0, levels=3)
                case["gx"], case["gy"], case["gz"] = _block_box(rng, 32, 64, 256)
        elif kind == "adjoint":
            case.update(warm=rng.choice([10, 30]), every=rng.choice([1, 2, 4]))
        return case
    levels = rng.choice([2, 3])
    gx, gz = (64 * rng.randint(2, 9) for _ in range(2))
    return {"kind": "terrain", "gx": gx, "gy": 32 * rng.randint(2, 5), "gz": gz, "levels": levels, "warm": 1,
            "steps": rng.choice([1, 2])}


# ---------------------------------------------------------------------------- scenes and inputs
def _box(case):
    return case["gx"], case["gy"], case["gz"]


def _smooth(shape, period, gen, channels=1):
    """Smooth random field on (z, y, x) cells: trilinear upsampling of a normal lattice."""
    d, h, w = shape
    lat = torch.randn(1, channels, max(2, d // period + 2), max(2, h // period + 2), max(2, w // period + 2),
                      generator=gen, device="cuda")
    f = torch.nn.functional.interpolate(lat, size=(d, h, w), mode="trilinear", align_corners=True)
    return f[0]


def _plume_params(case, seed, uniform=False):
    gx, gy, gz = _box(case)
    p = scenes.config(0 if uniform else (2 if max(_box(case)) > 256 else 1)).params.copy()
    p.gx, p.gy, p.gz = gx, gy, gz
    p.src_center[0], p.src_center[1], p.src_center[2] = gx / 2, gy / 8, gz / 2
    p.src_radius = min(gx, gy, gz) / 8
    p.seed = seed & 0x7FFFFFFF
    if not uniform:
        p.block_width = case.get("bw", 8)
        p.max_levels = case["levels"]
    return p


def _uniform_params(case, seed):
    if case["kind"] == "control":
        p = scenes.config(3).params.copy()
        p.gx, p.gy, p.gz = _box(case)
        p.seed = seed & 0x7FFFFFFF
        return p
    if case["scene"] == "plume":
        p = _plume_params(case, seed, uniform=True)
    else:  # the reference's defaults: inlet in the floor, solid sphere
        p = scenes.reference_params(*_box(case), kind="uniform")
        p.enable_additional_solids = 1
        p.dt = 0.5
        p.seed = seed & 0x7FFFFFFF
    if case["mode"] == "local":
        p.project_mode = PROJECT_LOCAL
        p.project_local_pairs = case["pairs"]
    else:
        p.project_mode = PROJECT_MULTILEVEL
        p.project_top_pairs, p.project_level_pairs = 2, 1
    return p


def _uniform_inputs(case, seed):
    """Density, velocity and temperature of a flow in progress, x-fastest cell order."""
    gx, gy, gz = _box(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    shape = (gz, gy, gx)
    n = gx * gy * gz
    p = _uniform_params(case, seed)
    speed = 0.4 / (p.dt * p.rdx)  # feet up to about a cell away
    vel = _smooth(shape, 12, gen, 3) * speed
    den = _smooth(shape, 16, gen).abs()
    tem = _smooth(shape, 16, gen).abs() * 0.5
    if case["kind"] == "control":
        vel = torch.randn((3,) + shape, generator=gen, device="cuda") * 0.1
    return den.reshape(n).contiguous(), vel.reshape(3, n).t().contiguous(), tem.reshape(n).contiguous()


def _terrain_params(case, seed):
    p = scenes.config(4).params.copy()
    gx, gy, gz = _box(case)
    if gx < 1024:  # the shorter lattice periods of a smaller domain
        p = scenes.terrain_scene(scenes.config(4, scale=2).params.copy(), 2)
    p.gx, p.gy, p.gz = gx, gy, gz
    p.max_levels = case["levels"]
    p.seed = seed & 0x7FFFFFFF
    return p


def _dense_budget(case, bw=8):
    gx, gy, gz = _box(case)
    return sum((gx // (bw << l)) * (gy // (bw << l)) * (gz // (bw << l)) for l in range(case["levels"]))


def _dcgrid(case, p, budget):
    """A DCGrid whose free blocks' cells hold zero in the fields and in the buffers they swap with;
    with "warm" seeded and stepped to an adapted topology."""
    sim = dcgrid_amd.Simulation("dcgrid", _box(case), p, budget)
    if p.storage == STORAGE_FP32:
        n = sim.field_size("density")
        zero = torch.zeros(3 * n, device="cuda")
        torch.cuda.synchronize()
        for first in (True, False):
            for f, c in (("density", 1), ("temperature", 1), ("velocity", 3)):
                sim.import_field_device(f, zero.data_ptr(), c * n)
            if first:
                sim.advect_velocity()
                sim.advect_density()
        sim.reset()
    if "warm" in case:
        sim.seed_scene()
        sim.step(case["warm"])
    sim.synchronize()
    return sim


def _export(sim, name, buf):
    sim.export_field_device(name, buf.data_ptr(), buf.numel())
    return buf


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("uniform", "control"):
        p = _uniform_params(case, seed)
        s["sim"] = dcgrid_amd.Simulation("uniform", _box(case), p)
        s["den"], s["vel"], s["tem"] = _uniform_inputs(case, seed)
        if kind == "control":
            gen = torch.Generator(device="cuda")
            gen.manual_seed(int(seed) + 1)
            target = _smooth((p.gz, p.gy, p.gx), 16, gen).abs().reshape(-1)
            s["g_den"] = target - s["den"]
            s["g_vel"] = 0.1 * torch.randn(s["vel"].shape, generator=gen, device="cuda")
            s["sim"].import_field_device("temperature", s["tem"].data_ptr(), s["tem"].numel())
            s["steps"], s["every"] = case["steps"], case["every"]
        else:
            s["steps"], s["thermal"] = case["steps"], p.source_mode == SOURCE_SPHERE_BUOYANT
            s["out"] = [torch.empty_like(s["den"]), torch.empty_like(s["vel"]), torch.empty_like(s["tem"])]
        torch.cuda.synchronize()
        return s
    if kind == "terrain":
        p = _terrain_params(case, seed)
        sim = dcgrid_amd.Simulation("dcgrid", _box(case), p, _dense_budget(case))
        sim.seed_scene()
        sim.step(case["warm"])
        n = sim.field_size("density")
        s.update(sim=sim, steps=case["steps"],
                 out=[torch.empty(n, device="cuda"), torch.empty(n, 3, device="cuda"), torch.empty(n, device="cuda"),
                      torch.empty(n, device="cuda")])
        sim.synchronize()
        return s
    if kind == "dcgrid" and case["scene"] == "reference":
        p = scenes.reference_params(*_box(case))
        p.enable_additional_solids = 1
        p.max_levels = case["levels"]
        p.init_velocity_noise = 20.0  # the reference starts at rest: seeded motion instead
        p.seed = seed & 0x7FFFFFFF
        budget = case["budget"]
    else:
        p = _plume_params(case, seed)
        budget = case["budget"]
        if case.get("scene") == "dense":
            budget = _dense_budget(case)
            p.emission_radius = 0.0
    p.storage = STORAGE[case.get("storage", "fp32")]
    if kind == "frame" and case["solve"]:
        p.project_mode = PROJECT_SOLVE
    sim = _dcgrid(case, p, budget)
    s["sim"] = sim
    if kind == "frame":
        s["steps"] = case["steps"]
        r = sim.default_render_params()
        r.width, r.height = case["width"], case["height"]
        s["render"] = r
        s["image"] = torch.empty(case["height"], case["width"], 4, device="cuda")
        return s
    n = sim.field_size("density")
    s["out"] = [torch.empty(n, device="cuda"), torch.empty(n, 3, device="cuda")]
    if kind == "dcgrid":
        s["steps"] = case["steps"]
        return s
    s["vel"] = _export(sim, "velocity", torch.empty(n, 3, device="cuda"))
    if kind == "adjoint":
        s["den"] = _export(sim, "density", torch.empty(n, device="cuda"))
        gen = torch.Generator(device="cuda")
        gen.manual_seed(int(seed) + 1)
        s["g_den"] = torch.randn(n, generator=gen, device="cuda")
        s["g_vel"] = 0.1 * torch.randn(n, 3, generator=gen, device="cuda")
        s["steps"], s["every"] = case["steps"], case["every"]
    torch.cuda.synchronize()
    return s


def run(s):
    kind, sim = s["kind"], s["sim"]
    if kind in ("control", "adjoint"):
        d0 = s["den"].detach().requires_grad_(True)
        v0 = s["vel"].detach().requires_grad_(True)
        den, vel = autograd.rollout(sim, d0, v0, s["steps"], s["every"])
        gd, gv = torch.autograd.grad([den, vel], [d0, v0], [s["g_den"], s["g_vel"]])
        return {"density": den.detach(), "velocity": vel.detach(), "grad_density": gd, "grad_velocity": gv}
    if kind in ("dcgrid", "frame"):
        sim.reset()
        sim.seed_scene()
    if kind == "frame":
        sim.step(s["steps"])
        sim.render_device(s["render"], s["image"].data_ptr())
        return s["image"]
    if kind == "solve":
        sim.import_field_device("velocity", s["vel"].data_ptr(), s["vel"].numel())
        sim.project_solve()
        return {"pressure": _export(sim, "pressure", s["out"][0]), "velocity": _export(sim, "velocity", s["out"][1])}
    if kind == "uniform":
        sim.import_field_device("density", s["den"].data_ptr(), s["den"].numel())
        sim.import_field_device("velocity", s["vel"].data_ptr(), s["vel"].numel())
        if s["thermal"]:
            sim.import_field_device("temperature", s["tem"].data_ptr(), s["tem"].numel())
    sim.step(s["steps"])
    out = {"density": _export(sim, "density", s["out"][0]), "velocity": _export(sim, "velocity", s["out"][1])}
    if kind == "terrain":
        out["temperature"] = _export(sim, "temperature", s["out"][2])
        out["vapor"] = _export(sim, "vapor", s["out"][3])
    elif kind == "uniform" and s["thermal"]:
        out["temperature"] = _export(sim, "temperature", s["out"][2])
    return out


# ---------------------------------------------------------------------------- compulsory work
def _uniform_levels(case):
    gx, gy, gz = _box(case)
    L, c = 1, 2
    while gx % c == 0 and gy % c == 0 and gz % c == 0 and c * 4 <= min(gx, gy, gz):
        L += 1
        c *= 2
    return L


def work(case):
    """Bytes: every stage of the step reads its input fields once and writes its outputs once (a
    Jacobi half-sweep 12 B a cell: pressure and divergence in, pressure out). Flops: the stencils'
    and samples' additions and multiplications (a half-sweep 9, a trilinear sample of one
    component about 16, its weights about 30)."""
    gx, gy, gz = _box(case)
    kind = case["kind"]
    if kind in ("uniform", "control"):
        n = gx * gy * gz
        local = case.get("mode") == "local"
        sweeps = 2 * case["pairs"] if local else 2 + 4 / 7
        thermal = 1 if case.get("scene") == "plume" else 0
        # advect u 24(+8), divergence 16, sweeps, gradient 28, advect scalars 12 + 8 each
        step_b = n * (24 + 8 * thermal + 16 + 12 * sweeps + 28 + 20 + 8 * thermal)
        step_f = n * (30 + 48 + 12 + 9 * sweeps + 15 + 30 + 16 * (1 + thermal))
        if kind == "control":  # forward, and backward with each segment's steps run again
            again = 0 if case["every"] == 1 else (case["every"] - 1) / case["every"]
            return {"bytes": case["steps"] * step_b * (3 + again), "flops": case["steps"] * step_f * (3 + again)}
        return {"bytes": case["steps"] * step_b + n * (16 + 4 * thermal) * 4, "flops": case["steps"] * step_f}
    if kind == "terrain":
        cells = 512 * _dense_budget(case)
        return {"bytes": cells * (case["steps"] * 310.0 + 48), "flops": cells * case["steps"] * 420.0}
    if case.get("scene") == "dense":
        cells = 512 * _dense_budget(case)
    else:  # the adaptation fills about this share of a budget
        share = {"reference": 0.6}.get(case.get("scene"), 0.25)
        cells = share * case["budget"] * case.get("bw", 8) ** 3
    es = 4 if case.get("storage", "fp32") == "fp32" else 2
    solve_b = 8 * 60 + 40  # about eight cycles a level: smoothing, transfers, residual; divergence and gradient
    if kind == "solve":
        return {"bytes": cells * solve_b, "flops": cells * 8 * 110.0}
    step_b = cells * 260 * es / 4
    step_f = cells * 330.0
    if kind == "adjoint":
        again = 0 if case["every"] == 1 else (case["every"] - 1) / case["every"]
        return {"bytes": case["steps"] * step_b * (3 + again), "flops": case["steps"] * step_f * (3 + again)}
    if kind == "frame" and case["solve"]:
        step_b += cells * (solve_b - 130)
        step_f += cells * 8 * 110.0
    out = case["width"] * case["height"] * 16 if kind == "frame" else cells * 32
    return {"bytes": case["steps"] * step_b + out, "flops": case["steps"] * step_f}


# ---------------------------------------------------------------------------- 64-bit values
class _Dense64:
    """The dense grid's step in 64 bits (plain torch, differentiable in density and velocity),
    with fields as (z, y, x) arrays and the velocity as three of them."""

    def __init__(self, p):
        self.p = p
        self.shape = (p.gz, p.gy, p.gx)
        z, y, x = (torch.arange(n, device="cuda", dtype=torch.float64) for n in self.shape)
        self.z, self.y, self.x = z[:, None, None], y[None, :, None], x[None, None, :]
        self.levels = []
        L = _uniform_levels({"gx": p.gx, "gy": p.gy, "gz": p.gz})
        for l in range(L):
            self.levels.append((p.gz >> l, p.gy >> l, p.gx >> l))
        self.flu = self._fluidity() if p.enable_additional_solids else None

    def _fluidity(self):
        p = self.p
        r = 2000.0 * p.rdx
        d = torch.sqrt((self.x + 0.5 - 0.5 * p.gx) ** 2 + (self.y + 0.5 - 0.45 * p.gy) ** 2 +
                       (self.z + 0.5 - 0.5 * p.gz) ** 2) - r
        return 1.0 - torch.clamp(0.5 - d / 1.73205, 0.0, 1.0)

    def _sample(self, vel, fields, bcs):
        """Trilinear samples of `fields` at the backtraced feet; bcs[i](value, x, y, z) applies the
        boundary condition of field i at unclamped corner coordinates."""
        p = self.p
        size = (p.gx, p.gy, p.gz)
        base, frac = [], []
        for c, g in zip(vel, (self.x, self.y, self.z)):
            f = g - c * (p.dt * p.rdx)
            b = torch.floor(f.detach())
            base.append(b.to(torch.int64))
            frac.append(f - b)
        acc = [0.0] * len(fields)
        wsum = 0.0
        for corner in range(8):
            bits = ((corner >> 2) & 1, (corner >> 1) & 1, corner & 1)
            w = 1.0
            at = []
            for a in range(3):
                w = w * (frac[a] if bits[a] else 1.0 - frac[a])
                at.append(base[a] + bits[a])
            idx = [at[a].clamp(0, size[a] - 1) for a in range(3)]
            lin = (idx[2] * p.gy + idx[1]) * p.gx + idx[0]
            if self.flu is not None:
                w = w * self.flu.reshape(-1)[lin]
            wsum = wsum + w
            for i, (f, bc) in enumerate(zip(fields, bcs)):
                acc[i] = acc[i] + w * bc(f.reshape(-1)[lin], *at)
        ok = wsum >= 1e-6
        return [torch.where(ok, a / wsum, torch.zeros_like(a)) for a in acc]

    def _bc(self, inlet, outer):
        p = self.p

        def apply(v, x, y, z):
            out = (x < 0) | (y < 0) | (z < 0) | (x >= p.gx) | (y >= p.gy) | (z >= p.gz)
            v = torch.where(out, torch.full_like(v, outer), v)
            if p.emission_radius > 0:
                r = torch.sqrt((x - 0.5 * p.gx).double() ** 2 + (z - 0.5 * p.gz).double() ** 2)
                v = torch.where((y < 0) & (r < p.emission_radius * p.rdx), torch.full_like(v, inlet), v)
            return v
        return apply

    @staticmethod
    def _shift(f, axis, step):
        """Values of the neighbour cell, the own cell's at the border."""
        n = f.shape[axis]
        if step > 0:
            return torch.cat([f.narrow(axis, 1, n - 1), f.narrow(axis, n - 1, 1)], axis)
        return torch.cat([f.narrow(axis, 0, 1), f.narrow(axis, 0, n - 1)], axis)

    def _jacobi(self, p, div, level, pairs):
        alpha = (self.p.dx * (1 << level)) ** 2
        for _ in range(2 * pairs):
            s = 0.0
            for axis in (2, 1, 0):
                s = s + self._shift(p, axis, -1) + self._shift(p, axis, 1)
            p = (s - alpha * div) / 6.0
        return p

    def _prolong(self, coarse, level):
        d, h, w = self.levels[level]
        lin = []
        for n in (d, h, w):
            i = torch.arange(n, device="cuda")
            s = torch.where((i == 0) | (i == n - 1), torch.zeros_like(i), 2 * (i % 2) - 1)
            lin.append((i // 2, i // 2 + s))
        for axis, (own, other) in enumerate(lin):
            a, b = coarse.index_select(axis, own), coarse.index_select(axis, other)
            coarse = 0.75 * a + 0.25 * b
        return coarse

    def _project(self, vel):
        p = self.p
        div = 0.0
        for c, (axis, coord) in enumerate(((2, 0), (1, 1), (0, 2))):
            bc = self._bc(p.velocity_emission_rate if coord == 1 else 0.0, 0.0)
            for step in (-1, 1):
                at = [g.to(torch.int64).expand(self.shape) for g in (self.x, self.y, self.z)]
                at[coord] = at[coord] + step
                v = bc(self._shift(vel[c], axis, step), *at)
                if self.flu is not None:
                    v = v * self._shift(self.flu, axis, step)
                div = div + step * v
        div = div * (0.5 * p.rdx)
        if p.project_mode == PROJECT_LOCAL:
            pre = self._jacobi(torch.zeros_like(div), div, 0, p.project_local_pairs)
        else:
            divs = [div]
            for _ in self.levels[1:]:
                d = divs[-1]
                a, b, c = (n // 2 for n in d.shape)
                divs.append(d.reshape(a, 2, b, 2, c, 2).mean((1, 3, 5)))
            top = len(self.levels) - 1
            pre = self._jacobi(torch.zeros_like(divs[top]), divs[top], top, p.project_top_pairs)
            for l in range(top - 1, -1, -1):
                pre = self._jacobi(self._prolong(pre, l), divs[l], l, p.project_level_pairs)
        out = []
        for c, axis in enumerate((2, 1, 0)):
            r, l = self._shift(pre, axis, 1) - pre, pre - self._shift(pre, axis, -1)
            if self.flu is not None:
                r, l = r * self._shift(self.flu, axis, 1), l * self._shift(self.flu, axis, -1)
            out.append(vel[c] - 0.5 * p.rdx * (r + l))
        return out

    def step(self, den, vel, tem):
        p = self.p
        thermal = p.source_mode == SOURCE_SPHERE_BUOYANT
        bcs = [self._bc(0.0, 0.0), self._bc(p.velocity_emission_rate, 0.0), self._bc(0.0, 0.0)]
        new = self._sample(vel, vel, bcs)
        if thermal:
            new[1] = new[1] + p.dt * (p.buoy_beta * (tem - p.t_ambient) - p.buoy_alpha * den)
        vel = self._project(new)
        fields, bcs = [den], [self._bc(p.density_emission_rate, 0.0)]
        if thermal:
            fields.append(tem)
            bcs.append(self._bc(p.t_ambient, p.t_ambient))
        got = self._sample(vel, fields, bcs)
        den = got[0]
        if thermal:
            inside = ((self.x + 0.5 - p.src_center[0]) ** 2 + (self.y + 0.5 - p.src_center[1]) ** 2 +
                      (self.z + 0.5 - p.src_center[2]) ** 2) < p.src_radius ** 2
            den = torch.where(inside, torch.full_like(den, p.src_density), den)
            tem = torch.where(inside, self._source_temperature(), got[1])
        return den, vel, tem

    def _source_temperature(self):
        """Source temperature plus the seeded hash noise of every cell (32-bit integer mixing)."""
        p = self.p
        mask = 0xFFFFFFFF

        def mix(h):
            h = h ^ (h >> 16)
            h = (h * 0x7FEB352D) & mask
            h = h ^ (h >> 15)
            h = (h * 0x846CA68B) & mask
            return h ^ (h >> 16)

        seed = (p.seed ^ 0x2545F491) ^ 0x9E3779B9
        h = mix(torch.tensor(seed & mask, device="cuda", dtype=torch.int64))
        h = mix(h ^ self.x.to(torch.int64))
        h = mix(h ^ self.y.to(torch.int64) ^ 0x68E31DA4)
        h = mix(h ^ self.z.to(torch.int64) ^ 0xB5297A4D)
        h = mix(h ^ 0x1B56C4E9)
        u = (h >> 8).double() / 16777216.0
        return p.src_temperature + p.src_noise * (2.0 * u - 1.0)


def _exact_uniform(case, seed):
    p = _uniform_params(case, seed)
    den, vel, tem = _uniform_inputs(case, seed)
    shape = (p.gz, p.gy, p.gx)
    S = _Dense64(p)
    den, tem = den.double().reshape(shape), tem.double().reshape(shape)
    vel = [c.contiguous().reshape(shape) for c in vel.double().t()]
    if case["kind"] == "uniform":
        for _ in range(case["steps"]):
            den, vel, tem = S.step(den, vel, tem)
        out = {"density": den.reshape(-1), "velocity": torch.stack([c.reshape(-1) for c in vel], 1)}
        if p.source_mode == SOURCE_SPHERE_BUOYANT:
            out["temperature"] = tem.reshape(-1)
        return out
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) + 1)
    g_den = (_smooth(shape, 16, gen).abs().reshape(-1) - den.reshape(-1).float()).double().reshape(shape)
    g_vel = (0.1 * torch.randn(den.numel(), 3, generator=gen, device="cuda")).double()
    g_vel = [c.contiguous().reshape(shape) for c in g_vel.t()]
    # forward keeping each step's input, then one step at a time in reverse
    states = [(den, vel)]
    for _ in range(case["steps"]):
        with torch.no_grad():
            d, v, _t = S.step(states[-1][0], states[-1][1], tem)
        states.append((d, v))
    gd, gv = g_den, g_vel
    for d, v in reversed(states[:-1]):
        d, v = d.detach().requires_grad_(True), [c.detach().requires_grad_(True) for c in v]
        d1, v1, _t = S.step(d, v, tem)
        got = torch.autograd.grad([d1] + v1, [d] + v, [gd] + gv)
        gd, gv = got[0], list(got[1:])
    flat = lambda vs: torch.stack([c.reshape(-1) for c in vs], 1)  # noqa: E731
    return {"density": states[-1][0].reshape(-1), "velocity": flat(states[-1][1]), "grad_density": gd.reshape(-1),
            "grad_velocity": flat(gv)}


def exact(case, seed):
    """The dense grid's steps and gradients in 64 bits. The other kinds run on a block topology
    that the library's own adaptation builds (or, on the terrain, part by 1e-3 a step between 32
    and 64 bits through the saturation adjustment): no value from outside the library."""
    if case["kind"] in ("uniform", "control"):
        return _exact_uniform(case, seed)
    return None
