"""GPU projection solve (DCG_PROJECT_SOLVE) through the C ABI: every level's system (the fixed
point of the reference's Jacobi sweeps) solved to a 1e-8 relative residual by FP64 iterative
refinement around FP32 multigrid cycles, checked against the FP64 oracle's SOR solution of the
same system (solved to 1e-12), against the all-FP32 and all-FP64 variants, and against the
reference Jacobi sweep itself (a solution is its fixed point)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import dcgrid_amd  # noqa: E402
from dcgrid_amd import scenes  # noqa: E402
from dcgrid_amd._abi import PROJECT_SOLVE, SOLVE_FP32, SOLVE_FP64, SOLVE_MIXED, STAGE_JACOBI  # noqa: E402
from parity_util import rel_l2  # noqa: E402


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def workload(name):
    if name == "cfg2_128":
        w = scenes.config(2, scale=4)
        return w.kind, w.size, w.params, w.max_num_blocks
    if name == "cfg1_128":
        w = scenes.config(1, scale=2)
        return w.kind, w.size, w.params, w.max_num_blocks
    if name == "ref64_bw4":
        p = scenes.reference_params(64)
        return "dcgrid", (64, 64, 64), p, 1500
    if name == "cfg4_128":  # terrain solids: fluidity in the divergence and the gradient
        w = scenes.config(4, scale=8)
        return w.kind, w.size, w.params, w.max_num_blocks
    raise KeyError(name)


def prepared(name, precision, steps=4):
    """GPU and FP64-oracle simulations after `steps` reference steps, the oracle's velocity
    replaced by the GPU's (identical tables, identical projection input)."""
    import oracle
    kind, size, p, b = workload(name)
    p = p.copy()
    p.solve_precision = precision
    p.solve_tol = 1e-8
    p.solve_max_cycles = 60
    say(f"[case] {name} precision={precision}")
    g = dcgrid_amd.Simulation(kind, size, p, b)
    c = oracle.OracleSim(kind, size, p, b, precision=64)
    if name != "ref64_bw4":
        g.seed_scene()
        c.seed_scene()
    g.step(steps)
    c.step(steps)
    assert all(np.array_equal(a, b_) for a, b_ in zip(
        (g.export_tables()[k] for k in ("block_levels", "parent_indices")),
        (c.export_tables()[k] for k in ("block_levels", "parent_indices"))))
    c.import_field("velocity", g.export_field("velocity"))
    return g, c


def level_cells(sim, level):
    inf = sim.info()
    t = sim.export_tables()
    return np.repeat(t["block_levels"] == level, inf.block_width ** 3)


@pytest.mark.parametrize("name", ["cfg2_128", "ref64_bw4", "cfg1_128", "cfg4_128"])
def test_mixed_solve_reaches_tolerance_and_matches_oracle(name):
    g, c = prepared(name, SOLVE_MIXED)
    g.project_solve()
    c.project_solve()
    rg, rc = g.solve_report(), c.solve_report()
    say("gpu", rg)
    say("oracle", {k: rc[k] for k in ("cycles", "rel_residual")})
    assert rg["converged"]
    assert max(rg["rel_residual"]) <= 1e-8
    assert rg["singular"] == rc["singular"]
    mask = (g.export_tables()["block_levels"] != 0xFF).repeat(g.info().block_width ** 3)
    pg, pc = g.export_field("pressure")[mask], c.export_field_f64("pressure")[mask]
    vg, vc = g.export_field("velocity")[mask], c.export_field_f64("velocity")[mask]
    say("pressure rel l2", rel_l2(pg, pc), "velocity rel l2", rel_l2(vg, vc))
    # measured: pressure 2.8e-8 / 8.7e-8 / 2.9e-8, velocity 1.0e-7 / 3.1e-8 / 3.5e-7
    assert rel_l2(pg, pc) <= 2e-7
    assert rel_l2(vg, vc) <= 1e-6


def test_fixed_point_of_the_reference_jacobi_sweep():
    """A converged pressure is (to FP32 rounding) unchanged by one Jacobi half-sweep of the
    reference schedule on every level (dcgrid_multigrid_solver.cu:5-41)."""
    g, _ = prepared("cfg2_128", SOLVE_MIXED)
    g.project_solve()
    # the projection changed the velocity, but the pressure and divergence are those solved
    inf = g.info()
    rep = g.solve_report()
    p = g.export_field("pressure")
    for level in range(inf.levels):
        g.run_stage(STAGE_JACOBI, level)
        tp = g.export_field("t_pressure")
        m = level_cells(g, level)
        d = tp[m].astype(np.float64) - p[m]
        scale = np.linalg.norm(p[m]) / np.sqrt(m.sum())
        if rep["singular"][level]:
            # the singular level was solved with its right-hand side projected to zero mean: the
            # sweep then shifts every cell by the same constant (the removed mean / 6)
            d = d - d.mean()
        err = np.sqrt(np.mean(d * d)) / scale
        say("level", level, "singular", rep["singular"][level], "jacobi change", err)
        assert err <= 3e-7  # measured about 6e-8 on every level


def test_full_size_config2_small_regions():
    """Configuration 2 at its full 512^3 size, where sparse levels' regions (the top-level blocks
    holding their cells) cover at most 1/16 of the top level, so their V-cycles end at the top
    level without the pyramid: every level still reaches 1e-8, and the solution is (to FP32
    rounding) a fixed point of the reference Jacobi half-sweep on every level."""
    w = scenes.config(2)
    p = w.params.copy()
    p.project_mode = PROJECT_SOLVE
    p.solve_precision = SOLVE_MIXED
    p.solve_tol = 1e-8
    say("[case] config 2 at 512^3, 6 solved steps")
    g = dcgrid_amd.Simulation(w.kind, w.size, p, w.max_num_blocks)
    g.seed_scene()
    g.step(6)
    inf = g.info()
    t = g.export_tables()
    lev, par = t["block_levels"], t["parent_indices"]
    L, top = inf.levels, inf.levels - 1
    full = [(512 // (8 << l)) ** 3 for l in range(L)]
    loads = list(inf.block_loads)[:L]
    none = np.uint64(0xFFFFFFFFFFFFFFFF)
    small = []
    for l in range(top):
        if loads[l] >= full[l]:
            continue  # dense level
        b = np.nonzero(lev == l)[0]
        for _ in range(top - l):
            b = (par[b] // 8).astype(np.int64)
        tops = np.unique(b)
        say("sparse level", l, "region covers", tops.size, "of", full[top], "top-level blocks")
        if tops.size * 16 <= full[top]:
            small.append(l)
    assert small, "no sparse level with a small region: the case does not exercise that cycle"
    assert not np.any(par[lev == top] != none)
    g.project_solve()
    rep = g.solve_report()
    say("cycles", rep["cycles"], "rel", rep["rel_residual"])
    assert rep["converged"] and all(r <= 1e-8 for r in rep["rel_residual"])
    pr = g.export_field("pressure")
    for level in range(L):
        g.run_stage(STAGE_JACOBI, level)
        tp = g.export_field("t_pressure")
        m = level_cells(g, level)
        d = tp[m].astype(np.float64) - pr[m]
        scale = np.linalg.norm(pr[m]) / np.sqrt(m.sum())
        if rep["singular"][level]:
            d = d - d.mean()
        err = np.sqrt(np.mean(d * d)) / scale
        say("level", level, "small region" if level in small else "", "jacobi change", err)
        assert err <= 3e-7
    g.close()


def test_precision_variants():
    """FP64 throughout also reaches 1e-8 and agrees with the mixed solve; FP32 throughout stops
    where its arithmetic runs out (reported, not converged at 1e-8) with a larger error."""
    res = {}
    for prec in (SOLVE_MIXED, SOLVE_FP64, SOLVE_FP32):
        g, c = prepared("cfg2_128", prec)
        g.project_solve()
        if prec == SOLVE_MIXED:
            c.project_solve()
            res["oracle"] = c.export_field_f64("pressure")
        res[prec] = (g.solve_report(), g.export_field("pressure"), g)
    mask = (res[SOLVE_MIXED][2].export_tables()["block_levels"] != 0xFF).repeat(512)
    ref = res["oracle"][mask]
    e_mixed = rel_l2(res[SOLVE_MIXED][1][mask], ref)
    e_64 = rel_l2(res[SOLVE_FP64][1][mask], ref)
    e_32 = rel_l2(res[SOLVE_FP32][1][mask], ref)
    say("errors vs oracle: mixed", e_mixed, "fp64", e_64, "fp32", e_32)
    say("fp32 report", res[SOLVE_FP32][0])
    assert res[SOLVE_FP64][0]["converged"]
    assert max(res[SOLVE_FP64][0]["rel_residual"]) <= 1e-8
    assert e_64 <= 2e-7 and e_mixed <= 2e-7  # measured 2.8e-8 (both)
    assert max(res[SOLVE_FP32][0]["rel_residual"]) > 1e-8 or e_32 <= 1e-5


# Dense grids around the direct solve's tiles, with the lines of the finest level's x, y and z passes: axes
# below and past multiples of 32 (padded transform halves), of one block, BW 4 and 8; the longest axes of the
# 32-line tiles (512) and of the 16-line ones (1024) along x, y and z (where 16 lines are part of a
# block column); 64-line tiles of 16 and of several matrix tiles, up to the longest (256), with padded
# halves (136, 132), and for BW 4 with four block columns a tile, the last one partial in every pass.
DIRECT_CASES = [((64, 96, 160), 8, 3, (32, 32, 32)), ((48, 16, 80), 8, 2, (32, 32, 32)), ((8, 8, 8), 8, 1, (32, 32, 32)),
                ((24, 8, 40), 8, 1, (32, 32, 32)), ((24, 40, 56), 4, 2, (32, 32, 32)), ((16, 16, 16), 4, 3, (32, 32, 32)),
                ((20, 4, 12), 4, 1, (32, 32, 32)), ((256, 16, 32), 8, 2, (32, 32, 32)), ((16, 320, 32), 8, 2, (32, 32, 32)),
                ((16, 32, 512), 8, 2, (64, 32, 32)), ((512, 16, 16), 8, 2, (32, 32, 32)),
                ((1024, 16, 16), 8, 2, (16, 64, 64)), ((16, 1024, 16), 8, 1, (64, 16, 64)),
                ((16, 16, 1024), 8, 1, (64, 64, 16)), ((8, 12, 520), 4, 1, (32, 32, 16)),
                ((256, 128, 256), 8, 2, (64, 64, 64)), ((136, 136, 136), 8, 1, (64, 64, 64)),
                ((132, 132, 132), 4, 1, (64, 64, 64))]


def direct_lines(size, bw):
    """The lines of a tile in the x, y and z passes by the direct solve's rule: 16 beyond 512 cells of the
    axis, 64 where the axis has at most 256 and the pass at least 256 tiles of them, else 32."""
    up = lambda a, b: -(-a // b)  # noqa: E731
    nx, ny, nz = size
    tiles = (up(ny * nz, 64), nx // bw * up(nz, 64 // bw), up(nx * ny, 64))
    return tuple(16 if n > 512 else 64 if n <= 256 and t >= 256 else 32 for n, t in zip(size, tiles))


@pytest.mark.parametrize("size,bw,levels,lines", DIRECT_CASES)
def test_dense_levels_against_cosine_transform(size, bw, levels, lines):
    """Every level of a fully dense grid is a box with Neumann walls: its pressure is the zero-mean
    solution of scipy's DCT-II in 64 bits, to the rounding of the stored FP32 pressure (1e-7 covers
    its 6e-8); throughout FP32 to the residual's rounding, which the smoothest mode of the longest axis
    (one of all cells) amplifies by (n / pi)^2: 6e-8 (20 + 40 (n / pi)^2 / sqrt(cells))."""
    from scipy.fft import dctn, idctn
    assert direct_lines(size, bw) == lines
    p = scenes.reference_params(*size)
    p.dt, p.dx, p.rdx = 0.1, 1.0, 1.0
    p.emission_radius = 0.0
    p.block_width, p.max_levels = bw, levels
    budget = sum((size[0] // (bw << l)) * (size[1] // (bw << l)) * (size[2] // (bw << l)) for l in range(levels))
    p.solve_tol = 1e-8
    g = dcgrid_amd.Simulation("dcgrid", size, p, budget)
    assert g.info().levels == levels
    rng = np.random.default_rng(sum(size) + bw)
    vel = rng.standard_normal((g.field_size("density"), 3)).astype(np.float32)
    t = g.export_tables()
    lev, pos = t["block_levels"], t["block_positions"]
    bits = bw.bit_length() - 1
    loc = np.arange(bw ** 3)
    lx, ly, lz = (sum(((loc >> (3 * b + k)) & 1) << b for b in range(bits)) for k in (2, 1, 0))
    for prec in (SOLVE_MIXED, SOLVE_FP64, SOLVE_FP32):
        p.solve_precision = prec
        g.set_params(p)
        g.import_field("velocity", vel)
        g.project_solve()
        rep = g.solve_report()
        say(size, bw, "precision", prec, "cycles", rep["cycles"], "rel", rep["rel_residual"])
        if prec != SOLVE_FP32:
            assert rep["converged"]
        pre, div = g.export_field("pressure"), g.export_field("divergence")
        for l in range(levels):
            n = [v >> l for v in size]
            b = np.nonzero(lev == l)[0]
            x, y, z = (pos[b, a][:, None] + o[None, :] for a, o in enumerate((lx, ly, lz)))
            cells = b[:, None] * bw ** 3 + loc[None, :]
            box_p, box_d = np.empty(n), np.empty(n)
            box_p[x, y, z], box_d[x, y, z] = pre[cells], div[cells]
            lam = sum((4 * np.sin(np.pi * np.arange(n[a]) / (2 * n[a])) ** 2).reshape([-1 if a == k else 1 for k in range(3)])
                      for a in range(3))
            lam[0, 0, 0] = 1.0
            f = dctn(-box_d * float(1 << l) ** 2, type=2, norm="ortho") / lam
            f[0, 0, 0] = 0.0
            want = idctn(f, type=2, norm="ortho")
            err = rel_l2(box_p, want)
            say("  level", l, n, "pressure rel l2", err)
            noise = 20 + 40 * (max(n) / np.pi) ** 2 / np.sqrt(np.prod(n))
            assert err <= (1e-7 if prec != SOLVE_FP32 else 6e-8 * noise)
    g.close()


def test_step_with_solve_mode():
    """dcg_step with project_mode = DCG_PROJECT_SOLVE: every step's solve converges."""
    kind, size, p, b = workload("cfg2_128")
    p = p.copy()
    p.project_mode = PROJECT_SOLVE
    g = dcgrid_amd.Simulation(kind, size, p, b)
    g.seed_scene()
    g.step(3)
    rep = g.solve_report()
    say("step report", rep)
    assert rep["converged"]
    assert np.all(np.isfinite(g.export_field("velocity")))
