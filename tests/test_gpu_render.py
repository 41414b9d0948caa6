"""The renderer (dcg_render / dcg_render_host) on the GPU against the oracle's restatement of the
reference's ray marcher, bit for bit: every channel, precise and coarse sampling, shadows, the
floor and the solid scene, anti-aliasing, on DCGrid (BW 4 and 8, sparse and dense levels, FP16
storage, terrain) and the uniform grid, with the same fields on both sides (the oracle steps in
lockstep and is bit-exact on them). The device-pointer entry point equals the host one, and
inputs for which the marcher's loops would not end are rejected."""
import sys

import numpy as np
import pytest

import dcgrid_amd
import oracle
from dcgrid_amd import scenes
from dcgrid_amd._abi import (RENDER_DENSITY, RENDER_FLUID, RENDER_FLUIDITY, RENDER_RESOLUTION, RENDER_VELOCITY,
                             STORAGE_FP16)

pytestmark = pytest.mark.gpu

CHANNELS = [RENDER_FLUID, RENDER_DENSITY, RENDER_VELOCITY, RENDER_FLUIDITY, RENDER_RESOLUTION]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def workload(name):
    if name == "ref64_bw4_solids":
        p = scenes.reference_params(64)
        p.enable_additional_solids = 1
        return "dcgrid", (64, 64, 64), p, 2000
    if name in ("cfg1_64", "cfg1_64_fp16"):
        w = scenes.config(1, scale=4)
        p = w.params.copy()
        if name.endswith("fp16"):
            p.storage = STORAGE_FP16
        return w.kind, w.size, p, w.max_num_blocks
    if name == "cfg4_128":
        w = scenes.config(4, scale=8)
        return w.kind, w.size, w.params, w.max_num_blocks
    if name == "cfg0_32_solids":
        w = scenes.config(0, scale=2)
        p = w.params.copy()
        p.enable_additional_solids = 1
        return w.kind, w.size, p, None
    raise KeyError(name)


def pair(name, steps=3):
    kind, size, p, b = workload(name)
    g = dcgrid_amd.Simulation(kind, size, p, b)
    c = oracle.OracleSim(kind, size, p, b, precision=32)
    if name.startswith("ref"):
        g.step(steps)
        c.step(steps)
    else:
        g.seed_scene()
        c.seed_scene()
        g.step(steps)
        c.step(steps)
    return g, c


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("name", ["cfg1_64", "ref64_bw4_solids", "cfg4_128", "cfg1_64_fp16", "cfg0_32_solids"])
def test_render_bitwise_vs_oracle(name):
    say(f"[case] render {name}")
    g, c = pair(name)
    r = g.default_render_params()
    r.width, r.height = 40, 28
    for ch in CHANNELS:
        for precise in (1, 0):
            r.channel, r.precise = ch, precise
            a, b = g.render(r), c.render(r)
            assert np.isfinite(a).all()
            bad = ~np.all(a.view(np.uint32) == b.view(np.uint32), axis=2)
            assert not bad.any(), (name, ch, precise, int(bad.sum()), np.argwhere(bad)[:3].tolist())
    if name in ("cfg1_64", "cfg0_32_solids"):  # anti-aliasing, shadows off, another view
        r.channel, r.precise, r.aa_samples, r.shadows = RENDER_FLUID, 1, 2.0, 0
        r.eye_dir[1], r.eye_dir[2] = 0.1, 0.995
        assert same(g.render(r), c.render(r)), (name, "aa")
    g.close()
    c.close()


def test_device_pointer_and_checks():
    import torch
    g, c = pair("cfg1_64", steps=2)
    r = g.default_render_params()
    r.width, r.height = 33, 17
    host = g.render(r)
    out = torch.empty((r.height, r.width, 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    g.render_device(r, out.data_ptr())
    g.synchronize()
    assert same(out.cpu().numpy(), host)
    for field, value in (("aa_samples", 0.0), ("aa_samples", -1.0), ("aa_samples", 9.0), ("width", 0),
                         ("height", 20000), ("channel", 7), ("fov", float("nan"))):
        bad = r.copy()
        setattr(bad, field, value)
        with pytest.raises(dcgrid_amd.DCGError):
            g.render(bad)
    bad = r.copy()
    bad.eye_origin[2] = -2e6 * g.params.dx  # 2e6 cells away
    with pytest.raises(dcgrid_amd.DCGError):
        g.render(bad)
    g.close()
    c.close()


@pytest.mark.parametrize("name,size", [("cfg1_64", (1, 1)), ("cfg1_64", (5, 3)), ("ref64_bw4_solids", (17, 9)),
                                       ("cfg0_32_solids", (4, 4)), ("cfg1_64", (1025, 512)),
                                       ("cfg0_32_solids", (1025, 512))])
def test_render_lanes_per_ray(name, size):
    """The marched channel at the edges of its launch shapes: partial tiles (an image smaller than a
    tile, one past it), and one pixel row past the 512 K pixels from which 4 lanes take a ray instead
    of 16. The small images equal the oracle's; the large one's inner rows equal those of an image
    two rows lower, which takes 16 lanes."""
    g, c = pair(name)
    r = g.default_render_params()
    r.width, r.height = size
    a = g.render(r)
    if size[0] * size[1] <= 1024:
        assert same(a, c.render(r)), (name, size)
    else:  # the same rays from a narrower image: the pixel pitch follows the larger side
        half = r.copy()
        half.height = size[1] - 2
        b = g.render(half)
        assert size[0] * size[1] > 512 * 1024 >= half.width * half.height
        assert same(a[1:-1], b), (name, size)
    g.close()
    c.close()
