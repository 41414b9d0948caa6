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
    if name == "ref48_uniform_solids":  # the sphere and the inlet's fluid in view
        p = scenes.reference_params(48, kind="uniform")
        p.enable_additional_solids = 1
        return "uniform", (48, 48, 48), p, None
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


@pytest.mark.parametrize("name", ["cfg1_64", "ref64_bw4_solids", "cfg4_128", "cfg1_64_fp16", "cfg0_32_solids",
                                  "ref48_uniform_solids"])
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
    tile, one past it), and one pixel row past the 512 K pixels from which 4 lanes take a DCGrid's ray
    instead of 16 (on the dense grid, where the camera is inside the solid, both images take 4). The small
    images equal the oracle's; the large one's inner rows equal those of an image two rows lower."""
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


# One pixel row past each line of the rule that gives a ray its lanes, and one before: (scene, image, shadows,
# launches on either side). Two launches where rays that meet no fluid are finished by a launch of
# their own (several lanes a ray and more than 2^16 pixels, or a solid scene), one otherwise.
LANE_LINES = [("cfg1_64", (1449, 1448), 1, (1, 2)), ("cfg1_64", (513, 512), 0, (2, 2)), ("cfg1_64", (1025, 1024), 0, (1, 2)),
              ("cfg0_32", (513, 256), 1, (2, 2)), ("cfg0_32", (1025, 1024), 1, (1, 2)), ("cfg0_32", (257, 128), 0, (1, 1)),
              ("cfg0_32", (513, 512), 0, (1, 2)), ("cfg0_32", (257, 256), 1, (2, 1)), ("ref48_uniform_solids", (33, 32), 1, (2, 2)),
              ("cfg4_128", (513, 512), 1, (1, 2))]


@pytest.mark.parametrize("name,size,shadows,launches", LANE_LINES)
def test_render_lane_lines(name, size, shadows, launches):
    """The image does not depend on the lanes per ray: the inner rows on one side of a line equal the
    same rays on the other side (the pixel pitch follows the larger side). A sky view has rays that pass
    the domain by."""
    kind, shape, p, b = workload("cfg0_32_solids" if name == "cfg0_32" else name)
    p = p.copy()
    if name == "cfg0_32":
        p.enable_additional_solids = 0
    g = dcgrid_amd.Simulation(kind, shape, p, b)
    if not name.startswith("ref"):
        g.seed_scene()
    g.step(3)
    r = g.default_render_params()
    r.shadows = shadows
    for up in (-.2, .3):
        r.eye_dir[1], r.eye_dir[2] = up, float(np.sqrt(1 - up * up))
        images = []
        for rows, n in zip((size[1], size[1] - 2), launches):
            r.width, r.height = size[0], rows
            g.set_timing(["other"])
            images.append(g.render(r))
            assert g.timing()["other"][1] == n, (name, size, rows)
        assert same(images[0][1:-1], images[1]), (name, size, up)
    g.close()


@pytest.mark.parametrize("name", ["cfg1_64", "ref48_uniform_solids", "ref64_bw4_solids", "cfg4_128"])
def test_render_several_rays_with_shadows(name):
    """Four rays per pixel with shadow marches equal the oracle's: 16 lanes a ray (without and with a solid
    sphere, whose traces the lanes repeat) and one (terrain)."""
    g, c = pair(name)
    r = g.default_render_params()
    r.width, r.height, r.aa_samples, r.shadows = 23, 14, 2.0, 1
    a, b = g.render(r), c.render(r)
    assert same(a, b), name
    assert len(np.unique(a.reshape(-1, 4), axis=0)) > 2
    g.close()
    c.close()
