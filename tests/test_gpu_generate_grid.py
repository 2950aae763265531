"""The gridded march of generate against the march summed node by node.

A call that records the rays' normalisation (ray_range) sums every ray's
moments node by node; without it, the rays whose samples resolve the largest
order take the gridded march. Both evaluate the same integral in FP64 and round
each moment to float once: per ray they may differ by one rounding of the
largest moment (2^-23 of it; the gridded stencils add up to 1.6e-8 next to 8192
steps from the camera, less elsewhere, and the node sums up to 4e-8 on their own
FP32 terms). Bounds and sample counts are the same bits.
Sizes: orders from far below to just past what the samples resolve, chunks of
moments, images that are no multiple of a tile, t that passes powers of two
(whose increments change there) up to 8192 steps from the camera and past them,
cameras inside the box, also with a znear behind them, and domains that are no
power of two in byte and float volumes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mray_amd import hip, synth  # noqa: E402
from mray_amd.types import GenParams  # noqa: E402

CASES = {
    # n, (dmin, dmax), camera, W, H, m, step
    "resolved": (64, (-1, 1), synth.ortho_camera(), 24, 17, 20, 1.0 / 64),
    "limit": (64, (-1, 1), synth.ortho_camera(), 16, 16, 41, 1.0 / 64),
    "past_limit": (64, (-1, 1), synth.ortho_camera(), 16, 16, 42, 1.0 / 64),
    "persp_mixed": (48, (0, 1), synth.perspective_camera(aspect=40 / 30), 40, 30, 24, 0.5 / 48),
    # tiles of both forms, and ones whose rays differ, in one launch
    "persp_edge": (64, (0, 1), synth.perspective_camera(aspect=9 / 7), 90, 70, 44, 0.5 / 64),
    "chunks2": (96, (0, 1), synth.perspective_camera(position=(0.45, 0.5, -0.9)), 19, 21, 61, 0.25 / 96),
    "chunks3": (96, (0, 1), synth.perspective_camera(), 16, 9, 101, 0.15 / 96),
    "increments": (80, (0, 1), synth.perspective_camera(position=(0.5, 0.5, -3.3), fov_half_deg=9.0), 24, 24, 33,
                   0.37 / 80),
    # a power of two passed 7800 steps from the camera
    "reach": (80, (0, 1), synth.perspective_camera(position=(0.5, 0.5, -15.4), fov_half_deg=1.7), 24, 24, 33, 0.00206),
    "reach_chunks": (80, (0, 1), synth.perspective_camera(position=(0.5, 0.5, -15.4), fov_half_deg=1.7), 16, 16, 101,
                     0.00206),
    "inside": (64, (0, 1), synth.perspective_camera(position=(0.5, 0.4, 0.3), fov_half_deg=60.0), 24, 24, 20, 0.3 / 64),
    "behind": (64, (0, 1), synth.perspective_camera(position=(0.5, 0.4, 0.6), znear=-0.45), 24, 24, 20, 0.3 / 64),
    "far": (32, (0, 1), synth.perspective_camera(position=(0.5, 0.5, -90.0), fov_half_deg=0.3), 8, 8, 16, 0.01),
    "oblong": (50, (0, 0.9375), synth.perspective_camera(position=(0.4, 0.5, -1.0)), 24, 24, 30, 0.5 / 50),
    "one": (32, (0, 1), synth.perspective_camera(), 9, 9, 1, 0.5 / 32),
    "two": (32, (0, 1), synth.perspective_camera(), 9, 9, 2, 0.5 / 32),
}


@pytest.mark.parametrize("bounded", [1, 0])
@pytest.mark.parametrize("dtype", ["f32", "u8"])
@pytest.mark.parametrize("name", list(CASES))
def test_gridded_march_matches_node_sums(name, dtype, bounded):
    n, (lo, hi), cam, W, H, m, step = CASES[name]
    vol = synth.marschner_lobb(n) if lo < 0 else synth.mixing_layer(n, width=0.05)
    v = torch.from_numpy(vol).cuda()
    if dtype == "u8":
        v = (v.clamp(0, 1) * 255).to(torch.uint8)
    vol = hip.Volume(v, (lo,) * 3, (hi,) * 3)
    gp = GenParams(step_size=step, transform_to_bounds=bounded, transform_bound_eps=0.01, compact_image=0,
                   prediction_coding=0, bias=1e-4)
    _check(name, vol, cam, gp, W, H, m)


def _check(name, vol, cam, gp, W, H, m):
    rr = torch.empty((H * W, 2), dtype=torch.float32, device="cuda")
    ref, b_ref, s_ref = hip.generate(vol, cam, gp, W, H, m, ray_range=rr, want_samples=True)
    mo, b, s = hip.generate(vol, cam, gp, W, H, m, want_samples=True)
    assert torch.equal(s, s_ref) and (torch.equal(b, b_ref) if gp.transform_to_bounds else b is None)
    d = (mo.double() - ref.double()).view(-1, m).abs().amax(1)
    size = ref.double().view(-1, m).abs().amax(1)
    assert bool((size > 0).any())
    bound = 2.0 ** -23 * size + 4e-8
    assert bool((d <= bound).all()), f"{name}: {float((d / bound).max()):.2f} of the bound"


# Images of few rays take four lanes per ray, so the cases above are theirs; the
# same rays' lengths in images of many rays, which take one lane.
@pytest.mark.parametrize("dtype", ["f32", "u8"])
@pytest.mark.parametrize("name", ["resolved", "limit", "persp_mixed", "persp_edge", "increments", "reach", "reach_chunks", "inside", "behind",
                                  "oblong", "two"])
def test_gridded_march_many_rays(name, dtype):
    n, (lo, hi), cam, W, H, m, step = CASES[name]
    vol = synth.marschner_lobb(n) if lo < 0 else synth.mixing_layer(n, width=0.05)
    v = torch.from_numpy(vol).cuda()
    if dtype == "u8":
        v = (v.clamp(0, 1) * 255).to(torch.uint8)
    vol = hip.Volume(v, (lo,) * 3, (hi,) * 3)
    gp = GenParams(step_size=step, transform_to_bounds=1, transform_bound_eps=0.01, compact_image=0,
                   prediction_coding=0, bias=1e-4)
    _check(name, vol, cam, gp, 261, 259, m)


# rays of 1 to 17 nodes: lanes without a node, of one, of a ragged last share;
# nodes fewer than the stencils are wide
@pytest.mark.parametrize("nodes", range(1, 18))
@pytest.mark.parametrize("cam", ["ortho", "persp"])
def test_gridded_march_few_nodes(nodes, cam):
    v = torch.from_numpy(synth.mixing_layer(24, width=0.3)).cuda()
    vol = hip.Volume(v, (0,) * 3, (1,) * 3)
    c = (synth.ortho_camera(pos=(0.5, 0.5, -1.0), right=(0.6, 0, 0), up=(0, 0.4, 0)) if cam == "ortho"
         else synth.perspective_camera(fov_half_deg=12.0))
    for m in (1, 2, 3, 4, 5, 6):
        gp = GenParams(step_size=1.0 / (nodes + 0.5), transform_to_bounds=1, transform_bound_eps=0.01,
                       compact_image=0, prediction_coding=0, bias=1e-4)
        _check(f"{nodes} nodes, {m} moments", vol, c, gp, 21, 13, m)
