"""Volumes of few voxels per row, and rays along their faces: the march loads the
two corners of a row together, moved inside the row at its end, and one by one
where a row has one voxel. Sample counts and bounds against the FP32 oracle, bit for
bit, through generate (both forms) and the reference renderer, f32 and u8."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mray_amd import hip, synth, tf as tfmod  # noqa: E402
from mray_amd.types import GenParams, RefParams  # noqa: E402
from oracle_ffi import Oracle  # noqa: E402


@pytest.mark.parametrize("dtype", ["f32", "u8"])
@pytest.mark.parametrize("shape", [(3, 4, 1), (1, 1, 2), (5, 1, 3), (2, 7, 2), (1, 3, 1), (4, 5, 6)])
@pytest.mark.parametrize("ext", [1.0, 0.75])
def test_thin_volumes(shape, dtype, ext):
    O = Oracle()
    rng = np.random.default_rng(sum(shape))
    v = rng.uniform(0.05, 0.95, shape).astype(np.float32)
    if dtype == "u8":
        v = (v * 255).astype(np.uint8)
    dmin, dmax = (0.0, 0.0, 0.0), (ext, ext, ext)
    W, H, m = 17, 13, 8
    # the orthographic image's outer pixels run along the box's faces
    for cam in (synth.ortho_camera(pos=(0.5 * ext, 0.5 * ext, -1.0), right=(0.5 * ext, 0, 0), up=(0, 0.5 * ext, 0)),
                synth.perspective_camera(position=(0.4 * ext, 0.55 * ext, -0.8), aspect=W / H)):
        gp = GenParams(step_size=0.07, transform_to_bounds=1, transform_bound_eps=0.01, compact_image=0,
                       prediction_coding=0)
        vol = hip.Volume(torch.from_numpy(v).cuda(), dmin, dmax)
        mo_ref, b_ref, s_ref = O.generate(v, dmin, dmax, cam, W, H, m, gp)
        for form in ("mixed", "plain"):
            mo, b, s = hip.generate(vol, cam, gp, W, H, m, form=form, want_samples=True)
            assert np.array_equal(b.cpu().numpy().view(np.uint32), b_ref)
            assert np.array_equal(s.cpu().numpy(), s_ref)
            # f32 sums of up to 25 segments in the oracle
            assert np.abs(mo.cpu().numpy().reshape(mo_ref.shape) - mo_ref).max() <= 2e-5
        rp = RefParams(step_size=0.05, medium_emission=1.0)
        table = tfmod.table_from_rgba8(synth.tf_ramps(0), 2.0)
        ref, st_ref = O.reference(v, dmin, dmax, cam, W, H, table, rp)
        img, st = hip.reference(vol, cam, torch.from_numpy(table), rp, W, H, want_steps=True)
        assert np.array_equal(st.cpu().numpy(), st_ref)
        assert np.array_equal(img.cpu().numpy().reshape(ref.shape), ref)
