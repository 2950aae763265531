"""Images of few rays take four lanes per ray, images of many take one: the same
image and step counts, bit for bit. Rays along z through the box see the same
positions in every pixel, so a pixel's result depends on its multipliers alone
and the pixels of a small image can be compared with those of a large one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mray_amd import hip, synth, tf as tfmod  # noqa: E402
from mray_amd.types import RecParams  # noqa: E402


# step counts of the march: none of, one short of, equal to and one past a
# multiple of four; early termination in the middle of one (ert 0.7)
@pytest.mark.parametrize("step,ert", [(0.3, 0.95), (0.0101, 0.95), (0.0099, 0.95), (0.25, 0.95), (2.0, 0.95),
                                      (0.004, 0.7)])
@pytest.mark.parametrize("m", [1, 8, 30, 50, 60, 96, 104, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_few_rays_as_many(m, step, ert, dtype):
    hip.init()
    g = torch.Generator().manual_seed(m)
    W, H = 17, 9
    n, NW, NH = W * H, 256, 200
    lag = torch.randn((n, m), generator=g, dtype=torch.float64) / torch.arange(1, m + 1) ** 1.5
    lag[:, 0] *= 3.0
    lag = lag.to(dtype).cuda()
    reps = (NW * NH + n - 1) // n
    many = lag.repeat(reps, 1)[: NW * NH].contiguous()
    cam = synth.ortho_camera(pos=(0.5, 0.5, -1.0), right=(0.4, 0, 0), up=(0, 0.4, 0))
    table = torch.from_numpy(tfmod.table_from_rgba8(synth.tf_ramps(0), 2.0))
    rp = RecParams(step_size=step, early_ray_termination=ert)
    box = ((0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
    a, sa = hip.reconstruct(cam, *box, lag.reshape(-1), W, H, m, table, rp, want_steps=True)
    b, sb = hip.reconstruct(cam, *box, many.reshape(-1), NW, NH, m, table, rp, want_steps=True)
    assert np.array_equal(sa.cpu().numpy(), sb.cpu().numpy()[:n])
    assert np.array_equal(a.cpu().numpy().reshape(n, 4), b.cpu().numpy().reshape(-1, 4)[:n])
    assert int(sa.min()) >= 1

    # compact: pixels of fewer and of no moments among them
    counts = torch.randint(0, m + 1, (n,), generator=g)
    keep = (torch.arange(m)[None, :] < counts[:, None]).cuda()
    bounds = torch.randint(0, 2**31 - 1, (n,), generator=g, dtype=torch.int32).cuda()

    def compact(rows, kp, c):
        idx = torch.zeros(c.numel() + 1, dtype=torch.int64)
        idx[1:] = torch.cumsum(c, 0)
        return torch.cat([rows[kp], rows.new_zeros(1)]), idx.to(torch.int32).cuda()

    data, index = compact(lag, keep, counts)
    big, bindex = compact(many, keep.repeat(reps, 1)[: NW * NH], counts.repeat(reps)[: NW * NH])
    bbounds = bounds.repeat(reps)[: NW * NH].contiguous()
    a, sa = hip.reconstruct(cam, *box, data, W, H, m, table, rp, index=index, bounds=bounds, want_steps=True)
    b, sb = hip.reconstruct(cam, *box, big, NW, NH, m, table, rp, index=bindex, bounds=bbounds, want_steps=True)
    assert np.array_equal(sa.cpu().numpy(), sb.cpu().numpy()[:n])
    assert np.array_equal(a.cpu().numpy().reshape(n, 4), b.cpu().numpy().reshape(-1, 4)[:n])
