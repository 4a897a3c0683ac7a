"""The packed walk's reciprocal (plain_rcp: the hardware's, corrected twice) is the correctly rounded
quotient for every direction component it is used for: a ray that starts one voxel before a solid block
along an axis enters it at t = 1 * (1 / d), which the record holds."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_gpu_reciprocal_of_every_plain_component(cq, gpu_ctx, axis):
    import torch

    dv = gpu_ctx.upload(cq.HostVolume.from_dense(np.ones((4, 4, 4), np.uint8), (0, 0, 0)))
    lo, hi = (int(np.float32(v).view(np.uint32)) for v in (1.0e-18, 9.99e17))
    n, seen = 1 << 24, 0
    rays = torch.full((n, 6), 1.5, device="cuda")
    rays[:, axis] = -1.5
    rays[:, 3:] = float(np.nextafter(np.float32(1.0e-18), np.float32(1.0)))
    out = torch.empty((n, 32), dtype=torch.uint8, device="cuda")
    for first in range(lo + 1, hi + 1, n):
        d = torch.arange(first, first + n, dtype=torch.int32, device="cuda").clamp_(max=hi).view(torch.float32)
        rays[:, 3 + axis] = d
        cq.intersectVolume(gpu_ctx, dv, rays, out=out)
        record = out.view(torch.int32)  # t, voxel, node, info, ..
        want = (1.0 / d.double()).float()  # 53 bits are enough for the quotient's second rounding to be harmless
        assert (record[:, 5] & 1).all()
        assert torch.equal(record[:, 0], want.view(torch.int32)), hex(first)
        seen += n
        print(hex(first), flush=True)
    assert seen >= 1000000000
    dv.free()
