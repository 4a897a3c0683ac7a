"""Context.intersect_host against the device-resident call, on both sides of the size up to which its rays
and records are in pinned host memory, growing and shrinking between calls."""
import numpy as np
import pytest

import cubiquity_amd as cq


@pytest.mark.gpu
def test_host_call_equals_device_call():
    import torch

    hv = cq.HostVolume.generate(cq.gen_default_params(7, 3))
    ctx = cq.Context(0)
    vol = ctx.upload(hv)
    for seed, n in enumerate([1, 65, 1000, 65535, 65536, 3, 65537, 97]):
        rays = cq.incoherent_rays(hv, 7, seed + 1, n)
        flags = 0 if seed == 4 else cq.CQX_SURFACE_PROPERTIES
        host = ctx.intersect_host(vol, rays, flags)
        dev = cq.intersectVolume(ctx, vol, torch.from_numpy(rays).cuda(), flags != 0)
        torch.cuda.synchronize()
        assert np.array_equal(host.view(np.uint8).reshape(-1), dev.cpu().numpy().reshape(-1))
