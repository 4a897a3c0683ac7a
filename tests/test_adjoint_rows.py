"""The adjoint's sums in LDS (pathtrace.hip, up to 16 materials) at the counts where the final row sums
change: 6 rows (1 material), 60 and 66 (one and two passes of the 64 lanes), 96 (the most), over paths
that leave the last wave part-full: the gradient equals the FP64 one of the same paths within 1e-4, the
tolerance of the adjoint's other tests."""
import numpy as np
import pytest

from cubiquity_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("materials,width,spp", [(1, 9, 1), (10, 37, 3), (11, 37, 3), (16, 64, 5)])
def test_adjoint_rows(cq, oracle, gpu_ctx, materials, width, spp):
    n = 48
    z, y, x = np.mgrid[0:n, 0:n, 0:n]
    grid = np.zeros((n, n, n), np.uint8)
    floor = y < 10 + ((x // 6 + z // 6) % 3)
    grid[floor] = (1 + (x // 3 + 16 * (z // 3)) % materials)[floor]
    hv = cq.HostVolume.from_dense(grid, (0, 0, 0))
    alb, em = cq.material_table(materials, 11)
    em = em + 0.01 * np.arange(1, materials + 1, dtype=np.float32)[:, None]
    s = cq.PathTraceSetup(W.Camera((24.0, 40.0, 4.0), (24.0, 8.0, 30.0), 70.0, width, 23), width, 23, spp, 3, alb, em)
    dv = gpu_ctx.upload(hv)
    img = cq.pathtrace(gpu_ctx, dv, s, 0).double()
    d_image = (2 * img - 0.1).float()
    da, de = cq.pathtrace_adjoint(gpu_ctx, dv, s, d_image)
    _, ra, re = oracle.pathtrace_f64(hv.nodes, hv.root, s.params, d_image.cpu().numpy().astype(np.float64))
    g = np.concatenate([da.cpu().numpy().astype(np.float64).ravel(), de.cpu().numpy().astype(np.float64).ravel()])
    r = np.concatenate([ra.ravel(), re.ravel()])
    assert np.abs(r).max() > 0
    scale = np.maximum(np.abs(r), 1e-3 * np.abs(r).max())
    assert (np.abs(g - r) <= 1e-4 * scale).all(), np.abs((g - r) / scale).max()
    dv.free()
