"""The on-device edit walk (edits_gpu.hip) at the sizes where it changes: regions of side 32 to 1024
(spheres from single voxels to radius 400), nearly equal spheres on one another (the interning of equal
nodes within one step), carves, and regions that outgrow their slices: the device store equals the
host's region-parallel edits node for node."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2,radius,n,kind", [
    (6, (0.0, 1.5), 400, "voxels"), (7, (2.0, 16.0), 300, "plain"), (7, (5.0, 9.0), 200, "stacked"),
    (8, (60.0, 90.0), 16, "plain"), (8, (20.0, 60.0), 40, "carve"), (9, (200.0, 400.0), 17, "plain"),
    (7, (2.0, 16.0), 200, "slices"), (7, (2.0, 16.0), 200, "far"),
])
def test_device_walk_equals_host(cq, gpu_ctx, monkeypatch, log2, radius, n, kind):
    if kind == "slices":
        monkeypatch.setenv("CQX_EDIT_FIRST_SLICE", "16")
    hv = cq.HostVolume.generate(cq.gen_default_params(log2, 3, n_materials=16))
    dv = gpu_ctx.upload(hv)
    rng = np.random.Generator(np.random.PCG64(log2 * 100 + n))
    side = float(1 << log2)
    for frame in range(2):
        e = np.zeros((n, 5))
        e[:, :3] = rng.uniform(0.0, side, (n, 3))
        e[:, 3] = rng.uniform(*radius, n)
        e[:, 4] = rng.integers(0, 17, n)
        if kind == "stacked":
            e[1:, :3] = e[0, :3] + rng.integers(-3, 4, (n - 1, 3)) * 0.5
        elif kind == "carve":
            e[:, 4] = np.where(rng.random(n) < 0.7, 0, e[:, 4])
        elif kind == "far":
            e[:, :3] -= float((1 << 22) + 17)
        elif kind == "voxels":
            e[::2, :3] = np.round(e[::2, :3])
        assert dv.edit_spheres(e) == hv.edit_spheres(e, threads=8)
        assert (dv.node_count, dv.root) == (hv.node_count, hv.root)
        eq = (dv.download() == hv.nodes).all(axis=1)
        assert eq.all(), f"frame {frame}: {(~eq).sum()} of {len(eq)} nodes differ, first at {np.nonzero(~eq)[0][:5]}"
    dv.free()


@pytest.mark.parametrize("n", [17, 64, 65, 130])
def test_levels_above_equal_regions(cq, gpu_ctx, n):
    """n equal spheres in n parents of regions, in a row through empty space and (every third) one that
    differs: levels of 64 entries and around, whose new nodes are equal in sets."""
    hv = cq.HostVolume.generate(cq.gen_default_params(6, 3, n_materials=16))
    dv = gpu_ctx.upload(hv)
    for frame in range(2):
        e = np.zeros((n, 5))
        e[:, 0] = 64.0 * np.arange(n) + 16.0
        e[:, 1] = -64.0 * (np.arange(n) % 4) + 16.0 + 4096.0 * frame
        e[:, 2] = 1024.0 + 16.0
        e[:, 3] = 6.0
        e[:, 4] = np.where(np.arange(n) % 3 == 2, 9, 5)
        assert dv.edit_spheres(e) == hv.edit_spheres(e, threads=8)
        assert (dv.node_count, dv.root) == (hv.node_count, hv.root)
        assert (dv.download() == hv.nodes).all()
    dv.free()
