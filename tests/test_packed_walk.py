"""The packed walk (cubiquity_amd/csrc/walk_packed.h) compiled for the host: every record equals the
oracle's, with the plain rays' step and with the general one, over level-of-detail cut-offs of every
sign, iteration caps, rays with zero, tiny and huge components, exact ties, small and degenerate
volumes, and volumes at the coordinate limit."""
import os
import subprocess

import numpy as np
import pytest

from tests.conftest import records_equal

EXE = os.path.join(os.path.dirname(__file__), "cpp", "packed_emulation")


def _run(tmp_path, cq, nodes, sub, rays, mode, surf, fp, max_iters=1 << 16):
    if not os.path.exists(EXE):
        from cubiquity_amd import build

        build.build_cpp_checks()
    paths = [str(tmp_path / f) for f in ("n.bin", "s.bin", "r.bin", "o.bin")]
    np.ascontiguousarray(nodes).tofile(paths[0])
    np.ascontiguousarray(sub).tofile(paths[1])
    np.ascontiguousarray(rays, dtype=np.float32).tofile(paths[2])
    r = subprocess.run([EXE, mode, *paths, str(int(surf)), repr(float(fp)), str(max_iters)], check=True, timeout=300,
                       stdout=subprocess.PIPE, text=True)
    return np.fromfile(paths[3], dtype=cq.HIT_DTYPE), int(r.stdout)


def _check(tmp_path, cq, oracle, hv, rays, mode, surf, fp, max_iters=1 << 16):
    sub = oracle.find_subdags(hv.nodes, hv.root)
    got, plain = _run(tmp_path, cq, hv.nodes, sub, rays, mode, surf, fp, max_iters)
    ref = oracle.intersect(hv.nodes, sub, rays, surf, fp, max_iters=max_iters, threads=8)
    eq = records_equal(got, ref)
    assert eq.all(), f"{mode} surf={surf} fp={fp}: {(~eq).sum()} of {len(eq)} differ, first {np.nonzero(~eq)[0][:4]}"
    return plain


def _odd_rays(rays):
    """Rays with scaled directions, huge and tiny components, NaN and infinities."""
    out = []
    for k, f in enumerate((1e-30, 1e-19, 3e-18, 1e-3, 7.5, 1e17, 3e18, 1e30)):
        r = rays[k::64][:64].astype(np.float64).copy()
        r[:, 3:] *= f
        out.append(r)
    r = rays[5::64][:64].astype(np.float64).copy()
    r[:16, 3] = 1e-20
    r[16:24, 0] = 1e18
    r[24:32, 1] = np.nan
    r[32:40, 5] = np.inf
    r[40:48, :3] = np.round(r[40:48, :3]) - 0.5
    r[48:56, :3] = -0.5 + 1e-7 * np.arange(8)[:, None]
    out.append(r)
    with np.errstate(over="ignore"):
        return np.concatenate(out).astype(np.float32)


@pytest.mark.parametrize("mode", ["plain", "any"])
def test_packed_walk_matches_oracle(tmp_path, cq, oracle, vol128, rays128, mode):
    from tests.raysets import lattice_rays

    rays = np.concatenate([rays128["camera"][::7], rays128["incoherent"][::2], rays128["special"],
                           lattice_rays(128, 4096, 3), _odd_rays(rays128["camera"])])
    for surf, fp in ((True, -1.0), (False, -1.0), (True, 0.05), (True, 0.0035), (False, 0.3), (True, 2.0), (True, 0.0),
                     (True, -0.5), (True, -3.0), (True, float("inf")), (True, 1e-38), (True, 3e38)):
        plain = _check(tmp_path, cq, oracle, vol128, rays, mode, surf, fp)
        assert mode == "any" or plain > len(rays) // 2


def test_packed_walk_iteration_cap(tmp_path, cq, oracle, vol128, rays128):
    for cap in (1, 2, 3, 5, 16, 17):
        _check(tmp_path, cq, oracle, vol128, rays128["camera"][30720:32768], "plain", True, -1.0, cap)


@pytest.mark.parametrize("mode", ["plain", "any"])
def test_packed_walk_small_and_degenerate_volumes(tmp_path, cq, oracle, mode):
    from tests.raysets import special_rays
    from tests.test_gpu_parity import _small_volumes
    from tests.test_oracle_pinning import _brute_rays

    for name, (hv, n, lower) in _small_volumes(cq).items():
        sp = special_rays(n)
        sp[:, :3] += np.asarray(lower, np.float32)
        rays = np.concatenate([_brute_rays(n, lower, 3000, 17), sp]).astype(np.float32)
        for fp in (-1.0, 0.05):
            _check(tmp_path, cq, oracle, hv, rays, mode, True, fp)


@pytest.mark.parametrize("mode", ["plain", "any"])
def test_packed_walk_deep_volumes(tmp_path, cq, oracle, mode):
    """SubDAGs of 21 and 22 levels, corners out to the 2^22 limit."""
    from tests.raysets import deep_volumes

    for name, (hv, rays) in deep_volumes(cq).items():
        for fp in (-1.0, 0.01):
            _check(tmp_path, cq, oracle, hv, rays, mode, True, fp)


def test_packed_walk_refuses_volumes_past_its_limits(tmp_path, cq, oracle):
    hv = cq.HostVolume.from_dense(np.zeros((4, 4, 4), np.uint8), (0, 0, 0))
    hv.edit_spheres([[1 << 22, 3, 3, 4, 2], [5, 5, 5, 4, 3]])
    sub = oracle.find_subdags(hv.nodes, hv.root)
    with pytest.raises(subprocess.CalledProcessError) as e:
        _run(tmp_path, cq, hv.nodes, sub, np.zeros((1, 6), np.float32), "plain", True, -1.0)
    assert e.value.returncode == 6


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 63, 65, 4097, 8193, 16385, 65537, 131073, (1 << 20) - 1, (1 << 20) + 1, 2621440,
                               2621441, (1 << 23) + 63])
@pytest.mark.parametrize("kind", ["incoherent", "camera"])
def test_open_launch_shapes(cq, oracle, gpu_ctx, vol128, n, kind):
    """The library's launches at the sizes where they change (rays per wave, dealt runs, sampled
    coherence, persistent waves): every record equals the raw store's walk, the small ones the oracle."""
    import torch

    if kind == "camera":
        from cubiquity_amd import workloads as W

        c, side = W.RAYCAST_128.camera, int(np.ceil(np.sqrt(n)))
        rays = cq.camera_rays(c.eye, c.target, c.fov_y, side, side)[:n]
    else:
        rays = cq.incoherent_rays(vol128, 7, 5 + n, n)
    dv = gpu_ctx.upload(vol128)
    r = torch.from_numpy(np.ascontiguousarray(rays)).cuda()
    for surf, fp in ((True, -1.0), (False, 0.0035)):
        got = cq.intersectVolume(gpu_ctx, dv, r, surf, fp)
        raw = cq.intersectVolume(gpu_ctx, dv, r, surf, fp, cfg=cq.LaunchCfg(variant=3))
        assert torch.equal(got, raw), int((got != raw).any(dim=1).sum())
        if n <= 70000:
            ref = oracle.intersect(vol128.nodes, oracle.find_subdags(vol128.nodes, vol128.root), rays, surf, fp, threads=8)
            assert records_equal(got.cpu().numpy().view(cq.HIT_DTYPE).reshape(-1), ref).all()
    dv.free()


@pytest.mark.gpu
def test_gpu_volumes_past_the_packed_limits(cq, oracle, gpu_ctx):
    """A volume whose corners lie past 2^22 takes the raw walk, alone and in a batch with one that
    does not, and comes back to the packed one after an undo on the device."""
    import torch

    rng = np.random.Generator(np.random.PCG64(3))
    near = [[20.0 * i, 3.0, 5.0 * i, 4.0, 1 + i % 3] for i in range(16)]
    far = [[float(1 << 22) + 50.0, 3.0, 3.0, 4.0, 2]] + near[1:]
    hv = cq.HostVolume.from_dense(np.ones((4, 4, 4), np.uint8), (0, 0, 0))
    dv = gpu_ctx.upload(hv)
    dv.edit_spheres(near)
    dv.checkpoint()
    o = rng.uniform(-40.0, 400.0, (5000, 3))
    d = rng.normal(size=(5000, 3))
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    r = torch.from_numpy(rays).cuda()

    def check():
        nodes = dv.download()
        ref = oracle.intersect(nodes, oracle.find_subdags(nodes, dv.root), rays, True, threads=8)
        hits = torch.zeros((5000, 32), dtype=torch.uint8, device="cuda")
        cq.intersect_batched(gpu_ctx, [(dv, r, hits, True, -1.0)])
        for got in (cq.intersectVolume(gpu_ctx, dv, r), hits):
            assert records_equal(got.cpu().numpy().view(cq.HIT_DTYPE).reshape(-1), ref).all()

    check()
    dv.edit_spheres(far)
    check()
    dv.undo()
    check()
    dv.free()


@pytest.mark.gpu
@pytest.mark.parametrize("batches,n", [(1, 1), (3, 0), (40, 777), (41, 777), (40, 110000)])
def test_batched_launch_shapes(cq, gpu_ctx, vol128, rays128, batches, n):
    """Descriptors in the kernel's arguments and in a table, dealt and claimed ids, empty batches: every
    record equals the batch's own launch over the raw store."""
    import torch

    dv = gpu_ctx.upload(vol128)
    rays = torch.from_numpy(np.concatenate([rays128["incoherent"], rays128["camera"]])).cuda()
    items = []
    for i in range(batches):
        m = 0 if n and i % 5 == 4 else n + 7 * i
        r = rays.roll(i * 911, 0).repeat((m + len(rays) - 1) // len(rays), 1)[:m] if m else rays[:0]
        hits = torch.zeros((max(1, m), 32), dtype=torch.uint8, device="cuda")
        items.append((dv, r.contiguous(), hits, i % 2 == 0, 0.0035 if i % 3 == 2 else -1.0))
    cq.intersect_batched(gpu_ctx, items)
    for i, (v, r, hits, surf, fp) in enumerate(items):
        if len(r):
            raw = cq.intersectVolume(gpu_ctx, v, r, surf, fp, cfg=cq.LaunchCfg(variant=3))
            assert torch.equal(hits[: len(r)], raw), i
    dv.free()
