"""The packed copy of a node store against the store it is made from: stores with unchecked words, and
the calls that change a store under its copy."""
import os
import subprocess

import numpy as np
import pytest

from tests.conftest import ROOT, records_equal


def _with_unreached(nodes):
    """The store with nodes that nothing refers to, whose words are past it in every way."""
    n = len(nodes)
    bad = np.array([[n + 3, n + 4, 1 << 24, (1 << 24) + 300, 1 << 27, 1 << 31, 0xfffffffe, 0xffffffff]] * 3, np.uint32)
    bad[1] = 0
    return np.concatenate([nodes, bad])


def test_packing_reads_inside_the_store(tmp_path, vol128):
    """Nodes that no root reaches are packed too: their children's indices are not checked at upload."""
    exe = str(tmp_path / "pack_check")
    inc = [f"-I{os.path.join(ROOT, d)}" for d in ("tests/cpp/host_shim", "include", "cubiquity_amd/csrc")]
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address", *inc,
                    os.path.join(ROOT, "tests/cpp/pack_check.cpp"), "-o", exe], check=True)
    nodes = _with_unreached(vol128.nodes)
    nodes.tofile(tmp_path / "n.bin")
    subprocess.run([exe, str(tmp_path / "n.bin"), str(tmp_path / "p.bin")], check=True, timeout=120)
    got = np.fromfile(tmp_path / "p.bin", np.uint32).reshape(-1, 8)
    mask = ((nodes != 0) << np.arange(8)).sum(axis=1).astype(np.uint64)
    kept = nodes.astype(np.uint64) < len(nodes)
    child = np.where(kept, nodes, 0)
    assert np.array_equal(got, np.where(child != 0, (child.astype(np.uint64) << 8) | mask[child], 0))


@pytest.mark.gpu
def test_gpu_store_with_unreached_nodes(cq, oracle, gpu_ctx, vol128, rays128):
    import torch

    nodes = _with_unreached(vol128.nodes)
    hv = cq.HostVolume.from_nodes(nodes, vol128.root)
    dv = gpu_ctx.upload(hv)
    rays = torch.from_numpy(rays128["incoherent"]).cuda()
    ref = oracle.intersect(nodes, oracle.find_subdags(nodes, hv.root), rays128["incoherent"], True, threads=8)
    got = cq.intersectVolume(gpu_ctx, dv, rays).cpu().numpy().view(cq.HIT_DTYPE).reshape(-1)
    assert records_equal(got, ref).all()
    dv.free()


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [0.02, 0.5, 0.9])
def test_gpu_update_that_replaces_uploaded_nodes(cq, oracle, gpu_ctx, vol128, rays128, keep):
    """An update may replace the tail of the uploaded store, whose earlier nodes have children there
    (a baked store holds parents first): the masks kept with those nodes' words follow. Then the store is
    cut short of its upload, and extended again."""
    import torch

    nodes, n = vol128.nodes.copy(), len(vol128.nodes)
    first = 256 + int(keep * (n - 256))
    assert (nodes[256:first] >= first).any() and vol128.root < first
    dv = gpu_ctx.upload(vol128)
    rays = torch.from_numpy(rays128["incoherent"]).cuda()

    def check(stored):
        ref = oracle.intersect(stored, oracle.find_subdags(stored, vol128.root), rays128["incoherent"], True, threads=8)
        got = cq.intersectVolume(gpu_ctx, dv, rays).cpu().numpy().view(cq.HIT_DTYPE).reshape(-1)
        eq = records_equal(got, ref)
        assert eq.all(), int((~eq).sum())

    check(nodes)
    rng = np.random.Generator(np.random.PCG64(int(100 * keep)))
    fresh = rng.integers(1, 256, (n - first, 8)).astype(np.uint32)  # materials: any node may have them as children
    fresh[rng.random(fresh.shape) < 0.6] = 0
    fresh[:, 0] = np.maximum(fresh[:, 0], 1)
    nodes[first:] = fresh
    dv.update(cq.HostVolume.from_nodes(nodes, vol128.root), first)
    check(nodes)
    tail = nodes[first:].copy()
    tail[:, 3] = 7
    nodes[first:] = tail
    nodes = np.concatenate([nodes, tail[:50]])
    dv.update(cq.HostVolume.from_nodes(nodes, vol128.root), first)
    check(nodes)
    dv.update(cq.HostVolume.from_nodes(nodes[:first], 3), first)  # the whole space material 3
    assert (cq.intersectVolume(gpu_ctx, dv, rays).cpu().numpy().view(cq.HIT_DTYPE)["info"] >> 16 == 3).all()
    dv.update(cq.HostVolume.from_nodes(nodes, vol128.root), first)
    check(nodes)
    dv.free()


@pytest.mark.gpu
@pytest.mark.parametrize("back", ["undo", "redo", "update", "edit"])
def test_gpu_copy_that_returns_is_whole(cq, oracle, gpu_ctx, rays128, monkeypatch, back):
    """A copy that cannot be had is left out, and made whole by whichever later call can have it: what
    other streams launch right after that call reads no word still to be packed."""
    import torch

    hv = cq.HostVolume.generate(cq.gen_default_params(9, 3))
    rays = cq.incoherent_rays(hv, 9, 11, 20000)
    side = torch.cuda.Stream()  # does not wait for the null stream
    r, hits = torch.from_numpy(rays).cuda(), torch.zeros((len(rays), 32), dtype=torch.uint8, device="cuda")
    spheres = [[20.0 * i, 250.0, 9.0 * i, 6.0, 1 + i % 5] for i in range(20)]
    monkeypatch.setenv("CQX_PACKED_NODES", "0")
    dv = gpu_ctx.upload(hv)
    dv.checkpoint()
    dv.edit_spheres(spheres)
    if back == "redo":
        dv.undo()
    elif back == "update":
        hv = cq.HostVolume.from_nodes(dv.download(), dv.root)
    torch.cuda.synchronize()
    monkeypatch.delenv("CQX_PACKED_NODES")
    {"undo": dv.undo, "redo": dv.redo, "update": lambda: dv.update(hv, dv.node_count),
     "edit": lambda: dv.edit_spheres(spheres)}[back]()
    cq.intersectVolume(gpu_ctx, dv, r, out=hits, stream=side.cuda_stream)
    side.synchronize()
    nodes = dv.download()
    ref = oracle.intersect(nodes, oracle.find_subdags(nodes, dv.root), rays, True, threads=8)
    assert records_equal(hits.cpu().numpy().view(cq.HIT_DTYPE).reshape(-1), ref).all()
    dv.free()


@pytest.mark.gpu
def test_gpu_copy_after_an_edit_that_fails_late(cq, oracle, gpu_ctx, vol128, rays128):
    """An edit of a store whose root is on a chain deeper than the tree (accepted by an update that
    brings its SubDAGs) fails once its nodes are in the store and the index. Later edits share those
    nodes: the copy has them."""
    import ctypes

    import torch

    nodes = vol128.nodes
    n, chain = len(nodes), np.zeros((40, 8), np.uint32)
    chain[0, 0] = 9
    chain[1:, 0] = np.arange(n, n + 39)  # the octant of the lowest coordinates, far from the edits
    deep = np.ascontiguousarray(np.concatenate([nodes, chain]))
    sub = np.ascontiguousarray(oracle.find_subdags(nodes, vol128.root))
    dv = gpu_ctx.upload(vol128)
    cq.cabi.check(cq.cabi.lib().cqx_volume_update(
        gpu_ctx._h, dv._h, deep.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), ctypes.c_uint64(len(deep)),
        ctypes.c_uint64(n), ctypes.c_uint32(len(deep) - 1), sub.ctypes.data_as(ctypes.c_void_p)))
    spheres = [[300.0 + 3 * i, 300.0 + i, 300.0, 3.0, 3] for i in range(16)]  # in empty space under either root
    with pytest.raises(cq.CqxError):
        dv.edit_spheres(spheres)
    dv._refresh()
    held = dv.node_count
    assert held > len(deep)
    dv.update(cq.HostVolume.from_nodes(dv.download(), vol128.root), held)
    rays = rays128["incoherent"].copy()
    aim = np.array(spheres, np.float32)[np.arange(8000) % 16, :3] - rays[:8000, :3]
    rays[:8000, 3:] = aim / np.linalg.norm(aim, axis=1, keepdims=True)
    r = torch.from_numpy(rays).cuda()
    for hit in (False, True):
        stored = dv.download()
        ref = oracle.intersect(stored, oracle.find_subdags(stored, dv.root), rays, True, threads=8)
        got = cq.intersectVolume(gpu_ctx, dv, r).cpu().numpy().view(cq.HIT_DTYPE).reshape(-1)
        assert records_equal(got, ref).all() and (got["voxel"][:8000, 0] > 290).any() == hit
        dv.edit_spheres(spheres)
        assert ((dv.download(held) >= len(deep)) & (dv.download(held) < held)).any()
    dv.free()


@pytest.mark.gpu
def test_gpu_upload_keeps_the_path_tracers_plan(cq, gpu_ctx, vol128):
    """Uploading one volume while another is rendered: the renderer's plan (buffers and graph, a third of a
    gigabyte here) is not made again for the next frame."""
    import torch

    from cubiquity_amd import workloads as W

    dv = gpu_ctx.upload(vol128)
    setup = cq.PathTraceSetup(W.RAYCAST_128.camera, 640, 480, 8, 2, *cq.material_table(9, 11))
    image = cq.pathtrace(gpu_ctx, dv, setup)
    free = torch.cuda.mem_get_info()[0]
    other = gpu_ctx.upload(cq.HostVolume.from_dense(np.ones((4, 4, 4), np.uint8)))
    assert torch.cuda.mem_get_info()[0] <= free
    assert torch.equal(cq.pathtrace(gpu_ctx, dv, setup), image)
    other.free()
    dv.free()


@pytest.mark.gpu
def test_gpu_path_tracer_follows_the_copy(cq, gpu_ctx, monkeypatch):
    """One image shape rendered, and its adjoint taken, while the volume's copy grows, is given up past the
    coordinate limit, cannot be had, and returns: each frame equals the megakernel's (which walks the raw
    store), each gradient that of a fresh context."""
    import torch

    from cubiquity_amd import workloads as W

    cam = W.Camera((60.0, 90.0, -120.0), (150.0, 0.0, 40.0), 70.0, 96, 64)
    setup = cq.PathTraceSetup(cam, 96, 64, 4, 3, *cq.material_table(5, 11))
    d_image = torch.rand((64, 96, 3), device="cuda")
    hv = cq.HostVolume.from_dense(np.ones((4, 4, 4), np.uint8), (0, 0, 0))
    dv = gpu_ctx.upload(hv)
    near = [[20.0 * i, 3.0, 5.0 * i, 8.0, 1 + i % 5] for i in range(16)]

    def check():
        image = cq.pathtrace(gpu_ctx, dv, setup)
        got = cq.pathtrace_adjoint(gpu_ctx, dv, setup, d_image)
        assert torch.equal(image, cq.pathtrace(gpu_ctx, dv, setup, mode=1))
        ctx = cq.Context(0)
        fresh = ctx.upload(cq.HostVolume.from_nodes(dv.download(), dv.root))
        ref = cq.pathtrace_adjoint(ctx, fresh, setup, d_image)
        fresh.free()
        ctx.close()
        assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])
        return image

    images = [check()]
    dv.edit_spheres(near)  # grows the store past its copy
    images.append(check())
    dv.checkpoint()
    dv.edit_spheres([[float(1 << 22) + 50.0, 3.0, 3.0, 4.0, 2]] + near[1:])
    check()
    monkeypatch.setenv("CQX_PACKED_NODES", "0")
    dv.undo()
    images.append(check())
    monkeypatch.delenv("CQX_PACKED_NODES")
    dv.redo()
    dv.undo()
    images.append(check())
    grown = [[20.0 * i, 40.0, 4.0 * i, 5.0 + 0.1 * i, 1 + i % 5] for i in range(40)]
    dv.edit_spheres(grown)
    images.append(check())
    assert torch.equal(images[1], images[2]) and torch.equal(images[1], images[3])
    assert not torch.equal(images[0], images[1]) and not torch.equal(images[1], images[4])
    dv.free()
