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
