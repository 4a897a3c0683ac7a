"""Device edits and updates from the host on one volume: an update may drop or replace nodes that device
edits appended, since only the nodes before it have to be as uploaded."""
import numpy as np
import pytest

from tests.conftest import records_equal
from tests.test_device_edits import _frame

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("replaced", [False, True])
def test_edits_after_an_update_that_drops_edited_nodes(cq, gpu_ctx, replaced):
    """The next edits make the host's store again, node for node: none of the dropped nodes is shared."""
    hv = cq.HostVolume.generate(cq.gen_default_params(7, 3, n_materials=16))
    first = hv.node_count
    dv = gpu_ctx.upload(hv)
    dv.edit_spheres(_frame(7, 0, 1500, "plain"))
    dv.edit_spheres(_frame(7, 1, 300, "plain"))
    dropped = dv.node_count
    if replaced:
        hv.edit_spheres(_frame(7, 2, 40, "plain"), threads=8)
        assert first < hv.node_count < dropped
    dv.update(hv, first)
    for f, n in ((0, 1500), (1, 300), (3, 200)):
        e = _frame(7, f, n, "plain")
        assert dv.edit_spheres(e) == hv.edit_spheres(e, threads=8)
        assert (dv.node_count, dv.root) == (hv.node_count, hv.root)
        assert np.array_equal(dv.download(), hv.nodes)
    dv.free()


def test_undo_to_a_root_that_an_update_cut_off(cq, oracle, gpu_ctx, monkeypatch):
    """The history of a device volume outlives an update that cuts its nodes off: undo shows what they
    held, also where the volume's packed copy was made again meanwhile, and an edit there is refused."""
    import torch

    hv = cq.HostVolume.generate(cq.gen_default_params(7, 3, n_materials=16))
    rays = cq.incoherent_rays(hv, 7, 5, 20000)
    r = torch.from_numpy(rays).cuda()
    dv = gpu_ctx.upload(hv)
    dv.edit_spheres(_frame(7, 0, 1500, "plain"))
    nodes, root = dv.download(), dv.root
    dv.checkpoint()
    dv.edit_spheres(_frame(7, 1, 300, "plain"))
    monkeypatch.setenv("CQX_PACKED_NODES", "0")
    dv.update(hv, hv.node_count)
    monkeypatch.delenv("CQX_PACKED_NODES")
    dv.undo()
    assert dv.root == root >= dv.node_count
    ref = oracle.intersect(nodes, oracle.find_subdags(nodes, root), rays, True, threads=8)
    got = cq.intersectVolume(gpu_ctx, dv, r).cpu().numpy().view(cq.HIT_DTYPE).reshape(-1)
    assert records_equal(got, ref).all()
    with pytest.raises(cq.CqxError):
        dv.edit_spheres(_frame(7, 1, 300, "plain"))
    dv.update(hv, hv.node_count)
    got = cq.intersectVolume(gpu_ctx, dv, r).cpu().numpy().view(cq.HIT_DTYPE).reshape(-1)
    ref = oracle.intersect(hv.nodes, oracle.find_subdags(hv.nodes, hv.root), rays, True, threads=8)
    assert records_equal(got, ref).all()
    dv.free()
