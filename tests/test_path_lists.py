"""The path tracer's lists in parts (pathtrace.hip: camera pass, bounce walks dealt part by part) at the
sizes where they change: one path, part-full waves and groups, exactly one group, 64 groups of paths and
one more, no bounce at all. The render equals the one-kernel form bit for bit, which shares no list with
it, and the gradient that of a launch shaped by the caller, which keeps one list."""
import numpy as np
import pytest

from cubiquity_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp,bounces", [
    (1, 1, 1, 2), (9, 7, 1, 3), (13, 5, 1, 0), (64, 64, 1, 1), (241, 17, 1, 4), (512, 512, 1, 2), (641, 411, 1, 3),
    (320, 180, 19, 2),
])
def test_lists_equal_other_forms(cq, gpu_ctx, width, height, spp, bounces):
    hv = cq.HostVolume.generate(cq.gen_default_params(7, 1, n_materials=9))
    dv = gpu_ctx.upload(hv)
    alb, em = cq.material_table(9, 5)
    cam = W._camera(7, width, height)
    s = cq.PathTraceSetup(cam, width, height, spp, bounces, alb, em)
    lists = cq.pathtrace(gpu_ctx, dv, s, 0).cpu().numpy()
    one = cq.pathtrace(gpu_ctx, dv, s, 1).cpu().numpy()
    assert np.array_equal(lists.view(np.uint32), one.view(np.uint32)), (lists != one).sum()
    d_image = (2 * cq.pathtrace(gpu_ctx, dv, s, 0).double() - 0.1).float()
    open_ = [t.cpu().numpy() for t in cq.pathtrace_adjoint(gpu_ctx, dv, s, d_image)]
    shaped = cq.LaunchCfg()
    shaped.variant = 2
    other = [t.cpu().numpy() for t in cq.pathtrace_adjoint(gpu_ctx, dv, s, d_image, cfg=shaped)]
    for a, b in zip(open_, other):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    dv.free()
