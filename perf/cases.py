"""Timed cases: the calls a program makes on this framework, over the sizes it makes them at.

Every case is one pass through the package's public entry points on a volume resident in HBM, with
the launch left at "auto" as in the entry points' defaults. The volumes are the generator's fBm
terrain with spheres (the benchmark's family); rays, cameras, random seeds, brush spheres and
output gradients are the inputs that change with `seed`. Coordinates follow the benchmark: the
volume of side N = 2^log2 occupies [-0.5, N - 0.5)^3.

Kinds of case:
  host        Context.intersect_host: rays from and records to host arrays (picking, line-of-sight
              and collision queries of an application; a few to a few thousand rays)
  incoherent  intersectVolume on uniform origins and directions (ambient occlusion, secondary rays,
              sampling); from one wave's worth of rays to the benchmark's 2^24
  camera      intersectVolume on a pinhole camera's primary rays, with or without the
              level-of-detail cut-off
  batched     intersect_batched: several volumes (objects of a scene, many tenants), each with a ray
              array of its own size, in one launch
  pathtrace   pathtrace: a whole frame
  adjoint     pathtrace_adjoint: gradients of the material tables for a given image gradient
  demo        demo_trace: a frame of the reference CPU tracer's shading
  edit        an interactive brush frame: checkpoint, edit_spheres on the device, the frame's
              primary rays against the edited volume, undo
"""
import functools

import numpy as np
import torch

import cubiquity_amd as cq
from cubiquity_amd import workloads as W


def listed():
    return [
        # an application's handful of line-of-sight queries in one frame, on a small world
        dict(name="host_97", kind="host", log2=7, n=97),
        # a few waves of device-resident query rays: launch latency and one ray's walk decide
        dict(name="incoherent_1021", kind="incoherent", log2=9, n=1021, surf=True, lod=-1.0),
        # the parity suite's 256 x 256 camera on its 128^3 volume
        dict(name="camera_128", kind="camera", log2=7, width=256, height=256, surf=True, lod=-1.0),
        # a viewer's primary rays with the reference demo's level-of-detail cut-off
        dict(name="camera_1024_lod", kind="camera", log2=10, width=1280, height=720, surf=True, lod=0.0035),
        # the benchmark: 2^24 incoherent rays on the 1024^3 volume
        dict(name="incoherent_1024", kind="incoherent", log2=10, n=1 << 24, surf=True, lod=-1.0),
        # occlusion-only rays (no surface properties) on a store larger than the last-level cache
        dict(name="occlusion_4096", kind="incoherent", log2=12, n=4000003, surf=False, lod=-1.0),
        # two dozen objects of 64^3 to 512^3, ray counts log-uniform from 1e3 to 4e5
        dict(name="batched_24", kind="batched", volumes=24, log2_min=6, log2_max=9, n_min=1000, n_max=400000),
        # a viewer's quick preview: one sample, two bounces, a small volume
        dict(name="pathtrace_preview", kind="pathtrace", log2=7, width=320, height=180, spp=1, bounces=2),
        # the benchmark's frame
        dict(name="pathtrace_1024", kind="pathtrace", log2=10, width=1280, height=720, spp=16, bounces=4),
        # the differentiable-rendering workload: 16 materials, 512 x 512, 8 samples, 3 bounces
        dict(name="adjoint_512", kind="adjoint", log2=9, width=512, height=512, spp=8, bounces=3, materials=16),
        # the reference tracer's shading, one frame of its viewer
        dict(name="demo_1024", kind="demo", log2=10, width=1280, height=720, lod=0.0035, noise=True),
        # the edit workload: 1000 brush spheres in a 2048^3 volume, then the frame's primary rays
        dict(name="edit_2048", kind="edit", log2=11, spheres=1000, width=640, height=360),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))))


def _frame_size(rng, w_lo, w_hi):
    """A width in [w_lo, w_hi] (log-uniform, odd ones among them) and a height of a usual aspect."""
    w = _log_int(rng, w_lo, w_hi)
    return w, max(1, int(w / rng.uniform(1.0, 1.8)))


def draw(rng):
    kind = rng.choice(["host", "incoherent", "camera", "batched", "pathtrace", "adjoint", "demo", "edit"])
    if kind == "host":
        return dict(kind=kind, log2=rng.randint(6, 10), n=_log_int(rng, 1, 4096))
    if kind == "incoherent":
        return dict(kind=kind, log2=rng.randint(7, 11), n=_log_int(rng, 64, 1 << 23), surf=rng.random() < 0.6,
                    lod=rng.choice([-1.0, -1.0, 0.0035]))
    if kind == "camera":
        w, h = _frame_size(rng, 128, 1920)
        return dict(kind=kind, log2=rng.randint(7, 11), width=w, height=h, surf=rng.random() < 0.8,
                    lod=rng.choice([-1.0, 0.0035]))
    if kind == "batched":
        hi = rng.randint(7, 9)
        return dict(kind=kind, volumes=rng.randint(2, 32), log2_min=6, log2_max=hi, n_min=_log_int(rng, 100, 2000),
                    n_max=_log_int(rng, 10000, 400000))
    if kind == "pathtrace":
        w, h = _frame_size(rng, 96, 1280)
        return dict(kind=kind, log2=rng.randint(7, 10), width=w, height=h, spp=rng.choice([1, 2, 3, 4, 8, 16]),
                    bounces=rng.randint(1, 4))
    if kind == "adjoint":
        w, h = _frame_size(rng, 64, 512)
        return dict(kind=kind, log2=rng.randint(7, 9), width=w, height=h, spp=rng.choice([1, 2, 4, 5, 8]),
                    bounces=rng.randint(1, 4), materials=rng.choice([4, 9, 16, 40]))
    if kind == "demo":
        w, h = _frame_size(rng, 160, 1280)
        return dict(kind=kind, log2=rng.randint(7, 10), width=w, height=h, lod=rng.choice([-1.0, 0.0035]),
                    noise=rng.random() < 0.7)
    w, h = _frame_size(rng, 160, 640)
    return dict(kind=kind, log2=rng.randint(8, 11), spheres=_log_int(rng, 32, 1000), width=w, height=h)


# ---- inputs -----------------------------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _volume(log2, scene, materials):
    """The generator's volume. The scene stands for the case; the seed moves what is done to it."""
    return cq.HostVolume.generate(cq.gen_default_params(log2, scene, n_materials=materials))


def _camera(log2, rng, width, height):
    """The benchmark's view of the terrain, moved a little by the seed."""
    s = (1 << log2) / 128.0
    j = rng.uniform(-6.0, 6.0, 6)
    eye = tuple(float(s * v) for v in (64.0 + j[0], 150.0 + j[1], -100.0 + j[2]))
    target = tuple(float(s * v) for v in (64.0 + j[3], 40.0 + 0.5 * j[4], 64.0 + j[5]))
    return W.Camera(eye, target, 60.0, width, height)


def _camera_rays(cam):
    return cq.camera_rays(cam.eye, cam.target, cam.fov_y, cam.width, cam.height)


def _gpu(array):
    return torch.from_numpy(np.ascontiguousarray(array)).cuda()


def _hits(n):
    return torch.empty((n, 32), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    kind = case["kind"]
    ctx = cq.Context(0)
    st = dict(case=case, ctx=ctx)
    if kind == "batched":
        items = []
        for i in range(case["volumes"]):
            log2 = case["log2_min"] + i % (case["log2_max"] - case["log2_min"] + 1)
            hv = _volume(log2, 100 + i, 3)
            n = int(round(float(np.exp(np.random.Generator(np.random.PCG64(42 + i)).uniform(
                np.log(case["n_min"]), np.log(case["n_max"]))))))
            if i % 2 == 0:  # camera rays and incoherent rays in turn, as in the benchmark's batches
                side = int(np.ceil(np.sqrt(n)))
                rays = _camera_rays(_camera(log2, rng, side, side))[:n]
            else:
                rays = cq.incoherent_rays(hv, log2, seed * 64 + i, n)
            items.append((ctx.upload(hv), _gpu(rays), _hits(n), True, -1.0))
        st["items"] = items
        return st
    log2 = case["log2"]
    materials = case.get("materials", 16 if kind == "edit" else 9)
    hv = _volume(log2, 21 if kind == "edit" else 1, materials)
    st["vol"] = ctx.upload(hv)
    if kind == "host":
        st["rays"] = cq.incoherent_rays(hv, log2, seed, case["n"])
    elif kind == "incoherent":
        st["rays"] = _gpu(cq.incoherent_rays(hv, log2, seed, case["n"]))
        st["out"] = _hits(case["n"])
    elif kind in ("camera", "demo", "edit"):
        st["rays"] = _gpu(_camera_rays(_camera(log2, rng, case["width"], case["height"])))
        n = case["width"] * case["height"]
        if kind == "demo":
            alb, em = cq.material_table(materials, 11)
            st["colours"] = cq.Materials.from_tables(alb, em).colour_table()
            st["out"] = torch.empty((n, 3), dtype=torch.float32, device="cuda")
            st["seed"] = seed
        else:
            st["out"] = _hits(n)
        if kind == "edit":
            # centre uniform in the volume, radius U[2, 16] (N / 2048)^(1/3), material 0 (carve) to 16
            side = float(1 << log2)
            e = np.zeros((case["spheres"], 5))
            e[:, :3] = rng.uniform(0.0, side, (case["spheres"], 3))
            e[:, 3] = rng.uniform(2.0, 16.0, case["spheres"]) * (side / 2048.0) ** (1.0 / 3.0)
            e[:, 4] = rng.integers(0, materials + 1, case["spheres"])
            st["edits"] = e
    else:  # pathtrace, adjoint
        alb, em = cq.material_table(materials, 11)
        cam = _camera(log2, rng, case["width"], case["height"])
        st["setup"] = cq.PathTraceSetup(cam, case["width"], case["height"], case["spp"], case["bounces"], alb, em,
                                        seed=seed & 0xffffffff)
        if kind == "adjoint":  # the gradient of a mean-square loss against some target image
            g = rng.normal(size=(case["height"], case["width"], 3)) * (2.0 / (case["height"] * case["width"] * 3))
            st["d_image"] = _gpu(g.astype(np.float32))
        else:
            st["out"] = torch.empty((case["height"], case["width"], 3), dtype=torch.float32, device="cuda")
    return st


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "host":
        return ctx.intersect_host(state["vol"], state["rays"]).view(np.uint8)
    if kind in ("incoherent", "camera"):
        return cq.intersectVolume(ctx, state["vol"], state["rays"], case["surf"], case["lod"], out=state["out"])
    if kind == "batched":
        cq.intersect_batched(ctx, state["items"])
        return [it[2] for it in state["items"]]
    if kind == "pathtrace":
        return cq.pathtrace(ctx, state["vol"], state["setup"], out=state["out"])
    if kind == "adjoint":
        return list(cq.pathtrace_adjoint(ctx, state["vol"], state["setup"], state["d_image"]))
    if kind == "demo":
        return cq.demo_trace(ctx, state["vol"], state["rays"], state["colours"], case["lod"], add_noise=case["noise"],
                             seed=state["seed"], out=state["out"])
    vol = state["vol"]
    vol.checkpoint()
    vol.edit_spheres(state["edits"])
    hits = cq.intersectVolume(ctx, vol, state["rays"], out=state["out"])
    root = vol.root
    vol.undo()
    return [hits, root]


# ---- what a pass cannot do without ------------------------------------------------------------------

# Measured on the benchmark volume's rays: walk steps per ray grow with the depth (about 4 per level),
# each about 12 additions, multiplications and comparisons in FP32; about 3 node entries per level.
_STEP_FLOPS = 12


def _store_bytes(log2):
    """The node store of the generator's volume: about 0.6 nodes per column of voxels, 32 bytes each."""
    return 0.6 * 4.0 ** log2 * 32


def _walk(log2, n):
    """(store bytes that n rays read once, flops) of n rays: they touch at most the whole store, and
    at most the nodes they enter."""
    return min(_store_bytes(log2), n * 3.0 * log2 * 32), n * 4.0 * log2 * _STEP_FLOPS


def work(case):
    kind = case["kind"]
    if kind == "batched":
        b = f = 0.0
        for i in range(case["volumes"]):
            log2 = case["log2_min"] + i % (case["log2_max"] - case["log2_min"] + 1)
            n = float(np.exp(np.random.Generator(np.random.PCG64(42 + i)).uniform(np.log(case["n_min"]),
                                                                                 np.log(case["n_max"]))))
            wb, wf = _walk(log2, n)
            b += n * 56 + wb
            f += wf
        return {"bytes": b, "flops": f}
    log2 = case["log2"]
    if kind in ("host", "incoherent"):
        wb, wf = _walk(log2, case["n"])
        return {"bytes": case["n"] * 56 + wb, "flops": wf}
    pixels = case["width"] * case["height"]
    if kind == "camera":
        wb, wf = _walk(log2, pixels)
        return {"bytes": pixels * 56 + wb, "flops": wf}
    if kind == "edit":
        # the rays and their records, and the nodes on the spheres' surfaces read and written once
        wb, wf = _walk(log2, pixels)
        radius = 9.0 * (2.0 ** log2 / 2048.0) ** (1.0 / 3.0)
        nodes = case["spheres"] * 4.0 * np.pi * radius ** 2
        return {"bytes": pixels * 56 + wb + nodes * 64, "flops": wf + nodes * 8 * 20}
    if kind == "demo":
        wb, wf = _walk(log2, pixels * 4.0)  # primary, two shadow rays, reflection on most pixels
        return {"bytes": pixels * 36 + wb, "flops": wf}
    paths = pixels * case["spp"]
    wb, wf = _walk(log2, paths * (0.5 * case["bounces"] + 1.0))  # about half the paths go on at each bounce
    return {"bytes": pixels * 12 + wb, "flops": wf}


def exact(case, seed):
    """No output here has a 64-bit counterpart. Traversal records are bytes defined by FP32 arithmetic
    operation by operation. The renderers' images and gradients follow from which voxel each FP32
    ray hits: in 64 bits, rays at edges take other voxels and whole paths differ; and tracing the
    same FP32 paths in numpy takes minutes."""
    return None
