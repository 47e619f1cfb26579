"""Edge selection with one node stack per wave against the breadth-first
selection (one tree level per launch), which expands the same nodes with the
same keyed draws: images and gradients of renders whose point counts sit at
the edges of waves (64 points, halves of 32), of fetches and of the list's
blocks (256), with light and heavy walks (a lobe near 1 splits at most nodes,
which spills the stack), several jobs in one launch, and the learned mixture.
The two runs differ in the order of float sums only: up to 2e-6 of the
gradient's norm between runs of one kind, 1e-5 asked."""
import numpy as np
import pytest

from delta_ray_amd import _abi, workloads
from delta_ray_amd import delta_ray as dr
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _heightfield(grid, res, f0):
    w = workloads.heightfield(grid=grid, resolution=res)
    m = w["materials"][0]
    m.diffuse_reflectance = np.full(3, 0.5 * (1.0 - f0), np.float32)
    m.specular_reflectance = np.full(3, f0, np.float32)
    return w


def _jobs(scenes, spp, nb, flags):
    import torch
    jobs = []
    for k, (sc, (W, H)) in enumerate(scenes):
        g = torch.Generator(device="cuda").manual_seed(k)
        jobs.append(dict(scene=sc, options=dr.DeviceScene.options(W, H, spp, nb, 11 + k, flags),
                         image=torch.empty((H, W, 3), device="cuda"), grads=torch.empty(sc.grad_size, device="cuda"),
                         d_image=torch.randn((H, W, 3), generator=g, device="cuda")))
    return jobs


# image sizes and samples: points (at most) 1, 63, 64, 65, 255, 257, 2049
@pytest.mark.parametrize("size", [(1, 1, 1), (9, 7, 1), (8, 4, 2), (13, 5, 1), (17, 15, 1), (257, 1, 1), (683, 1, 3)])
@pytest.mark.parametrize("f0", [0.32, 0.98])
def test_selection_matches_breadth_first(gpu, size, f0):
    W, H, spp = size
    w = _heightfield(48, (W, H), f0)
    sc = dr.DeviceScene(w["camera"], w["shapes"], w["materials"], w["lights"])
    out = {}
    for refill in (0, 1, 64):
        jobs = _jobs([(sc, (W, H))], spp, 2, _abi.DR_FLAGS_PARITY)
        b = dr.Batch()
        b.set_tuning(1 << 22, 1 << 20, refill)
        b.render(jobs)
        out[refill] = (jobs[0]["image"].cpu().numpy(), jobs[0]["grads"].cpu().numpy())
    for refill in (1, 64):
        assert rel_err(out[refill][0], out[0][0]) < 1e-6
        assert rel_err(out[refill][1], out[0][1]) < 1e-5


@pytest.mark.parametrize("learned", [False, True])
def test_selection_of_mixed_jobs(gpu, learned):
    """jobs of different scenes, one of them tiny, in one launch"""
    sizes = [(3, 3), (40, 21), (1, 1), (33, 32)]
    scenes = []
    for k, (W, H) in enumerate(sizes):
        w = workloads.shadow(resolution=(W, H), light_intensity=1000.0) if k == 1 else \
            _heightfield(20 + 9 * k, (W, H), 0.9)
        sc = dr.DeviceScene(w["camera"], w["shapes"], w["materials"], w["lights"])
        if learned:
            n = int(sc.lib.dr_scene_edge_count(sc.handle))
            wt = np.exp(np.random.default_rng(k).normal(size=n)).astype(np.float32)
            _abi.check(sc.lib, sc.lib.dr_scene_set_edge_weights(sc.handle, wt.ctypes.data), "weights")
        scenes.append((sc, (W, H)))
    flags = _abi.DR_LEARNED_EDGES if learned else 0
    out = {}
    for refill in (0, 64):
        jobs = _jobs(scenes, 3, 3, flags)
        b = dr.Batch()
        b.set_tuning(1 << 22, 1 << 20, refill)
        b.render(jobs)
        out[refill] = [(j["image"].cpu().numpy(), j["grads"].cpu().numpy()) for j in jobs]
    for a, b in zip(out[64], out[0]):
        assert rel_err(a[0], b[0]) < 1e-6
        assert rel_err(a[1], b[1]) < 1e-5
