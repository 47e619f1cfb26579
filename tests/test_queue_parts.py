"""Passes that select more edges than the queue may hold are sampled in parts (the
line lies at 2^27 entries; the tests lower it).  A render must not notice: the same
rays are traced (their number is compared exactly, so no sample is lost or walked
twice at the ends of the lists, however ragged), and images and gradients agree up
to the order of float sums (up to 2e-6 of the gradient's norm between runs of one
kind, 1e-5 asked)."""
import ctypes

import numpy as np
import pytest

from delta_ray_amd import _abi, workloads
from delta_ray_amd import delta_ray as dr
from tests.helpers import rel_err


def _limit(batch, entries):
    before = ctypes.c_int64()
    st = batch.lib.dr_test_batch_queue_limit(batch.handle, entries, ctypes.byref(before))
    return st, before.value


def test_queue_stays_below_32_bit_positions():
    """no queue may be allowed that 32-bit positions do not reach"""
    b = dr.Batch()
    for n in (0, -1, (1 << 27) + 1, 1 << 31, 1 << 40):
        assert _limit(b, n)[0] != _abi.DR_OK
    assert _limit(b, 1000) == (_abi.DR_OK, 1 << 27)
    assert _limit(b, 1 << 27) == (_abi.DR_OK, 1000)


SIZES = [(1, 1, 1), (5, 3, 1), (40, 33, 3)]


def _render(sc, size, limit, refill=64, graph=False, times=1):
    import torch
    W, H, spp = size
    b = dr.Batch()
    b.set_tuning(1 << 22, 1 << 20, refill)
    if limit:
        assert _limit(b, limit)[0] == _abi.DR_OK
    g = torch.Generator(device="cuda").manual_seed(3)
    job = dict(scene=sc, options=dr.DeviceScene.options(W, H, spp, 2, 11, _abi.DR_FLAGS_PARITY),
               image=torch.empty((H, W, 3), device="cuda"), grads=torch.empty(sc.grad_size, device="cuda"),
               d_image=torch.randn((H, W, 3), generator=g, device="cuda"))
    out = []
    for _ in range(times):
        sc.stats(True)
        b.render([job], graph=graph)
        torch.cuda.synchronize()
        st = sc.stats(False)
        out.append((job["image"].cpu().numpy().copy(), job["grads"].cpu().numpy().copy(), st["rays"]))
    return out


def _same(a, b, rays=True):
    assert rel_err(a[0], b[0]) < 1e-6
    assert rel_err(a[1], b[1]) < 1e-5
    assert not rays or a[2] == b[2], (a[2], b[2])


def _scene(size):
    w = workloads.heightfield(grid=24, resolution=size[:2])
    return dr.DeviceScene(w["camera"], w["shapes"], w["materials"], w["lights"])


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("limit", [700, 1021, 4097])
def test_parts_match_one_pass(gpu, size, limit):
    sc = _scene(size)
    whole = _render(sc, size, None)[0]
    _same(_render(sc, size, limit)[0], whole)


@pytest.mark.gpu
def test_parts_of_the_breadth_first_selection_and_of_graphs(gpu):
    size = SIZES[-1]
    sc = _scene(size)
    whole = _render(sc, size, None)[0]
    _same(_render(sc, size, 1021, refill=0)[0], whole)
    # the first replay finds the queue too long and runs again (its rays are counted twice)
    for k, r in enumerate(_render(sc, size, 1021, graph=True, times=3)):
        _same(r, whole, rays=k > 0)


@pytest.mark.gpu
def test_queue_shorter_than_a_point_is_refused(gpu):
    size = SIZES[-1]
    with pytest.raises(Exception, match="edge queue"):
        _render(_scene(size), size, 1)
