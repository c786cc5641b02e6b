"""Frames and query sets around the sizes where fewer lanes of a wave take work (8 lanes a
wave at the least, 64 from one full wave per SIMD on): the megakernel forms and the queue
kernels give the same image bit for bit, and a query set the same hits as its parts."""
import numpy as np
import pytest

from rustracer_amd import layouts as L
from rustracer_amd import rt
from rustracer_amd import scenes as S
from tests import gpu_kit as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (9, 7), (64, 64), (97, 90), (256, 255), (257, 260)])
def test_modes_agree(gpu_ctx, size):
    sc = S.cornell_sphere(width=size[0], height=size[1], spp=2, bounces=4, seed=3)
    ds = G.DeviceScene(gpu_ctx, sc)
    images = []
    for mode in (rt.MODE_MEGAKERNEL, rt.MODE_WAVEFRONT):
        for finish in (0, 1 << 20):
            gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, finish)
            acc = rt.new_accumulation(sc.width, sc.height)
            rt.trace_rays(gpu_ctx, ds.tlas, ds.buffers, sc.ubo, acc, sc.width, sc.height, mode=mode)
            gpu_ctx.sync()
            images.append(acc.cpu().numpy())
    gpu_ctx.reset_options()
    assert all(np.array_equal(images[0], i) for i in images[1:])


@pytest.mark.parametrize("n", [1, 8191, 8193, 65535, 65537])
def test_query_sets_equal_their_parts(gpu_ctx, n):
    sc = S.cornell_sphere(width=8, height=8, spp=1, bounces=1, seed=3)
    ds = G.DeviceScene(gpu_ctx, sc)
    rng = np.random.default_rng(n)
    rays = np.zeros(n, L.RAY)
    rays["origin"] = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32)
    rays["direction"] = rng.normal(size=(n, 3)).astype(np.float32)
    rays["tmax"] = 100.0

    def hits(r):
        h = rt.trace_ray_queries(gpu_ctx, ds.tlas, r)
        return h.tobytes()

    step = 1 + n // 3
    assert hits(rays) == b"".join(hits(rays[i:i + step]) for i in range(0, n, step))
