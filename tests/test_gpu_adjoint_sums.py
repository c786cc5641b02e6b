"""The gradient of a light's intensity does not depend on the order in which the frame's
contributions are added: with pixel weights of either sign, whose sum is small against
its terms, repeated calls, the counting form and the frame taken in strips agree.

Bound: the sums are fp64 and rounded to fp32 once per call, so a value v is off by at most
2^-24 |v| (strips: each its own, added here in fp64), and by the fp64 additions of fewer
than 2^23 terms, each of at most 2^-53 of the sum of the terms' magnitudes: 2^-30 of it.
That sum is the gradient for the weights' magnitudes, as a light's terms carry the sign of
their pixel's weight."""
import numpy as np
import pytest
import torch

from rustracer_amd import scenes as S
from tests import gpu_kit as G
from tests.test_gpu_adjoint import _adjoint

pytestmark = pytest.mark.gpu
BOUNCES = 4


@pytest.mark.parametrize("lights,width,height,spp", [(1, 512, 512, 4), (300, 160, 128, 8)])
def test_intensity_gradient_does_not_depend_on_the_order(gpu_ctx, lights, width, height, spp):
    sc = S.cornell_params(width=width, height=height, spp=spp, bounces=BOUNCES, tex_size=8)
    if lights > 1:  # more than the 256 whose sums are held in LDS
        sc.plights = np.stack([S.point_light((-0.4 + 0.8 * k / lights, 1.9, 0.0), 50.0 / lights) for k in range(lights)])
    assert spp * width * height * BOUNCES < 2 ** 23
    ds = G.DeviceScene(gpu_ctx, sc)
    rng = np.random.default_rng(17)
    w = rng.normal(size=(height, width, 4)).astype(np.float32)
    w[..., 3] = 0
    # the same weight in every channel: a light's terms have its sign
    w[..., :3] = w[..., :1]
    g = torch.from_numpy(w).cuda()
    runs = [_adjoint(gpu_ctx, ds, g, stats=k == 2)[1:3] for k in range(4)]
    mags = _adjoint(gpu_ctx, ds, g.abs())[1:3]
    strips = [np.zeros_like(m) for m in mags]
    size = [np.zeros_like(m) for m in mags]
    for y in range(0, height, 8):
        one = torch.zeros_like(g)
        one[y:y + 8] = g[y:y + 8]
        for k, v in enumerate(_adjoint(gpu_ctx, ds, one)[1:3]):
            strips[k] += v
            size[k] += np.abs(v)
    for k, what in enumerate(("point", "directional")):
        assert mags[k].max() > 0
        for r in runs:
            v = r[k]
            off = np.abs(v - strips[k])
            tol = 2.0 ** -24 * (np.abs(v) + size[k]) + 2.0 ** -29 * mags[k]
            print(what, "largest difference from the strips", off.max(), "of", np.abs(v).max(), "allowed", tol.max())
            assert np.all(off <= tol)
            assert np.all(np.abs(v - runs[0][k]) <= 2.0 ** -23 * np.abs(v) + 2.0 ** -29 * mags[k])
