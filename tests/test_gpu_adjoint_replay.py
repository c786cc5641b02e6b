"""The adjoint's second pass takes the hits of a path's first eight bounces from the first
pass and traces beyond them; the counting form traces them all.  Both give the same
gradients up to the order of their float sums, with
paths shorter and longer than that, on opaque geometry and on blended geometry, whose
any-hit tests draw random numbers along the ray."""
import numpy as np
import pytest
import torch

from rustracer_amd import layouts as L
from rustracer_amd import scenes as S
from tests import gpu_kit as G
from tests.test_gpu_adjoint import _adjoint

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blend", [False, True])
@pytest.mark.parametrize("bounces", [1, 8, 9, 24])
def test_kept_hits_give_the_retraced_gradient(gpu_ctx, bounces, blend):
    sc = S.cornell_params(width=56, height=40, spp=3, bounces=bounces, tex_size=9)
    if blend:
        sc.geometries["opaque"] = 0
        sc.materials["alpha_mode"] = L.ALPHA_BLEND
        sc.ubo["fully_opaque"] = 0
        sc.materials["base_color"][:, 3] = 0.6
    ds = G.DeviceScene(gpu_ctx, sc)
    g = torch.ones((sc.height, sc.width, 4), dtype=torch.float32, device="cuda")
    a0, p0, d0, _ = _adjoint(gpu_ctx, ds, g)
    a1, p1, d1, st = _adjoint(gpu_ctx, ds, g, stats=True)
    assert st["rays"] > 0 and np.abs(a0[1]).max() > 0
    for k in a0:
        assert np.allclose(a0[k], a1[k], rtol=1e-5, atol=1e-6 * np.abs(a0[k]).max())
    assert np.allclose(p0, p1, rtol=1e-5) and np.allclose(d0, d1, rtol=1e-5, atol=1e-9)
