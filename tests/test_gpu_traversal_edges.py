"""The box test of the traversal at its edges: rays parallel to the axes (components
0, -0 and denormal), origins far outside the scene, open t ranges, and leaves of 1 to
16 triangles.  A box wrongly culled would make a hit depend on the tree's shape, so
trees of other leaf sizes and collapses must give the same hit records bit for bit;
near the scene the hits are also the brute-force oracle's."""
import numpy as np
import pytest

from oracle import binding as B
from rustracer_amd import layouts as L, rt
from rustracer_amd import scenes as S
from tests import gpu_kit as G

pytestmark = pytest.mark.gpu


def _rays(kind, n=6000):
    rng = np.random.default_rng(31)
    r = np.zeros(n, L.RAY)
    r["tmin"], r["tmax"] = 0.0, np.inf
    target = rng.uniform((-1.0, 0.0, -1.0), (1.0, 2.0, 1.0), (n, 3))
    if kind == "axis":
        axis, sign = rng.integers(0, 3, n), rng.choice([-1.0, 1.0], n)
        d = np.zeros((n, 3), np.float32)
        d[np.arange(n), axis] = sign
        other = np.array([0.0, -0.0, 1e-42, -1e-42, 1e-36], np.float32)
        for k in range(3):
            fill = axis != k
            d[fill, k] = other[rng.integers(0, len(other), int(fill.sum()))]
        r["direction"] = d
        r["origin"] = target - 4.0 * sign[:, None] * np.eye(3)[axis]
    else:
        far = {"near": 5.0, "far": 3000.0}[kind]
        d = rng.normal(size=(n, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        r["direction"] = d
        r["origin"] = target - far * d
    return r


@pytest.mark.parametrize("kind", ["axis", "near", "far"])
def test_hits_do_not_depend_on_the_tree(gpu_ctx, kind):
    rays = _rays(kind)
    sc = S.cornell_sphere()
    got = []
    try:
        for leaf, collapse, treelets, flat in ((1, 1, 2, True), (2, 1, 2, False), (16, 1, 0, True), (5, 0, 0, False)):
            gpu_ctx.set_option(rt.OPTION_BLAS_LEAF_SIZE, leaf)
            gpu_ctx.set_option(rt.OPTION_BVH_COLLAPSE, collapse)
            gpu_ctx.set_option(rt.OPTION_BVH_TREELET_PASSES, treelets)
            ds = G.DeviceScene(gpu_ctx, sc, flatten=flat)
            got.append(rt.trace_ray_queries(gpu_ctx, ds.tlas, rays, rt.RAY_FLAG_OPAQUE))
    finally:
        gpu_ctx.reset_options()
    assert (got[0]["primitive_id"] != G.MISS).mean() > 0.2
    for other in got[1:]:
        assert got[0].tobytes() == other.tobytes()
    if kind != "far":
        oh, otuv = B.OracleScene(sc).trace_rays(rays, brute=True)
        assert len(G.explain_mismatches(sc, rays["origin"], rays["direction"], got[0], oh, otuv[:, 0])) == 0
