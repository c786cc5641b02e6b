"""BVH builds at the sizes where their kernels change: tiles of 512 leaves and their
multiples by 16 (by 4 where a tree is too deep for that), the one-launch sort's limit of 16,384 keys, and batches of many small
segments that share tiles.  Every tree passes the validity walk (bit-exact: every triangle
in exactly one leaf, inside every box on its path)."""
import numpy as np
import pytest
import torch

from rustracer_amd import bvhcheck, rt
from rustracer_amd import layouts as L
from rustracer_amd import scenes as S
from tests import gpu_kit as G

pytestmark = pytest.mark.gpu


def _scene(counts, seed, kind):
    """One geometry of counts[i] triangles per segment i."""
    rng = np.random.default_rng(seed)
    b = S.Builder()
    mat = b.add_material(L.default_material())
    entries = []
    for k, n in enumerate(counts):
        c = rng.uniform(-1, 1, (n, 1, 3))
        if kind == "line":      # the codes differ in one axis: a deep tree
            c = np.concatenate([np.geomspace(1e-6, 1.0, n).reshape(n, 1, 1), np.zeros((n, 1, 2))], 2)
        elif kind == "same":    # equal codes: ties by index
            c = np.zeros((n, 1, 3))
        p = (c + rng.normal(scale=0.02, size=(n, 3, 3))).reshape(-1, 3)
        if kind == "same":
            p = np.tile(p[:3], (n, 1))
        g = b.add_primitive(S.make_vertices(p, np.tile([0.0, 1.0, 0.0], (3 * n, 1))), np.arange(3 * n), mat)
        entries.append((None if k % 2 else np.diag([1.0, 1.0, 1.5, 1.0]), g))
    cam = S.cornell_sphere().ubo
    return b.finish("sizes", S.make_instances(entries), [S.point_light((0, 3, 0), 1.0)], [L.default_dlight()], cam, 8, 8)


def _check(ctx, sc):
    ds = G.DeviceScene(ctx, sc)
    want = [int(g["prim_count"]) for g in sc.geometries]
    assert all(e == [] for e in bvhcheck.check_blases(ctx, ds.blases, want))
    return ds


@pytest.mark.parametrize("kind", ["cloud", "line", "same"])
@pytest.mark.parametrize("n", [1, 2, 3, 255, 511, 512, 513, 1025, 4099, 8193, 16383, 16384, 16385, 70001])
def test_one_segment(gpu_ctx, n, kind):
    _check(gpu_ctx, _scene([n], n, kind))


@pytest.mark.parametrize("passes", [0, 2])
@pytest.mark.parametrize("counts", [[1] * 700, [2, 1, 300, 1, 1, 255, 513, 1] * 3, [7] * 400 + [3000] + [1] * 50])
def test_many_segments(gpu_ctx, counts, passes):
    gpu_ctx.set_option(rt.OPTION_BVH_TREELET_PASSES, passes)
    try:
        _check(gpu_ctx, _scene(counts, 5, "cloud"))
    finally:
        gpu_ctx.reset_options()


@pytest.mark.parametrize("tiles", [16, 40])
def test_deep_paths_between_tiles(gpu_ctx, tiles):
    """Every tile of 512 leaves starts with 56 codes whose distances double, so it leaves
    57 subtrees and sixteen tiles do not fit a larger one: the build starts over."""
    rng = np.random.default_rng(tiles)
    keys = []
    for i in range(tiles):
        p = i << 57
        keys += [p] + [p + (1 << j) for j in range(55)]
        keys += [p + (1 << 54) + int(x) for x in rng.integers(1, 1 << 55, 456 - (i == 0))]
    k = np.array(keys + [(1 << 63) - 1], np.uint64)
    c = np.zeros((len(k), 3))
    for b in range(63):
        c[:, 2 - b % 3] += ((k >> np.uint64(b)) & np.uint64(1)).astype(np.float64) * 2.0 ** (b // 3)
    c += 0.5
    c[0], c[-1] = 0.0, 2.0**21 - 1.0     # box centres: cells of unit size
    p = (c[:, None, :] + np.array([[-0.25] * 3, [0.25] * 3, [0.25, -0.25, 0.25]])).reshape(-1, 3)
    b = S.Builder()
    mat = b.add_material(L.default_material())
    n = len(k)
    g = b.add_primitive(S.make_vertices(p, np.tile([0.0, 1.0, 0.0], (3 * n, 1))), np.arange(3 * n), mat)
    cam = S.cornell_sphere().ubo
    sc = b.finish("deep", S.make_instances([(None, g)]), [S.point_light((0, 3, 0), 1.0)], [L.default_dlight()], cam, 8, 8)
    _check(gpu_ctx, sc)


@pytest.mark.parametrize("counts", [[3], [0, 5, 0], [1] * 700, [2, 1, 300, 1, 1, 255, 513, 1] * 3, [4096] * 5, [70001]])
def test_refit_there_and_back(gpu_ctx, counts):
    """Refit to other vertices and back gives the built nodes bit for bit: boxes, padding
    by the segment's largest coordinate, quantising."""
    sc = _scene(counts, 9, "cloud")
    ds = G.DeviceScene(gpu_ctx, sc)

    def nodes():
        return [rt.read_nodes(gpu_ctx, i).tobytes() for i in (ds.blases[0].info(), ds.tlas.flat_info(), ds.tlas.info())
                if i.num_nodes]

    built = nodes()
    moved = ds.buffers.vertices.clone()
    v = moved.view(torch.float32).reshape(-1, L.VERTEX.itemsize // 4)
    k = L.VERTEX.fields["pos"][1] // 4
    v[:, k:k + 3] *= -3.0
    rt.refit_as(gpu_ctx, sc, ds.buffers, ds.blases, vertices=moved, tlas=ds.tlas)
    assert all(e == [] for e in bvhcheck.check_blases(gpu_ctx, ds.blases, counts))
    assert not bvhcheck.check_tlas(gpu_ctx, ds.tlas, len(counts))
    assert nodes()[0] != built[0]
    rt.refit_as(gpu_ctx, sc, ds.buffers, ds.blases, tlas=ds.tlas)
    assert nodes() == built
