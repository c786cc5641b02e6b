"""The queue kernels of the wavefront form at small sizes.  A frame that starts with fewer
paths than the finishing threshold, and with no more than two rounds of the chip's lanes
(one where hits are alpha-tested), runs in the finishing launch alone, so each test here
either switches that launch off (RT_OPTION_WAVEFRONT_FINISH 0: every path of every frame
goes through the trace and shade queues) or takes a frame above those rounds, whose paths
change hands in the middle."""
import numpy as np
import pytest
import torch

from rustracer_amd import rt
from rustracer_amd import scenes as S
from tests import gpu_kit as G
from tests import scene_kit as K
from tests import volume_kit as VK

pytestmark = pytest.mark.gpu


def _mask_soup():
    sc = K.triangle_soup(400, seed=31, opaque=False)
    rng = np.random.default_rng(32)
    sc.vertices["color"][:, 3] = rng.random(len(sc.vertices))
    sc.ubo["fully_opaque"] = 0
    sc.ubo["number_of_bounces"] = 5
    sc.ubo["number_of_samples"] = sc.ubo["total_number_of_samples"] = 3
    sc.plights = np.array([S.point_light((0.0, 3.0, 4.0), 30.0)])
    return sc


def _textured(width=100, height=60, spp=2):
    return S.textured_instances(width=width, height=height, spp=spp, bounces=4, num_instances=60, tex_size=64,
                                tri_range=(2000, 20000))


def _cornell(width=256, height=256, spp=4):
    return S.cornell_sphere(width=width, height=height, spp=spp, bounces=4)


SCENES = {"cornell": _cornell, "ragged": lambda: _cornell(37, 21), "mask": _mask_soup, "textured": _textured,
          "blend": lambda: VK.blend_layer(alpha=0.3)}
COUNTS = ("rays", "primary_rays", "extension_rays", "shadow_rays", "shade_events", "light_candidates")


def _scene(ctx, name):
    return G.device_scene(ctx, f"queue_{name}", SCENES[name])


def _trace(ctx, ds, mode, ubo=None, stats=False, accum=None, out=None):
    sc = ds.scene
    acc = rt.new_accumulation(sc.width, sc.height) if accum is None else accum
    st = rt.trace_rays(ctx, ds.tlas, ds.buffers, sc.ubo if ubo is None else ubo, acc, sc.width, sc.height, mode=mode,
                       stats=stats, out=out)
    ctx.sync()
    return acc, st


def _reference(ctx, ds, **more):
    """One lane per pixel, each traversal run to its end."""
    ctx.set_option(rt.OPTION_MEGAKERNEL_PERSISTENT, 0)
    return _trace(ctx, ds, rt.MODE_MEGAKERNEL, **more)


@pytest.mark.parametrize("name", sorted(SCENES))
def test_queues_equal_the_megakernel(gpu_ctx, name):
    ds = _scene(gpu_ctx, name)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 0)
    want, count = _reference(gpu_ctx, ds, stats=True)
    for streams in (1, 2, 4):
        gpu_ctx.set_option(rt.OPTION_WAVEFRONT_STREAMS, streams)
        got, st = _trace(gpu_ctx, ds, rt.MODE_WAVEFRONT, stats=True)
        assert torch.equal(got, want)
        for k in COUNTS:
            assert st[k] == count[k], k
        assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT)[0], want)
    # a second frame on the first one's image
    ubo = ds.scene.ubo.copy()
    ubo["total_number_of_samples"] = 2 * int(ubo["number_of_samples"])
    ubo["frame_count"] = 1
    images = [_trace(gpu_ctx, ds, m, ubo=ubo, accum=want.clone())[0] for m in (rt.MODE_MEGAKERNEL, rt.MODE_WAVEFRONT)]
    assert torch.equal(*images) and not torch.equal(images[0], want)


@pytest.mark.parametrize("name", ["cornell", "mask", "textured"])
def test_variants_and_refills(gpu_ctx, name):
    ds = _scene(gpu_ctx, name)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 0)
    want, _ = _reference(gpu_ctx, ds)
    for v in range(rt.NUM_TRAVERSAL_VARIANTS):
        gpu_ctx.set_option(rt.OPTION_TRAVERSAL_VARIANT, v)
        for extend, shadow in ((16, 1), (1, 1), (64, 64), (17, 33)):
            gpu_ctx.set_option(rt.OPTION_EXTEND_REFILL, extend)
            gpu_ctx.set_option(rt.OPTION_SHADOW_REFILL, shadow)
            assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT)[0], want), (v, extend, shadow)


@pytest.mark.parametrize("name", ["cornell", "textured"])
@pytest.mark.parametrize("streams", [1, 2, 3])
def test_graph_replay(gpu_ctx, name, streams):
    """Captured chunks, replayed over frames of different UBOs (the executable graphs
    are updated), with eager work in between."""
    ds = _scene(gpu_ctx, name)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 0)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_STREAMS, streams)
    ubos, want = [], []
    for k in range(3):
        ubos.append(ds.scene.ubo.copy())
        ubos[k]["frame_count"] = k
        want.append(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT, ubo=ubos[k])[0])
        assert torch.equal(want[k], _trace(gpu_ctx, ds, rt.MODE_MEGAKERNEL, ubo=ubos[k])[0])
    assert not torch.equal(want[0], want[1])
    gpu_ctx.set_option(rt.OPTION_GRAPH, 1)
    for rep in range(2):
        for k in range(3):
            assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT, ubo=ubos[k])[0], want[k]), (rep, k)
            _trace(gpu_ctx, ds, rt.MODE_MEGAKERNEL, ubo=ubos[k])


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("alpha", [False, True])
def test_batch(gpu_ctx, alpha, graph):
    scs = [S.batch_scene(seed, spp=3, bounces=5, tri_range=(500, 40_000), resolutions=(side,))
           for seed, side in zip(range(5), (40, 64, 96, 33, 128))]
    scs += [_cornell(50, 30, 2)] + ([_textured(72, 40)] if alpha else [])
    dss = [G.device_scene(gpu_ctx, f"queue_batch_{k}", lambda s=s: s) for k, s in enumerate(scs)]
    want = [_reference(gpu_ctx, ds)[0] for ds in dss]
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 0)
    gpu_ctx.set_option(rt.OPTION_GRAPH, graph)
    for variant in range(rt.NUM_TRAVERSAL_VARIANTS):
        gpu_ctx.set_option(rt.OPTION_TRAVERSAL_VARIANT, variant)
        got = [torch.full_like(w, 7.0) for w in want]
        rt.trace_rays_batch(gpu_ctx, [(ds.tlas, ds.buffers, ds.scene.ubo, a, ds.scene.width, ds.scene.height)
                                      for ds, a in zip(dss, got)])
        for k, (a, w) in enumerate(zip(got, want)):
            assert torch.equal(a, w), (variant, k)


# above twice the lanes of two waves a SIMD, so above any frame that starts in the finishing launch
BIG = 520


@pytest.mark.parametrize("name", ["opaque", "alpha"])
@pytest.mark.parametrize("streams", [1, 3])
@pytest.mark.parametrize("graph", [0, 1])
def test_paths_change_hands_in_mid_frame(gpu_ctx, name, streams, graph):
    """A threshold above the pixel count on a frame that starts in the queues: after the
    first iterations every set's paths go to the finishing launch, with and without a
    pending shadow ray, and pixels about to retire among them."""
    ds = G.device_scene(gpu_ctx, f"queue_big_{name}", lambda: _cornell(BIG, BIG, 8) if name == "opaque"
                        else _textured(BIG, BIG, 8))
    assert BIG * BIG > 2 * (2 * 4 * 64 * torch.cuda.get_device_properties(0).multi_processor_count)
    sc = ds.scene
    shape = (sc.height, sc.width, 4)
    display = [torch.zeros(shape, dtype=torch.uint8, device="cuda") for _ in range(2)]
    want, count = _reference(gpu_ctx, ds, stats=True, out=display[0])
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_STREAMS, streams)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 1 << 30)
    gpu_ctx.set_option(rt.OPTION_GRAPH, graph)
    got, st = _trace(gpu_ctx, ds, rt.MODE_WAVEFRONT, stats=True, out=display[1])
    assert torch.equal(got, want) and torch.equal(*display)
    for k in COUNTS:
        assert st[k] == count[k], k
    assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT)[0], want)


@pytest.mark.parametrize("alpha", [False, True])
def test_both_sides_of_the_direct_start(gpu_ctx, alpha):
    """Frames around one and around two rounds of the chip's lanes, at a threshold above
    all of them: the ones below start in the finishing launch, the ones above in the
    queues."""
    lanes = 4 * 64 * torch.cuda.get_device_properties(0).multi_processor_count
    tiles = (lanes if alpha else 2 * lanes) // 64
    base = next(k for k in range(int(tiles ** 0.5), 0, -1) if tiles % k == 0)
    gpu_ctx.set_option(rt.OPTION_WAVEFRONT_FINISH, 1 << 30)
    for more in (-1, 0, 1):
        width, height = 8 * (tiles // base + more), 8 * base
        sc = _textured(width, height, 2) if alpha else _cornell(width, height, 2)
        ds = G.DeviceScene(gpu_ctx, sc)
        want = _reference(gpu_ctx, ds)[0]
        for streams in (1, 2):
            gpu_ctx.set_option(rt.OPTION_WAVEFRONT_STREAMS, streams)
            assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT)[0], want), (width, height, streams)


@pytest.mark.parametrize("width,height,inert", [(96, 96, True), (BIG, BIG, False)])
def test_autotune_leaves_settings_without_effect_alone(gpu_ctx, width, height, inert):
    """A frame that runs no queue kernel says nothing about their settings: the tuner
    keeps the ones the context has (graph replay on, a variant and a refill threshold
    other than the defaults), and the image stays the same."""
    ds = G.device_scene(gpu_ctx, f"queue_tune_{width}", lambda: _cornell(width, height, 2))
    want, _ = _trace(gpu_ctx, ds, rt.MODE_MEGAKERNEL)
    gpu_ctx.set_option(rt.OPTION_GRAPH, 1)
    gpu_ctx.set_option(rt.OPTION_TRAVERSAL_VARIANT, 1)
    gpu_ctx.set_option(rt.OPTION_EXTEND_REFILL, 40)
    t = gpu_ctx.autotune(ds.tlas, ds.buffers, ds.scene.ubo, width, height)
    print(t)
    if inert:
        assert t["wavefront_finish"] > 0
        assert (t["graph"], t["traversal_variant"], t["extend_refill"]) == (1, 1, 40)
    assert torch.equal(_trace(gpu_ctx, ds, rt.MODE_WAVEFRONT)[0], want)
