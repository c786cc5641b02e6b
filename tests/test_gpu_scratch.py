"""What a context keeps of a build's device scratch: at most 64 MiB, whatever it built."""
import gc

import pytest
import torch

from rustracer_amd import rt
from rustracer_amd import scenes as S

pytestmark = pytest.mark.gpu
KEEP = 64 << 20
# the allocator's granularity on the few blocks alive
SLACK = 8 << 20


def test_a_large_build_gives_its_scratch_back():
    sc = S.displaced_sphere(width=64, height=64, spp=1, bounces=1, freq=150)
    assert sc.geometries["prim_count"].sum() * 300 > 2 * KEEP  # what it builds with
    buf = rt.Buffers(sc)
    # what the runtime itself allocates at a kernel's first launch comes before the count
    small = S.displaced_sphere(width=64, height=64, spp=1, bounces=1, freq=32)
    first = rt.Context(0)
    held = rt.create_as(first, small, rt.Buffers(small))
    first.sync()
    del held
    first.close()
    ctx = rt.Context(0)
    try:
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        held = rt.create_as(ctx, sc, buf)
        ctx.sync()
        del held
        gc.collect()
        torch.cuda.empty_cache()
        torch.cuda.synchronize()
        kept = before - torch.cuda.mem_get_info()[0]
        print("kept", kept)
        assert kept <= KEEP + SLACK
    finally:
        ctx.close()
