"""blas_inputs fills its records as arrays; each equals the record written out for its
geometry alone, for index runs that follow one another, in any other order, and empty."""
import numpy as np
import pytest

from rustracer_amd import layouts as L
from rustracer_amd import rt
from rustracer_amd import scenes as S


class _Buffer:
    def __init__(self, address):
        self.address = address

    def data_ptr(self):
        return self.address


class _Buffers:
    vertices, indices = _Buffer(1 << 40), _Buffer((1 << 41) + 16)


@pytest.mark.parametrize("change", ["none", "reversed", "empty runs", "overlap", "no geometry"])
def test_records(change):
    sc = S.displaced_sphere(seed=1, freq=24)
    geo = sc.geometries.copy()
    assert len(geo) > 3
    geo["opaque"][1] = 0
    if change == "reversed":
        geo = geo[::-1].copy()
    elif change == "empty runs":
        geo["prim_count"][[0, len(geo) - 1]] = 0
    elif change == "overlap":
        geo["index_offset"][2] = geo["index_offset"][1] + 3
    elif change == "no geometry":
        geo = geo[:0]
    sc.geometries = geo
    ins = rt.blas_inputs(sc, _Buffers)
    assert len(ins) == len(geo)
    for got, g in zip(ins, geo):
        first, offset, count, opaque = (int(x) for x in g)
        run = sc.indices[offset:offset + 3 * count]
        want = rt.BlasInput(1 << 40, L.VERTEX.itemsize, int(np.max(run, initial=0)), (1 << 41) + 16, first, 4 * offset,
                            count, rt.GEOMETRY_OPAQUE if opaque else 0)
        assert bytes(got) == bytes(want)
