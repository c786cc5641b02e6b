"""The host BVH walk checks what the traversal reads of a quantised node: its planes
unrounded (rounded to fp32 they can lie half an ulp further out) and the stack entries of
its children."""
import numpy as np

from rustracer_amd import bvhcheck as V
from rustracer_amd import rt

BASE = 2.0 ** 24  # fp32 numbers are 2 apart from here on


def _leaf(lo_q, hi_q, origin=BASE, exp=0, count=1):
    n = np.zeros(1, rt.QNODE)
    n["origin"], n["exp"], n["child"] = origin, exp, V.EMPTY
    q = n["q"].reshape(1, 3, 2, 4)
    q[0, :, 0, 0], q[0, :, 1, 0] = lo_q, hi_q
    n["child"][0, 0], n["count"][0, 0], n["tag"][0, 0] = 0, count, 0x80 | (count - 1) << 3
    return n


def _tri(lo, hi):
    t = np.zeros(1, V.TRI)
    t["v0"], t["v1"][:, :3], t["v2"][:, :3] = lo, hi, lo
    return t


def _errors(node, tri):
    return V._check(V._Pool(node), 0, 0, 1, tri, "triangle")


def test_planes_are_taken_unrounded():
    inside = _tri(BASE + 2, BASE + 6)
    assert _errors(_leaf(2, 6), inside) == []
    # as fp32 numbers BASE + 3 and BASE + 5 are BASE + 4 (ties to even): no nearer than
    # the triangle below; unrounded, the second lies inside it
    tri = _tri(BASE + 4, BASE + 6)
    assert rt.decode_nodes(_leaf(5, 6))["lo_x"][0, 0] == BASE + 4
    assert _errors(_leaf(3, 6), tri) == []
    assert any("not inside every box" in e for e in _errors(_leaf(5, 6), tri))


def test_a_wrong_stack_entry_is_reported():
    tri = _tri(BASE + 2, BASE + 6)
    for tag in (0, 0x80 | 1 << 3, 0x08):
        node = _leaf(2, 6)
        node["tag"][0, 0] = tag
        assert any("stack entry" in e for e in _errors(node, tri))
    # the entries of children that are not there are not read
    node = _leaf(2, 6)
    node["tag"][0, 1:] = 7
    assert _errors(node, tri) == []
