"""The lifters' turn beside the re-sort for lifters of fewer than eight
vertices and faces of fewer than four: the area of a face reads its four
orders whatever its vertex count, also those that name a vertex the lifter
does not turn.  Vertices, normals, centroids and areas equal the host's turn."""
import pytest

from bdem import scenarios as S
from helpers import make_pair

pytestmark = pytest.mark.gpu


def _v(f):
    return (f.x, f.y, f.z)


def test_faces_that_name_unturned_vertices():
    deck = S.mill_deck(300)
    for k, d in enumerate(deck["dobj"]):
        if k % 2:
            d.num_vertex = 6          # vertices 6 and 7 stay where they are
            d.num_edges = 0
            for j, order in enumerate(((0, 4, 5, 7), (2, 3, 1, 6), (5, 4, 1, 7))):
                d.faces[j].num_vertex = 3
                for q in range(4):
                    d.faces[j].vertex_Order[q] = order[q]
    dev, ora = make_pair(deck)
    try:
        dev.set_lifter_rotation(deck["rad_per_step"], deck["lifter_about"])
        dev.step(40)   # the first step sorts in full and turns in a launch of its own
        for _ in range(40):
            ora.turn_lifters(deck["rad_per_step"], deck["lifter_about"])
        for g, w in zip(dev.get_dobj(), ora.get_dobj()):
            assert _v(g.COM) == _v(w.COM)
            assert [_v(g.vertex[k]) for k in range(8)] == [_v(w.vertex[k]) for k in range(8)]
            for j in range(3):
                assert _v(g.faces[j].normal) == _v(w.faces[j].normal)
                assert _v(g.faces[j].centroid) == _v(w.faces[j].centroid)
                assert g.faces[j].area == w.faces[j].area
    finally:
        dev.close()
        ora.close()
