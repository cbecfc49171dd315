"""The LDS layout of the step on quads of lanes over the capacity sets that it
takes, on the CPU: regions alive at the same time do not overlap, the
workgroup's rows fit its LDS, and the packed words hold every index."""
import ctypes as C
import os

import numpy as np
import pytest

from puffysics_amd.b3types import signature

FIELDS = ("hits jkeys last pos level order jlast jlev jgeo jconst heads y bounds masks keys clip cw law words hw "
          "shape_words jgeo_words jconst_words body_rows clip_words wg_words cols").split()
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu", "libquadlayout.so")


def layout(caps, waves, law):
    lib = C.CDLL(LIB)
    lib.quadlayout.argtypes = [C.c_ulonglong, C.c_int, C.c_int, C.c_void_p]
    out = np.zeros(len(FIELDS), np.int32)
    if not lib.quadlayout(signature(*caps), waves, law, out.ctypes.data):
        return None
    return dict(zip(FIELDS, out.tolist()))


def disjoint(spans, end):
    """[(start, words)] lie within `end` words and do not overlap."""
    spans = sorted((a, a + n) for a, n in spans if n > 0)
    assert spans[0][0] >= 0 and spans[-1][1] <= end, (spans, end)
    for (_, b), (c, _) in zip(spans, spans[1:]):
        assert b <= c, spans


def check(caps, waves, law):
    q = layout(caps, waves, law)
    if q is None:
        return False
    b, s, c, j = caps
    # a body, a contact and its level, a joint's level in both iterations
    assert b <= 255 and c <= 1023 and (c | (c << 10)) < 1 << 31 and 2 * j <= 255 and s <= 64
    cand = s * (s - 1) // 2
    assert q["hw"] * 32 >= cand and min(4, cand) <= q["cw"] <= 4 * waves
    assert 4 * (q["wg_words"] + q["words"] * q["cols"]) <= 163840 * waves // 8
    end = q["words"]
    shapes = (0, q["shape_words"] * s)
    hits, jkeys, heads = (q["hits"], q["hw"] + 1), (q["jkeys"], j), (q["heads"], c)
    rows, law_rows = (q["y"], q["body_rows"]), (q["law"], law * b)
    # candidates and manifolds; the contacts written while the bodies' rows are staged; the solve
    disjoint([shapes, hits, jkeys, (q["bounds"], 6 * s), (q["masks"], 2 * s), (q["keys"], c),
              (q["clip"], q["cw"] * q["clip_words"])], end)
    disjoint([shapes, hits, heads, rows, law_rows], end)
    disjoint([(q["last"], b), (q["pos"], c + 2), (q["level"], c), (q["order"], c), (q["jlast"], b), (q["jlev"], j),
              (q["jgeo"], q["jgeo_words"] * j), (q["jconst"], q["jconst_words"] * j), heads, rows, law_rows], end)
    return True


@pytest.mark.parametrize("waves,law", [(8, 0), (8, 9), (4, 0), (4, 9)])
def test_regions(waves, law):
    rng = np.random.default_rng(waves + law)
    taken = 0
    for _ in range(4000):
        caps = tuple(int(round(np.exp(rng.uniform(0.0, np.log(m))))) for m in (80, 80, 600, 20))
        taken += check(caps, waves, law)
    assert taken > 400


@pytest.mark.parametrize("axis", range(4))
def test_limits(axis):
    """The largest capacity of each kind that is taken, the others small."""
    caps, last = [2, 2, 2, 1], 0
    for n in range(1, 1100):
        caps[axis] = n
        if check(tuple(caps), 8, 0):
            last = n
    assert last == (91, 64, 483, 16)[axis]
    for over in ((256, 3, 4, 1), (4, 65, 4, 1), (4, 3, 1024, 1), (4, 3, 4, 17)):
        assert layout(over, 8, 0) is None
