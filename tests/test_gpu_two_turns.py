"""Shared tiles in two turns (between one and two tiles per CU, worlds of many
shapes) against one wave per tile, word for word: the same operations in the
same order, so the tolerance is zero.
"""
import numpy as np
import pytest

from b3test import diff_words
from puffysics_amd import scenes

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# The first batch past one tile per CU (256 CUs), a ragged one, the last of
# the rule and the first past it.
@pytest.mark.parametrize("scene,count", [(5, 16385), (5, 20001), (5, 32768), (5, 32769), (4, 16385)])
def test_two_turns(scene, count):
    from puffysics_amd.engine import B3_ENGINE_ONE_WAVE_PER_TILE, B3Engine
    sc = scenes.SCENES[scene]
    some = 509                                 # the batch repeats these
    start = scenes.build(scene, some)[np.arange(count) % some]
    got = []
    for options in (0, B3_ENGINE_ONE_WAVE_PER_TILE):
        eng = B3Engine(start, sc.sig)
        eng.set_options(options)
        rng = np.random.default_rng(count)
        for _ in range(40):
            reset = torch.from_numpy((rng.random(count) < 0.02).astype(np.uint8)).cuda()
            active = torch.from_numpy((rng.random(count) < 0.9).astype(np.uint8)).cuda()
            eng.step(sc.dt, sc.substeps, active, reset)
        torch.cuda.synchronize()
        got.append(eng.download()[-1024:])     # the last tiles are the second turn's
        eng.close()
    assert (got[0]["contact_count"] > 0).any()
    bad = diff_words(got[0], got[1], sc.sig)
    assert len(bad) == 0, "%d differing words, first %s" % (len(bad), bad[:4].tolist())
