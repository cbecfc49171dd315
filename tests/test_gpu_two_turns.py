"""Shared tiles in two turns (between one and two tiles per CU, worlds of many
shapes) and the one-wave step past them against the oracle, word for word (the
contract is the reference's fp32 bits, so the tolerance is zero).
"""
import numpy as np
import pytest

from b3test import clone, diff_words, oracle_step_batch
from puffysics_amd import scenes

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# The first batch past one tile per CU (256 CUs), a ragged one, the last of
# the rule and the first past it.
@pytest.mark.parametrize("scene,count", [(5, 16385), (5, 20001), (5, 32768), (5, 32769), (4, 16385)])
def test_two_turns(scene, count):
    """The batch repeats 509 worlds, which the oracle steps; every world of
    every tile is compared, the first 509 with the oracle's and the others
    with them (their bits, whatever the tile and lane)."""
    from puffysics_amd.engine import B3_ENGINE_KEEP_SOLVER_FIELDS, B3Engine
    sc = scenes.SCENES[scene]
    some = 509
    start = scenes.build(scene, some)
    ref, pick = clone(start), np.arange(count) % some
    eng = B3Engine(start[pick], sc.sig)
    eng.set_options(B3_ENGINE_KEEP_SOLVER_FIELDS)
    rng = np.random.default_rng(count)
    for _ in range(30):
        reset = (rng.random(some) < 0.02).astype(np.uint8)
        active = (rng.random(some) < 0.9).astype(np.uint8)
        ref[reset != 0] = start[reset != 0]
        oracle_step_batch(ref, sc.sig, sc.dt, sc.substeps, active)
        eng.step(sc.dt, sc.substeps, torch.from_numpy(active[pick]).cuda(), torch.from_numpy(reset[pick]).cuda())
    torch.cuda.synchronize()
    got = eng.download()
    eng.close()
    assert (ref["contact_count"] > 0).any()
    bad = diff_words(got[:some], ref, sc.sig)
    assert len(bad) == 0, "%d differing words, first %s" % (len(bad), bad[:4].tolist())
    first = got[:some].view(np.uint32).reshape(some, -1)
    for k in range(some, count, some):
        part = got[k:k + some].view(np.uint32).reshape(-1, first.shape[1])
        assert np.array_equal(part, first[:len(part)]), "worlds from %d" % k
