"""The step with articulated contacts one world to a wave (b3k_step_art_world)
and the batch size at which 64 worlds to a wave take over, against the oracle
word for word (the contract is the reference's fp32 bits, so the tolerance is
zero); and that worlds which go through no joint tree take no wave each.
"""
import numpy as np
import pytest

import b3test as T
from b3test import clone, diff_words
from puffysics_amd import scenes

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# One world; the edges of the sixteen worlds that share an XCD, of eight such
# groups and of a tile; the largest batch of the kernel and the first of the
# other.  Families with trees and contacts (arm), trees that touch nothing
# (chains) and contacts without trees (stacks, bin).
@pytest.mark.parametrize("scene,count,steps", [(5, 1, 6), (5, 17, 6), (5, 129, 4), (3, 65, 3), (2, 127, 6), (4, 20, 8),
                                               (5, 16384, 1), (5, 16385, 1)])
def test_batch_edges(scene, count, steps):
    from puffysics_amd.engine import B3_ENGINE_ART_CONTACTS, B3Engine
    sc = scenes.SCENES[scene]
    some = min(count, 192)                     # the oracle steps these and the batch repeats them
    start = scenes.build(scene, some)
    T.oracle_run(scene, start, clone(start), 0, 12, threads=8)
    ref, first = clone(start), clone(start)
    pick = np.arange(count) % some
    eng = B3Engine(start[pick], sc.sig)
    eng.set_options(B3_ENGINE_ART_CONTACTS)
    rng = np.random.default_rng(count)
    for _ in range(steps):
        reset = (rng.random(some) < 0.1).astype(np.uint8)
        active = (rng.random(some) < 0.8).astype(np.uint8)
        ref[reset != 0] = first[reset != 0]
        T.oracle_step_art(ref, sc.sig, sc.dt, sc.substeps, active)
        eng.step(sc.dt, sc.substeps, torch.from_numpy(active[pick]).cuda(), torch.from_numpy(reset[pick]).cuda())
        torch.cuda.synchronize()
    got = eng.download()
    eng.close()
    for k in range(0, count, some):
        part = got[k:k + some]
        bad = diff_words(part, ref[:len(part)], sc.sig)
        assert len(bad) == 0, "worlds from %d: %d differing words, first %s" % (k, len(bad), bad[:4].tolist())
    assert scene != 5 or count < 17 or (ref["contact_count"] > 0).any()


# Chains touch nothing, stacks have no joints.
@pytest.mark.parametrize("scene", [2, 3])
def test_worlds_without_trees_and_contacts(scene):
    """With the option on, worlds without articulated contacts step 64 to a
    wave as the ordinary one-wave step does.  Measured at 8,192 worlds the
    two take about the same time; a wave to each world took five times it."""
    from puffysics_amd.engine import B3_ENGINE_ART_CONTACTS, B3_ENGINE_ONE_WAVE_PER_TILE, B3Engine
    sc = scenes.SCENES[scene]
    eng = B3Engine(scenes.build(scene, 512)[np.arange(8192) % 512], sc.sig)
    took = {}
    for options in (B3_ENGINE_ONE_WAVE_PER_TILE, B3_ENGINE_ART_CONTACTS):
        eng.set_options(options)
        ends = [torch.cuda.Event(enable_timing=True) for _ in range(11)]
        for _ in range(40):
            eng.step(sc.dt, sc.substeps)
        for end in ends:
            end.record()
            eng.step(sc.dt, sc.substeps)
        torch.cuda.synchronize()
        took[options] = sorted(a.elapsed_time(b) for a, b in zip(ends, ends[1:]))[5]
    eng.close()
    assert took[B3_ENGINE_ART_CONTACTS] < 2.5 * took[B3_ENGINE_ONE_WAVE_PER_TILE], took
