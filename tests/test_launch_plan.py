"""Which kernel a batch steps on, and what happens where its memory is not to
be had, on a machine without a GPU (tests/hipstand.py)."""
import pytest

from hipstand import plan
from puffysics_amd import scenes
from puffysics_amd.b3types import signature

OUT_OF_MEMORY = 2


def sig(scene):
    return scenes.SCENES[scene].sig


# On 8 CUs: a quarter tile per CU is 2 tiles (128 worlds), half a tile 4, one
# tile 8, two 16.  Scene capacities as in puffysics_amd.scenes; 17 joints are
# more than the quad step takes, 11 shapes fewer than share the candidate
# search.
@pytest.mark.parametrize("caps,count,kernel,groups", [
    (1, 64, "b3k_step<1,1>", 1), (1, 1025, "b3k_step<1,1>", 17),
    (5, 128, "b3k_step_quad<8,2,1>", 8), (5, 129, "b3k_step_quad<4,3,1>", 12), (5, 256, "b3k_step_quad<4,3,1>", 16),
    (5, 257, "b3k_step_shared<1,1>", 5), (5, 1024, "b3k_step_shared<1,1>", 16), (5, 1025, "b3k_step<1,0>", 17),
    (3, 256, "b3k_step_quad<4,2,2>", 16), (3, 257, "b3k_step_shared<0,1>", 5), (3, 512, "b3k_step_shared<0,1>", 8),
    (3, 513, "b3k_step<1,0>", 9), (4, 128, "b3k_step_quad<8,2,1>", 8), (4, 129, "b3k_step_shared<1,1>", 6),
    (4, 1024, "b3k_step_shared<1,1>", 16), (2, 257, "b3k_step_shared<0,1>", 5),
    ((17, 17, 64, 16), 128, "b3k_step_quad<8,2,2>", 8), ((9, 8, 8, 9), 129, "b3k_step_quad<4,1,4>", 12),
    ((17, 17, 64, 17), 128, "b3k_step_shared<1,0>", 8), ((17, 17, 64, 17), 256, "b3k_step_shared<1,0>", 8),
    ((9, 11, 16, 17), 513, "b3k_step<0,0>", 9), ((9, 12, 16, 17), 513, "b3k_step_shared<1,0>", 9)])
def test_kernel_of_a_batch(caps, count, kernel, groups):
    s = sig(caps) if isinstance(caps, int) else signature(*caps)
    one, = plan([{"sig": s, "count": count, "cus": 8}])
    assert (one["create"], one["step"], one["left"]) == (0, 0, 0)
    assert [x[:2] for x in one["launches"]] == [[kernel, groups]]
    assert one["launches"][0][3] <= 160 * 1024


# The quad steps, a shared tile and shared tiles in two turns.
@pytest.mark.parametrize("scene,count,kernel", [(5, 100, "b3k_step_quad<8,2,1>"), (5, 200, "b3k_step_quad<4,3,1>"),
                                                (5, 300, "b3k_step_shared<1,1>"), (4, 600, "b3k_step_shared<1,1>")])
def test_without_room_for_the_stage(scene, count, kernel):
    """A device without room for the manifold stage steps the batch one wave
    per tile; only one without room for the worlds and their scratch refuses
    it."""
    call = {"sig": sig(scene), "count": count, "cus": 8}
    ample, = plan([call])
    assert ample["launches"][0][0] == kernel
    tight, = plan([dict(call, budget=ample["used"] - 1)])
    assert tight["create"] == 0 and tight["step"] == 0 and tight["left"] == 0
    one_wave = "b3k_step<0,0>" if scene == 4 else "b3k_step<1,0>"
    assert [x[:2] for x in tight["launches"]] == [[one_wave, (count + 63) // 64]]
    assert tight["used"] < ample["used"]
    least, less = plan([dict(call, budget=tight["used"]), dict(call, budget=tight["used"] - 1)])
    assert least["create"] == 0 and least["used"] == tight["used"]
    assert less["create"] == OUT_OF_MEMORY and less["left"] == 0
    gravity, = plan([dict(call, budget=tight["used"], step="gravity")])
    assert gravity["step"] == 0 and gravity["launches"][0][0] == "b3k_step_gravity"


# The largest batch with a wave to a world is eight turns of the waves that 8
# CUs hold: eight waves a CU for 17 bodies, five for 34, two for 68.
@pytest.mark.parametrize("caps,limit", [((17, 17, 64, 4), 512), ((34, 34, 128, 8), 320), ((68, 68, 256, 16), 128)])
def test_articulated_contacts(caps, limit):
    """Up to the limit worlds are handed to a wave each; past it, and on a
    device without room for the worlds' copy, all step 64 to a wave."""
    call = {"sig": signature(*caps), "count": limit, "cus": 8, "options": 2}
    most, past = plan([call, dict(call, count=limit + 1)])
    assert [x[:2] for x in most["launches"]] == [["b3k_step_art<0>", (limit + 63) // 64],
                                                 ["b3k_step_art_world", (limit + 127) // 128 * 128]]
    assert [x[:2] for x in past["launches"]] == [["b3k_step_art<0>", (limit + 64) // 64]]
    tight, reduced = plan([dict(call, budget=most["used"] - 1), dict(call, step="art_step")])
    assert tight["options"] == 0 and tight["step"] == 0 and tight["left"] == 0
    assert [x[:2] for x in tight["launches"]] == [["b3k_step_art<0>", (limit + 63) // 64]]
    assert [x[:2] for x in reduced["launches"]] == [["b3k_step_art<1>", (limit + 63) // 64]]


@pytest.mark.parametrize("stand,options,kernels", [
    ("libhipstand.so", 0, ["hk_step"]),
    ("libhipstand.so", 2, ["hk_action", "b3k_step_art<0>", "b3k_step_art_world", "hk_reward", "b3k_restore",
                           "hk_observe"]),
    ("libhipstand_other.so", 0, ["hk_action", "b3k_step<1,1>", "hk_reward", "b3k_restore", "hk_observe"])])
def test_hover_with_an_engine_of_another_build(stand, options, kernels):
    """The hover library steps in one launch only with the engine that it was
    built with, whose structures it reads; with another, and with articulated
    contacts, through the engine's public calls."""
    one, = plan([{"count": 130, "step": "hover", "options": options}], stand)
    assert (one["create"], one["options"], one["step"], one["left"]) == (0, 0, 0, 0)
    assert [x[0] for x in one["launches"]] == kernels
