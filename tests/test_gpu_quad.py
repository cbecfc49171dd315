"""The step on quads of lanes (b3k_step_quad: a quarter tile to a workgroup,
one contact or joint solve to four lanes) and the batch sizes at which the
other step kernels take over, against the oracle word for word (the step's
contract is the reference's fp32 bits, so the tolerance is zero).
"""
import numpy as np
import pytest

from b3test import clone, diff_words, feature_worlds, gpu_run, oracle_run, oracle_step_batch
from puffysics_amd import scenes
from puffysics_amd.b3types import empty_worlds, signature

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _engine(worlds, sig):
    from puffysics_amd.engine import B3_ENGINE_KEEP_SOLVER_FIELDS, B3Engine
    eng = B3Engine(worlds, sig)
    eng.set_options(B3_ENGINE_KEEP_SOLVER_FIELDS)
    return eng


def _same(eng, ref, sig):
    torch.cuda.synchronize()
    bad = diff_words(eng.download(), ref, sig)
    eng.close()
    assert len(bad) == 0, "%d differing words, first %s" % (len(bad), bad[:4].tolist())


# One world, the edges of a workgroup's 16 worlds and of a 64-world tile;
# then batches on both sides of a quarter and of half a tile per CU (64 and
# 128 tiles on 256 CUs), and chains on the most shared tiles of one turn.
@pytest.mark.parametrize("scene,count,steps", [
    (1, 1, 40), (1, 17, 40), (2, 15, 30), (2, 65, 30), (3, 16, 20), (3, 33, 20), (4, 1, 60), (4, 31, 25), (5, 63, 25),
    (5, 49, 25), (2, 4096, 4), (2, 4097, 4), (3, 4100, 3), (4, 4100, 2), (5, 4100, 4), (3, 8192, 3), (5, 8200, 3), (2, 8200, 3),
    (3, 8200, 3), (3, 16384, 2)])
def test_batch_edges(scene, count, steps):
    worlds = scenes.build(scene, count)
    ref = clone(worlds)
    oracle_run(scene, ref, clone(worlds), 0, steps, threads=8)
    eng = _engine(worlds, scenes.SCENES[scene].sig)
    gpu_run(eng, scene, 0, steps)
    _same(eng, ref, scenes.SCENES[scene].sig)


def _enlarge(worlds, sig, bodies=1):
    """The worlds in a larger capacity set, `bodies` copies of each world's
    bodies, shapes and joints side by side in one world (the copies 40 m
    apart, so that they do not touch)."""
    out = empty_worlds(sig, len(worlds))
    for f in worlds.dtype.names:
        if f not in ("bodies", "shapes", "contacts", "joints"):
            out[f] = worlds[f]
    nb, ns, nj = (int(worlds[f][0]) for f in ("body_count", "shape_count", "joint_count"))
    assert all((worlds[f] == n).all() for f, n in (("body_count", nb), ("shape_count", ns), ("joint_count", nj)))
    for k in range(bodies):
        out["bodies"][:, k * nb:(k + 1) * nb] = worlds["bodies"][:, :nb]
        for f in ("position", "center"):
            out["bodies"][f]["x"][:, k * nb:(k + 1) * nb] += 40.0 * k
        out["shapes"][:, k * ns:(k + 1) * ns] = worlds["shapes"][:, :ns]
        out["shapes"]["body"][:, k * ns:(k + 1) * ns] += k * nb
        out["joints"][:, k * nj:(k + 1) * nj] = worlds["joints"][:, :nj]
        for f in ("body_a", "body_b"):
            out["joints"][f][:, k * nj:(k + 1) * nj] += k * nb
    out["body_count"], out["shape_count"], out["joint_count"] = bodies * nb, bodies * ns, bodies * nj
    return out


# Joints past one to a wave (max_joints 8 < n <= 16), and past what the quad
# step takes (17 and more: the shared tiles).
@pytest.mark.parametrize("copies,caps", [(1, (9, 8, 8, 9)), (2, (18, 16, 32, 16)), (2, (18, 16, 32, 17)),
                                         (3, (27, 24, 32, 24))])
@pytest.mark.parametrize("count", [20, 4100])
def test_many_joints(copies, caps, count):
    sig = signature(*caps)
    worlds = _enlarge(scenes.build(3, count), sig, copies)
    rng = np.random.default_rng(3)
    worlds["joints"]["target_angle"][:] = rng.uniform(-0.5, 0.5, worlds["joints"]["target_angle"].shape)
    ref = clone(worlds)
    eng = _engine(worlds, sig)
    for _ in range(12 if count < 100 else 2):
        oracle_step_batch(ref, sig, 1.0 / 120.0, 4)
        eng.step(1.0 / 120.0, 4)
    assert np.abs(ref["joints"]["spring_impulse"][:, :8 * copies]).min(axis=0).max() > 0
    _same(eng, ref, sig)


@pytest.mark.parametrize("capacity", [128, 40, 7])
def test_contacts_past_the_kept_rows(capacity):
    """The bin's ~40 contacts a world: more than the waves keep in
    registers, and a capacity that drops some."""
    sig = signature(33, 37, capacity, 1)
    worlds = _enlarge(scenes.build(4, 20), sig)
    ref = clone(worlds)
    eng = _engine(worlds, sig)
    for _ in range(45):
        oracle_step_batch(ref, sig, 1.0 / 60.0, 4)
        eng.step(1.0 / 60.0, 4)
    assert ref["contact_count"].max() >= min(capacity, 24)
    assert capacity > 16 or ref["contacts_dropped"].max() > 0
    _same(eng, ref, sig)


def test_unsorted_old_contacts():
    """Uploaded contacts out of shape order (the warm start then searches
    them all, the last match winning), on the coverage worlds."""
    from puffysics_amd.creation import CUSTOM_SIG
    worlds = feature_worlds(40)
    for _ in range(30):
        oracle_step_batch(worlds, CUSTOM_SIG, 1.0 / 60.0, 4)
    for k in range(0, 40, 2):
        n = int(worlds["contact_count"][k])
        if n > 1:
            worlds["contacts"][k, :n] = worlds["contacts"][k, :n][::-1].copy()
    ref = clone(worlds)
    eng = _engine(worlds, CUSTOM_SIG)
    for _ in range(3):
        oracle_step_batch(ref, CUSTOM_SIG, 1.0 / 60.0, 3)
        eng.step(1.0 / 60.0, 3)
    assert (ref["contact_count"] > 1).any()
    _same(eng, ref, CUSTOM_SIG)


# 0: the step on quads; 4: one wave per tile.
@pytest.mark.parametrize("options", [0, 4])
def test_joint_of_a_body_with_itself(options):
    """Welds and hinges whose two ends are one body (the creation API takes
    them): the warm start moves the body by end a and then, from there, by
    end b."""
    from puffysics_amd.creation import CUSTOM_SIG
    worlds = feature_worlds(20)
    for k in range(20):
        for j in range(k % 2, int(worlds["joint_count"][k]), 2):
            worlds["joints"]["body_a"][k, j] = worlds["joints"]["body_b"][k, j]
    ref = clone(worlds)
    eng = _engine(worlds, CUSTOM_SIG)
    eng.set_options(1 | options)
    for _ in range(6):
        oracle_step_batch(ref, CUSTOM_SIG, 1.0 / 60.0, 4)
        eng.step(1.0 / 60.0, 4)
    own = ref["joints"]["body_a"] == ref["joints"]["body_b"]
    assert (np.abs(ref["joints"]["linear_impulse"]["x"]) > 0)[own].any() and np.isfinite(ref["bodies"]["lin_vel"]["x"]).all()
    _same(eng, ref, CUSTOM_SIG)


def _step_worlds(worlds, sig, steps, dt, substeps, active=None, pad=0):
    """`steps` calls of b3_batch_step_worlds_gpu on a device copy of the
    worlds, `pad` bytes apart."""
    from puffysics_amd import _native
    from puffysics_amd.b3types import B3Batch
    n, wb = len(worlds), worlds.dtype.itemsize
    host = np.full((n, wb + pad), 0x5a, np.uint8)
    host[:, :wb] = worlds.view(np.uint8).reshape(n, wb)
    dev = torch.from_numpy(host).cuda()
    act = None if active is None else torch.from_numpy(active).cuda()
    for _ in range(steps):
        rc = _native.engine_lib().b3_batch_step_worlds_gpu(
            B3Batch(dev.data_ptr(), wb + pad, 0, n), sig, dt, substeps, None if act is None else act.data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        assert rc == 0
    torch.cuda.synchronize()
    out = dev.cpu().numpy()
    assert (out[:, wb:] == 0x5a).all()
    return np.ascontiguousarray(out[:, :wb]).view(worlds.dtype).reshape(n)


# In place on quads: one world, a part of a workgroup, chunks of the array
# (1,300 arm worlds are two); staged as tiles: more than 16 joints.
@pytest.mark.parametrize("scene,count,steps,pad", [(1, 1, 30, 4), (5, 17, 20, 0), (5, 1300, 3, 12), (4, 300, 3, 0),
                                                   (2, 1000, 3, 8)])
def test_step_worlds_edges(scene, count, steps, pad):
    sc = scenes.SCENES[scene]
    worlds = scenes.build(scene, count)
    oracle_run(scene, worlds, clone(worlds), 0, 25, threads=8)
    ref = clone(worlds)
    active = (np.arange(count) % 5 != 3).astype(np.uint8)
    for _ in range(steps):
        oracle_step_batch(ref, sc.sig, sc.dt, sc.substeps, active)
    got = _step_worlds(worlds, sc.sig, steps, sc.dt, sc.substeps, active, pad)
    diff = diff_words(got, ref, sc.sig)
    from b3test import solver_field_words
    allowed = solver_field_words(ref)              # not written back by this call
    assert allowed[diff[:, 0], diff[:, 1]].all(), diff[:4].tolist()
    idle = active == 0
    raw = [x.view(np.uint32).reshape(count, -1)[idle] for x in (got, worlds)]   # with the structs' padding
    assert (raw[0] == raw[1]).all()


def test_step_worlds_staged():
    sig = signature(27, 24, 32, 24)
    worlds = _enlarge(scenes.build(3, 70), sig, 3)
    ref = clone(worlds)
    for _ in range(4):
        oracle_step_batch(ref, sig, 1.0 / 120.0, 4)
    got = _step_worlds(worlds, sig, 4, 1.0 / 120.0, 4)
    assert len(diff_words(got, ref, sig)) == 0


# Gravity: a worker sums one body's pairs, with the masses of the bodies and
# with the caller's; four-wave workgroups past a quarter tile per CU; at one
# lane a world past half a tile per CU.
@pytest.mark.parametrize("scene,count,steps,caller", [(4, 20, 12, False), (2, 65, 12, True), (5, 33, 6, True),
                                                      (2, 4100, 2, True), (2, 8200, 2, False)])
def test_gravity(scene, count, steps, caller):
    from b3test import oracle_step_gravity
    sc = scenes.SCENES[scene]
    worlds = scenes.build(scene, count)
    masses = None
    if caller:
        masses = np.random.default_rng(2).uniform(0.0, 3.0, (count, sc.caps[0])).astype(np.float32)
        masses[:, 2] = 0.0                         # a body that neither feels nor sources it
        masses[::2, 0] = 5.0                       # the static ground as a source
    ref = clone(worlds)
    eng = _engine(worlds, sc.sig)
    dev = None if masses is None else torch.from_numpy(masses).cuda()
    for _ in range(steps):
        oracle_step_gravity(ref, sc.sig, sc.dt, sc.substeps, 4.0, 0.15, masses)
        eng.step_gravity(sc.dt, sc.substeps, 4.0, 0.15, dev)
    _same(eng, ref, sc.sig)
