"""b3_batch_step_worlds_gpu, the step without allocation, against
b3_batch_step_gpu (the engine's step) on the same worlds.

The entry point steps caller-owned device B3World structs in place with its
scratch in a fixed device array of the library, a batch larger than the
array chunk after chunk.  Its results must equal the engine's word for word;
it must leave unselected worlds, corrupt worlds and the bytes around each
world (an Env struct's other fields) untouched, and refuse what it cannot
step without launching.  Two calls in a row, the second on a smaller batch
of another signature, share the array; so do two calls in flight on two
streams at once, which take turns.  A first-ever call inside HIP graph
capture sets the array up and replays like eager calls, and a warm call
takes no device memory.
"""
import numpy as np
import pytest

from b3test import clone, diff_words, oracle_run
from puffysics_amd import _native, scenes
from puffysics_amd.b3types import B3Batch

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

HIP_ERROR_INVALID_VALUE = 1
HIP_ERROR_OUT_OF_MEMORY = 2
FILL = 0xA5


def _lib():
    return _native.engine_lib()


def _to_device(worlds, stride, offset):
    """Worlds embedded at `offset` in `stride`-byte records (the rest FILL)."""
    wb = worlds.dtype.itemsize
    host = np.full((len(worlds), stride), FILL, np.uint8)
    host[:, offset:offset + wb] = worlds.view(np.uint8).reshape(len(worlds), wb)
    return torch.from_numpy(host.ravel()).cuda()


def _from_device(dev, dtype, count, stride, offset):
    host = dev.cpu().numpy().reshape(count, stride)
    wb = dtype.itemsize
    worlds = np.ascontiguousarray(host[:, offset:offset + wb]).reshape(-1).view(dtype)
    return worlds, host


def _engine_steps(worlds, sig, dt, substeps, active, steps):
    from puffysics_amd.engine import B3Engine
    eng = B3Engine(worlds, sig)
    act = None if active is None else torch.from_numpy(active).cuda()
    for _ in range(steps):
        eng.step(dt, substeps, act)
    torch.cuda.synchronize()
    out = eng.download()
    eng.close()
    return out


def _warm_worlds(scene, count, steps=10):
    worlds = scenes.build(scene, count)
    oracle_run(scene, worlds, clone(worlds), 0, steps, threads=8)
    return worlds


@pytest.mark.parametrize("order", [0, 1])
def test_no_alloc_step_equals_engine_step(order):
    """Call 1: 300 arm worlds inside 37,336-byte records at offset 32, with
    a step mask, stepped 3 times.  Call 2: 70 box-stack worlds packed, every
    world, twice.  Each equals the engine's step on the same worlds; the
    record padding and the unselected worlds keep their bytes."""
    lib = _lib()
    stream = torch.cuda.current_stream().cuda_stream
    cases = [(5, 300, 64, 32, 3), (2, 70, 0, 0, 2)]
    if order:
        cases = cases[::-1]
    for scene, count, pad, offset, steps in cases:
        sc = scenes.SCENES[scene]
        worlds = _warm_worlds(scene, count)
        wb = worlds.dtype.itemsize
        stride = wb + pad
        active = None
        if scene == 5:
            active = (np.arange(count) % 7 != 3).astype(np.uint8)
        dev = _to_device(worlds, stride, offset)
        act = None if active is None else torch.from_numpy(active).cuda()
        batch = B3Batch(dev.data_ptr(), stride, offset, count)
        for _ in range(steps):
            rc = lib.b3_batch_step_worlds_gpu(batch, sc.sig, sc.dt, sc.substeps,
                                              None if act is None else act.data_ptr(), stream)
            assert rc == 0
        torch.cuda.synchronize()
        got, raw = _from_device(dev, worlds.dtype, count, stride, offset)
        want = _engine_steps(worlds, sc.sig, sc.dt, sc.substeps, active, steps)
        bad = diff_words(got, want, sc.sig)
        assert len(bad) == 0, "scene %d: %d differing words, first %s" % (scene, len(bad), bad[:4].tolist())
        assert (raw[:, :offset] == FILL).all() and (raw[:, offset + wb:] == FILL).all()
        if active is not None:
            # raw words (indexing a structured array does not copy its padding)
            idle = active == 0
            before = worlds.view(np.uint32).reshape(count, -1)
            after = got.view(np.uint32).reshape(count, -1)
            assert (after[idle] == before[idle]).all()
        assert (got["contact_count"] > 0).any()


def test_no_alloc_step_skips_corrupt_worlds():
    """A world whose shape names a body past its body count is left exactly
    as it is; the others step as the engine steps them."""
    lib = _lib()
    scene, count = 4, 100
    sc = scenes.SCENES[scene]
    worlds = _warm_worlds(scene, count, 5)
    bad_worlds = clone(worlds)
    bad_worlds["shapes"]["body"][7, 2] = 99
    dev = _to_device(bad_worlds, worlds.dtype.itemsize, 0)
    rc = lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), worlds.dtype.itemsize, 0, count), sc.sig, sc.dt,
                                      sc.substeps, None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    got, _ = _from_device(dev, worlds.dtype, count, worlds.dtype.itemsize, 0)
    assert (got.view(np.uint32).reshape(count, -1)[7] == bad_worlds.view(np.uint32).reshape(count, -1)[7]).all()
    active = np.ones(count, np.uint8)
    active[7] = 0
    want = _engine_steps(worlds, sc.sig, sc.dt, sc.substeps, active, 1)
    keep = np.arange(count) != 7
    assert len(diff_words(got[keep], want[keep], sc.sig)) == 0


def test_no_alloc_step_runs_a_large_batch_in_chunks():
    """2,000 arm worlds with a step mask are two chunks of the 64 MiB array
    (1,152 + 848 worlds): equal to the engine's step on the same
    worlds."""
    lib = _lib()
    scene, count = 5, 2000
    sc = scenes.SCENES[scene]
    worlds = _warm_worlds(scene, count, 5)
    active = (np.arange(count) % 11 != 5).astype(np.uint8)
    dev = _to_device(worlds, worlds.dtype.itemsize, 0)
    act = torch.from_numpy(active).cuda()
    rc = lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), worlds.dtype.itemsize, 0, count), sc.sig, sc.dt,
                                      sc.substeps, act.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    got, _ = _from_device(dev, worlds.dtype, count, worlds.dtype.itemsize, 0)
    want = _engine_steps(worlds, sc.sig, sc.dt, sc.substeps, active, 1)
    bad = diff_words(got, want, sc.sig)
    assert len(bad) == 0, "%d differing words, first %s" % (len(bad), bad[:4].tolist())


def test_no_alloc_step_refuses_what_it_cannot_step():
    """Refused without a launch, the worlds untouched: a tile of worlds with
    its scratch larger than the array (4,000 contacts per world:
    hipErrorOutOfMemory); worlds or a step mask in host memory
    (hipErrorInvalidValue); invalid arguments."""
    from puffysics_amd.b3types import signature, world_dtype
    lib = _lib()
    sc = scenes.SCENES[5]
    wb = 37272
    dev = torch.full((40 * wb,), 7, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    big = signature(2, 2, 4000, 1)
    big_wb = world_dtype(big).itemsize
    assert 64 * big_wb > 64 << 20
    big_dev = torch.full((big_wb,), 7, dtype=torch.uint8, device="cuda")
    assert lib.b3_batch_step_worlds_gpu(B3Batch(big_dev.data_ptr(), big_wb, 0, 1), big, sc.dt, sc.substeps, None,
                                        stream) == HIP_ERROR_OUT_OF_MEMORY
    host = np.full(10 * wb, 7, np.uint8)
    assert lib.b3_batch_step_worlds_gpu(B3Batch(host.ctypes.data, wb, 0, 10), sc.sig, sc.dt, sc.substeps, None,
                                        stream) == HIP_ERROR_INVALID_VALUE
    host_mask = np.ones(10, np.uint8)
    assert lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), wb, 0, 10), sc.sig, sc.dt, sc.substeps,
                                        host_mask.ctypes.data, stream) == HIP_ERROR_INVALID_VALUE
    assert lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), wb - 4, 0, 10), sc.sig, sc.dt, sc.substeps,
                                        None, stream) != 0
    assert lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr() + 2, wb, 0, 10), sc.sig, sc.dt, sc.substeps,
                                        None, stream) != 0
    assert lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), wb, 0, 10), sc.sig, float("nan"), sc.substeps,
                                        None, stream) != 0
    assert lib.b3_batch_step_worlds_gpu(B3Batch(None, wb, 0, 0), sc.sig, sc.dt, sc.substeps, None, stream) == 0
    torch.cuda.synchronize()
    assert int((dev != 7).sum()) == 0 and int((big_dev != 7).sum()) == 0
    assert (host == 7).all()
    # the refusals leave no error behind for the next call
    small = _warm_worlds(2, 64, 3)
    d2 = _to_device(small, small.dtype.itemsize, 0)
    s2 = scenes.SCENES[2]
    assert lib.b3_batch_step_worlds_gpu(B3Batch(d2.data_ptr(), small.dtype.itemsize, 0, 64), s2.sig, s2.dt,
                                        s2.substeps, None, stream) == 0
    torch.cuda.synchronize()


def test_no_alloc_calls_on_two_streams_take_turns():
    """300 arm worlds on one stream and 200 box stacks on another, issued
    back to back with no synchronisation between them, both through the
    one array: each batch equals the engine's step of it."""
    lib = _lib()
    cases = [(5, 300), (2, 200)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    devs, inputs = [], []
    for scene, count in cases:
        worlds = _warm_worlds(scene, count, 5)
        inputs.append(worlds)
        devs.append(_to_device(worlds, worlds.dtype.itemsize, 0))
    torch.cuda.synchronize()
    for rep in range(3):
        for (scene, count), dev, worlds, st in zip(cases, devs, inputs, streams):
            sc = scenes.SCENES[scene]
            rc = lib.b3_batch_step_worlds_gpu(B3Batch(dev.data_ptr(), worlds.dtype.itemsize, 0, count), sc.sig,
                                              sc.dt, sc.substeps, None, st.cuda_stream)
            assert rc == 0
    torch.cuda.synchronize()
    for (scene, count), dev, worlds in zip(cases, devs, inputs):
        sc = scenes.SCENES[scene]
        got, _ = _from_device(dev, worlds.dtype, count, worlds.dtype.itemsize, 0)
        want = _engine_steps(worlds, sc.sig, sc.dt, sc.substeps, None, 3)
        bad = diff_words(got, want, sc.sig)
        assert len(bad) == 0, "scene %d: %d differing words, first %s" % (scene, len(bad), bad[:4].tolist())


CAPTURE_SCRIPT = r"""
import sys
import numpy as np
import torch
sys.path[:0] = [%(root)r, %(tests)r]
from b3test import clone, diff_words, oracle_run
from puffysics_amd import _native, scenes
from puffysics_amd.b3types import B3Batch

lib = _native.engine_lib()
scene, count = 2, 200
sc = scenes.SCENES[scene]
worlds = scenes.build(scene, count)
oracle_run(scene, worlds, clone(worlds), 0, 5)
wb = worlds.dtype.itemsize
raw = worlds.view(np.uint8)
graphed = torch.from_numpy(raw.copy()).cuda()
eager = torch.from_numpy(raw.copy()).cuda()
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    # the first call of this process: the array is set up under capture
    rc = lib.b3_batch_step_worlds_gpu(B3Batch(graphed.data_ptr(), wb, 0, count), sc.sig, sc.dt, sc.substeps,
                                      None, torch.cuda.current_stream().cuda_stream)
assert rc == 0, rc
torch.cuda.synchronize()
assert bool((graphed.cpu().numpy() == raw).all()), "capture ran the step"
stream = torch.cuda.current_stream().cuda_stream
for r in range(3):
    graph.replay()
    assert lib.b3_batch_step_worlds_gpu(B3Batch(eager.data_ptr(), wb, 0, count), sc.sig, sc.dt, sc.substeps,
                                        None, stream) == 0
    torch.cuda.synchronize()
    a = graphed.cpu().numpy().view(worlds.dtype)
    b = eager.cpu().numpy().view(worlds.dtype)
    bad = diff_words(a, b, sc.sig)
    assert len(bad) == 0, "replay %%d: %%d differing words" %% (r, len(bad))
free_before = torch.cuda.mem_get_info()[0]
assert lib.b3_batch_step_worlds_gpu(B3Batch(eager.data_ptr(), wb, 0, count), sc.sig, sc.dt, sc.substeps, None,
                                    stream) == 0
torch.cuda.synchronize()
free_after = torch.cuda.mem_get_info()[0]
assert free_after == free_before, (free_before, free_after)
print("capture ok", flush=True)
"""


def test_no_alloc_first_call_under_graph_capture():
    """In a fresh process, the first call is made inside torch.cuda.graph
    capture: it returns hipSuccess, the capture runs nothing, and each
    replay equals an eager call on a twin copy of the worlds.  Afterwards a
    warm call leaves the device's free memory unchanged."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    script = CAPTURE_SCRIPT % {"root": root, "tests": os.path.join(root, "tests")}
    out = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-4000:]
    assert "capture ok" in out.stdout
