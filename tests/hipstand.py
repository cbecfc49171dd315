"""What the engine allocates and launches, on a machine without a GPU: run as
`python hipstand.py LIBRARY < calls.json`, a process of its own in which the stand-in
for the HIP runtime (tests/emu/hipstand.c) takes the libraries' HIP calls.
`plan(calls)` runs it and returns one result per call."""
import json
import os
import re
import subprocess
import sys

TESTS = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(TESTS)


def plan(calls, stand="libhipstand.so"):
    """Each call: {"sig", "count", "cus"} and optionally "budget" (bytes of
    device memory), "options", "step" ("step", "gravity", "art_step" or
    "hover").  Each result: {"create", "options", "step"} codes, "used" and
    "peak" bytes and the step's "launches" [name, grid, block, LDS bytes]."""
    run = subprocess.run([sys.executable, os.path.abspath(__file__), stand], input=json.dumps(calls), capture_output=True,
                         text=True, timeout=120)
    assert run.returncode == 0, run.stderr
    return json.loads(run.stdout)


def template(name):
    """b3k_step_quad<8,2,1> of a mangled kernel name."""
    m = re.search(r"(hk_[a-z_]+|b3k_[a-z_]+?)(?:I((?:L[a-z]\w+?E|NS_\w+E)+)E)?Ev|(hk_[a-z_]+|b3k_[a-z_]+)", name)
    base, args = m.group(1) or m.group(3), m.group(2)
    if not args:
        return base
    return base + "<%s>" % ",".join(re.findall(r"L[a-z](\w+?)E", args))


def _main():
    sys.modules["torch"] = None            # its own HIP runtime stays out of this process
    sys.path.insert(0, ROOT)
    import ctypes as C
    stand = C.CDLL(os.path.join(TESTS, "emu", sys.argv[1]), mode=C.RTLD_GLOBAL)
    stand.hipstand_budget.argtypes = [C.c_size_t]
    stand.hipstand_used.restype = C.c_size_t
    stand.hipstand_launch.restype = C.c_char_p
    from puffysics_amd import _native
    from puffysics_amd.b3types import batch_of, empty_worlds
    lib = _native.engine_lib()
    out = []
    for call in json.loads(sys.stdin.read()):
        res = {}
        stand.hipstand_cus(call.get("cus", 256))
        stand.hipstand_budget(call.get("budget", (1 << 64) - 1))
        engine, envs = C.c_void_p(), C.c_void_p()
        if call.get("step") == "hover":
            from puffysics_amd.hover import hover_lib
            hover = hover_lib()
            config = hover.b3_hover_default_config()
            res["create"] = hover.b3_hover_create(C.byref(envs), call["count"], config, 1, 4096, 4096, 4096, 4096)
            engine = C.c_void_p(hover.b3_hover_engine(envs))
        else:
            worlds = empty_worlds(call["sig"], call["count"])
            res["create"] = lib.b3_engine_create(C.byref(engine), batch_of(worlds), call["sig"])
        res["used"] = stand.hipstand_used()
        if res["create"] == 0:
            res["options"] = lib.b3_engine_set_options(engine, call.get("options", 0))
            res["used"] = stand.hipstand_used()
            stand.hipstand_clear()
            step = call.get("step", "step")
            if step == "gravity":
                from puffysics_amd.engine import B3GravityLaw
                res["step"] = lib.b3_batch_step_gravity_gpu(engine, 0.1, 4, None, None, B3GravityLaw(1.0, 0.1), None, None)
            elif step == "art_step":
                res["step"] = lib.b3_batch_art_step_gpu(engine, 0.1, 4, None, None, None)
            elif step == "hover":
                res["step"] = hover.b3_hover_step(envs, None)
            else:
                res["step"] = lib.b3_batch_step_gpu(engine, 0.1, 4, None, None, None)
            res["launches"] = []
            for i in range(stand.hipstand_launches()):
                grid, block, lds = C.c_uint(), C.c_uint(), C.c_size_t()
                name = stand.hipstand_launch(i, C.byref(grid), C.byref(block), C.byref(lds))
                res["launches"].append([template(name.decode()), grid.value, block.value, lds.value])
            if envs:
                hover.b3_hover_destroy(envs)
            else:
                lib.b3_engine_destroy(engine)
        res["left"] = stand.hipstand_used()
        out.append(res)
    print(json.dumps(out))


if __name__ == "__main__":
    _main()
