"""Acceleration structures built with little device memory, in a process of
its own whose hipMalloc has a budget (tests/native/malloc_budget.cpp, whose
built path is the argument).  Run by tests/test_accel_gpu.py as
`python -m tests.memory_check SHIM`; prints one JSON line."""
import ctypes as C
import json
import sys

import numpy as np


def main(path):
    shim = C.CDLL(path, mode=C.RTLD_GLOBAL)
    shim.budget_room.argtypes = [C.c_size_t]
    shim.budget_used.restype = shim.budget_asked.restype = C.c_size_t
    shim.budget_asked.argtypes = [C.c_void_p, C.c_size_t]

    def asked():
        out = np.zeros(64, np.uint64)
        n = shim.budget_asked(out.ctypes.data, out.size)
        return [int(x) for x in out[:n]]

    import raymond_amd.api as api
    from tests.test_accel_gpu import description, rays_at, soup, world

    rng = np.random.default_rng(3)
    d = description(soup(rng, 100000))
    rays = rays_at(world(d), rng, 2000)
    dev = api.Device(0)
    scene = api.Scene(dev, d)
    asked()
    scene.build_accel()
    sizes = asked()  # scratch, nodes before they are counted, sources, triangles, nodes, spill rows
    assert len(sizes) == 6, sizes
    tree = sizes[3] + sizes[4]
    hits = scene.trace_closest(rays)
    out = {}

    def rebuild(name, room):
        shim.budget_room(room)
        try:
            scene.build_accel()
            shim.budget_off()
            asked()
            out[name] = all(np.array_equal(a, b) for a, b in zip(hits, scene.trace_closest(rays)))
        except api.RmError as e:
            out[name] = str(e)
        shim.budget_off()

    rebuild("no room for the scratch arrays", tree + (1 << 20))
    rebuild("room for the device build alone", sum(sizes[:4]))
    rebuild("no room beside the old tree", tree // 2)
    first, again = api.Scene(dev, d), api.Scene(dev, d)
    again.build_accel(two_level=True)
    for form, other, room in (("flat", first, tree // 2), ("two-level", again, -tree)):  # less than was in use
        shim.budget_room(room % (1 << 64))
        for name, call in (("no room", lambda: other.build_accel(two_level=form != "flat")),
                           ("trace", lambda: other.trace_closest(rays))):
            try:
                call()
                out[form + ", " + name] = True
            except api.RmError as e:
                out[form + ", " + name] = str(e)
        shim.budget_off()
        other.build_accel()
        out[form + ", room again"] = all(np.array_equal(a, b) for a, b in zip(hits, other.trace_closest(rays)))
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main(sys.argv[1])
