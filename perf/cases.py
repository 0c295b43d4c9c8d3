"""The work a user of raymond_amd has it do, as measurable cases.

A case is a dict of plain values; `kind` selects the entry points it runs:

  render    Renderer.reset / execute / image (or resolve): a frame of a scene
  batch     Batch.render / image: uneven jobs in one bounce loop
  cached    Renderer with a frozen RadianceCache attached (mode 2)
  queries   Scene.trace_closest and Scene.trace_any on host ray arrays
  device    Scene.trace_closest_noalloc on device ray arrays
  network   RadianceCache.infer and RadianceCache.gradients on a host batch
  setup     Scene.build_accel, build_envmap and the first rays through them

prepare(case, seed) draws geometry placement, camera, rays or features from
the seed; the material libraries are the bundled scenes' (their code objects
are compiled with the library).
"""
import functools
import math

import numpy as np
import torch

import raymond_amd.api as api
import raymond_amd.scenes as scenes

PRIMES = (1, 3, 7, 13, 29)


def listed():
    return [
        # the smallest call: one sample of a thumbnail, as an interactive
        # preview renders after every edit; launches and waits dominate
        dict(name="preview 64x64", kind="render", scene="cornell", width=64, height=64, depth=8, rr=3, spp=1, spl=1,
             sort=0, show=1),
        # a still of a small scene: trees two levels deep, shading and queues
        dict(name="cornell 512x512", kind="render", scene="cornell", width=512, height=512, depth=8, rr=3, spp=32,
             spl=32, sort=1, show=0),
        # the benchmark's headline: 5.2M triangles, full HD, depth 12
        dict(name="sphere field 1080p", kind="render", scene="spheres", spheres=64, level=6, width=1920, height=1080,
             depth=12, rr=0, spp=16, spl=8, sort=1, show=0),
        # large node-graph materials, shading sorted by material
        dict(name="graphs 1280x720", kind="render", scene="graphs", materials=32, width=1280, height=720, depth=8,
             rr=0, spp=4, spl=4, sort=1, show=0),
        # instancing: 256 placed copies of 4 shapes through the two-level tree
        dict(name="instances 1080p", kind="render", scene="instances", instances=256, level=5, width=1920, height=1080,
             depth=8, rr=0, spp=8, spl=8, sort=1, show=0),
        # every analytic lamp through a spectral lens, at an odd size, unsorted,
        # with more samples than the queue holds (paths regenerate)
        dict(name="lens 501x333", kind="render", scene="lens", width=501, height=333, depth=8, rr=0, spp=24, spl=8,
             sort=0, show=1),
        # a render farm's mix: uneven jobs sharing the queues
        dict(name="batch of 6 jobs", kind="batch", jobs=6, triangles=200000, edge=640, spp=24, depth=10, pick=3),
        # a frame that ends its paths in a trained cache
        dict(name="cached 1080p", kind="cached", width=1920, height=1080, depth=12, rr=3, spp=8, spl=8, log2=15),
        # baking: a large host batch of visibility queries
        dict(name="queries 1M", kind="queries", spheres=16, level=5, rays=1048576, two_level=0),
        # a picking or sensor loop on device arrays, ragged size
        dict(name="device rays 100003", kind="device", spheres=4, level=5, rays=100003, two_level=0),
        # one step of fitting the network outside a render, default table
        dict(name="network batch 8192", kind="network", rows=8192, log2=19),
        # opening a scene: acceleration structure, importance map, first rays
        dict(name="setup 1.3M triangles", kind="setup", spheres=16, level=6, rays=65536, env=2048, two_level=0),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["cornell", "spheres", "graphs", "instances", "lens", "batch", "cached", "queries", "device",
                       "network", "setup"])
    w = size(48, 1600)
    h = max(32, int(w * rng.uniform(0.5, 1.0)))
    spl = max(1, min(size(1, 16), (1 << 23) // (w * h)))
    spp = max(1, min(size(1, 32), (1 << 24) // (w * h)))
    frame = dict(kind="render", width=w, height=h, depth=rng.randint(4, 12), rr=rng.choice([0, 3]), spp=spp, spl=spl,
                 sort=rng.choice([0, 1]), show=rng.choice([0, 1]))
    if kind == "cornell":
        return dict(frame, scene="cornell")
    if kind == "spheres":
        return dict(frame, scene="spheres", spheres=rng.randint(1, 24), level=rng.randint(3, 6))
    if kind == "graphs":
        return dict(frame, scene="graphs", materials=8, sort=1)
    if kind == "instances":
        return dict(frame, scene="instances", instances=size(2, 600), level=rng.randint(2, 5))
    if kind == "lens":
        return dict(frame, scene="lens")
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(2, 8), triangles=size(1000, 200000), edge=size(64, 640),
                    spp=rng.randint(2, 24), depth=rng.randint(6, 12), pick=rng.randint(0, 1000))
    if kind == "cached":
        return dict(kind="cached", width=w, height=h, depth=rng.randint(6, 12), rr=3, spp=min(spp, 8),
                    spl=min(spl, 8), log2=rng.choice([15, 17, 19]))
    if kind == "queries":
        return dict(kind="queries", spheres=rng.randint(1, 24), level=rng.randint(2, 5), rays=size(257, 1000000),
                    two_level=rng.choice([0, 1]))
    if kind == "device":
        return dict(kind="device", spheres=rng.randint(1, 4), level=rng.randint(2, 5), rays=size(64, 262144),
                    two_level=rng.choice([0, 1]))
    if kind == "network":
        return dict(kind="network", rows=size(33, 65536), log2=rng.choice([12, 15, 17, 19]))
    return dict(kind="setup", spheres=rng.randint(1, 16), level=rng.randint(3, 6), rays=size(64, 65536),
                env=rng.choice([256, 512, 1024, 2048]), two_level=rng.choice([0, 1]))


# ---------------------------------------------------------------------------
# Inputs


@functools.lru_cache(None)
def device():
    return api.Device(0)


@functools.lru_cache(None)
def library():
    """Materials of the benchmark's sphere field: 64 Principled and the ground."""
    d = scenes.sphere_field(64, 64, grid=8, level=0)
    return d.surface_materials, d.light_materials


@functools.lru_cache(None)
def blob(level, which):
    """A noise-displaced icosphere around the origin, as the sphere field's."""
    v0, f0 = scenes.icosphere(level)
    v = v0 * (0.4 + 0.05 * scenes.value_noise(v0, 1000 + which))[:, None]
    return scenes.Shape(v, scenes.vertex_normals(v, f0), f0, 0)


def turned(rng, place, size):
    a, b = rng.uniform(0.0, 2.0 * math.pi, 2)
    rx = np.eye(4)
    rx[1:3, 1:3] = [[math.cos(b), -math.sin(b)], [math.sin(b), math.cos(b)]]
    return scenes.translate(place) @ scenes.rotate_z(math.degrees(a)) @ rx @ scenes.scale((size, size, size))


def placed(rng, n):
    """n jittered grid places in an 8 x 8 field, and the grid spacing."""
    g = int(math.ceil(math.sqrt(n)))
    step = 8.0 / max(g, 4)
    k = np.arange(n)
    xy = np.stack([k % g, k // g], 1) - (g - 1) / 2.0 + rng.uniform(-0.25, 0.25, (n, 2))
    return xy * step, step


def field(rng, shapes_n, level, instances=0, env=2048):
    """The sphere field's materials, sky and ground over seeded placements:
    one shape per sphere, or `instances` copies of 4 shapes."""
    d = scenes.SceneDescription("field")
    d.surface_materials, d.light_materials = library()
    d.envmap_resolution = env
    n = instances or shapes_n
    xy, step = placed(rng, n)
    ids = []
    for i in range(4 if instances else n):
        b = blob(level, i % 4)
        s = scenes.Shape(b.vertices, b.normals, b.faces, i, b.texcoords)
        ids.append(d.add_shape(s))
    for i in range(n):
        size = step * (rng.uniform(0.6, 1.4) if instances else 1.0)
        d.add_entity(ids[i % len(ids)], turned(rng, (xy[i, 0], xy[i, 1], 0.4 * size), size))
    g = 50.0
    d.add_entity(d.add_shape(scenes.merge([scenes.quad((-g, -g, 0), (g, -g, 0), (g, g, 0), (-g, g, 0), 64)])))
    eye = np.array([0.0, -8.5, 5.5]) + rng.uniform(-0.4, 0.4, 3)
    d.camera = dict(transform=scenes.look_at(eye, (0.0, 0.3, 0.0)), near=1e-3, far=1e4, focal=2.0)
    return d


def box(rng, d):
    """A Cornell-box scene seen from a seeded place in front of it."""
    d.envmap_resolution = 64  # black world
    eye = np.array([0.5, -1.35, 0.5]) + rng.uniform(-0.1, 0.1, 3)
    d.camera = dict(transform=scenes.look_at(eye, (0.5, 0.5, 0.5)), near=1e-3, far=1e4, focal=2.4)
    return d


def scene_of(case, rng):
    name = case["scene"]
    if name == "cornell":
        return box(rng, scenes.cornell_box(case["width"], case["height"]))
    if name == "lens":
        return box(rng, scenes.lamp_box(case["width"], case["height"]))
    if name == "graphs":
        return box(rng, scenes.shader_graph_scene(case["width"], case["height"], materials=case["materials"]))
    if name == "instances":
        return field(rng, 0, case["level"], instances=case["instances"])
    return field(rng, case["spheres"], case["level"])


def lens():
    """The singlet focused at infinity, opened and scaled for a 1-unit room."""
    surfaces = scenes.singlet_lens(50.0, 2.8)
    return api.lens_desc(surfaces, stop_index=3, relative_stop=0.7, camera_scale=0.01, spectral=True)


def ray_batch(rng, n, bounded):
    """Half camera-like rays over the field, half rays leaving its surfaces."""
    k = n // 2
    o = np.empty((n, 3))
    t = np.empty((n, 3))
    o[:k] = np.array([0.0, -8.5, 5.5]) + rng.normal(0.0, 0.01, (k, 3))
    t[:k] = np.concatenate([rng.uniform(-4.5, 4.5, (k, 2)), rng.uniform(0.0, 0.8, (k, 1))], 1)
    o[k:] = np.concatenate([rng.uniform(-4.0, 4.0, (n - k, 2)), rng.uniform(0.01, 0.9, (n - k, 1))], 1)
    t[k:] = o[k:] + rng.normal(0.0, 1.0, (n - k, 3))
    d = t - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    far = rng.uniform(0.5, 12.0, n) if bounded else np.full(n, 1e4)
    return np.concatenate([o, np.full((n, 1), 1e-4), d, far[:, None]], 1).astype(np.float32)


def network_batch(rng, n):
    """Vertex features in the ranges a render records: positions on a few
    surfaces of the unit box, directions, roughness, albedo, lobe share."""
    f = rng.uniform(0.0, 1.0, (n, api.CACHE_FEATURES))
    wall = rng.integers(0, 3, n)
    f[np.arange(n), wall] = rng.integers(0, 2, n) * 0.98 + 0.01
    f[:, 7] = rng.choice([0.4, 1.0], n)
    f[:, 11] = rng.choice([0.0, 0.5], n)
    targets = rng.gamma(0.7, 0.6, (n, 3))
    return f.astype(np.float32), targets.astype(np.float32)


def network_params(rng, log2):
    """Weights and a table as after some training: Glorot-scaled layers over
    the inputs in use, table entries of the size Adam reaches."""
    mlp = np.zeros(api.CACHE_MLP_PARAMS, np.float32)
    w1, w2, w3 = mlp[:3072].reshape(48, 64), mlp[3072:7168].reshape(64, 64), mlp[7168:].reshape(64, 32)
    w1[:42] = rng.uniform(-0.24, 0.24, (42, 64))
    w2[:] = rng.uniform(-0.22, 0.22, (64, 64))
    w3[:, :3] = rng.uniform(-0.3, 0.3, (64, 3))
    return mlp, rng.uniform(-0.5, 0.5, 16 * 2 ** log2 * 2).astype(np.float32)


def prepare(case, seed):
    rng = np.random.default_rng([seed, 17])
    dev, kind = device(), case["kind"]
    state = {"case": case}
    if kind == "render":
        scene = scenes.build_device_scene(dev, scene_of(case, rng), two_level=case["scene"] == "instances",
                                          noinline=False if case["scene"] == "graphs" else None)
        r = api.Renderer(scene, case["width"], case["height"], max_depth=case["depth"],
                         samples_per_launch=case["spl"])
        r.set_uniforms(rr_depth=case["rr"], material_sort=case["sort"])
        if case["scene"] == "lens":
            r.set_lens(lens())
        state["renderer"] = r
    elif kind == "cached":
        scene = scenes.build_device_scene(dev, box(rng, scenes.cornell_box(case["width"], case["height"])))
        r = api.Renderer(scene, case["width"], case["height"], max_depth=case["depth"],
                         samples_per_launch=case["spl"])
        r.set_uniforms(rr_depth=case["rr"], material_sort=1)
        cache = api.RadianceCache(dev, log2_table_size=case["log2"], seed=seed % 1000)
        cache.write_params(*network_params(rng, case["log2"]))
        r.set_cache(cache, mode=2)
        state["renderer"] = r
    elif kind == "batch":
        mix = np.random.default_rng(case["pick"])
        jobs = []
        for k in range(case["jobs"]):
            tris = int(math.exp(mix.uniform(math.log(1000), math.log(max(1001, case["triangles"])))))
            edge = max(16, case["edge"] // int(mix.integers(1, 4)) - PRIMES[k % 5])
            spp = max(1, case["spp"] // int(mix.integers(1, 5)))
            d = box(rng, scenes.tessellated_cornell_box(edge, edge, tris))
            scene = scenes.build_device_scene(dev, d)
            jobs.append((scene, edge, max(16, edge * 3 // 4), spp, case["depth"] - k % 3, 1 + k))
        state["batch"] = api.Batch(dev, jobs)
        state["jobs"] = len(jobs)
    elif kind in ("queries", "device", "setup"):
        d = field(rng, case["spheres"], case["level"], env=case.get("env", 64))
        state["scene"] = scene = api.Scene(dev, d)
        if kind == "setup":
            scene.compile_materials(d.material_source())
            state["rays"] = ray_batch(rng, case["rays"], False)
            return state
        scene.build_accel(two_level=bool(case["two_level"]))
        rays = ray_batch(rng, case["rays"], False)
        if kind == "queries":
            state["rays"], state["shadow"] = rays, ray_batch(rng, case["rays"], True)
            return state
        n = case["rays"]
        state["rays"] = torch.from_numpy(rays).cuda()
        for name, shape, dtype in (("t", (n,), torch.float32), ("inst", (n,), torch.int32),
                                   ("prim", (n,), torch.int32), ("bary", (n, 2), torch.float32)):
            state[name] = torch.empty(shape, dtype=dtype, device="cuda")
        torch.cuda.synchronize()
    else:
        cache = api.RadianceCache(dev, log2_table_size=case["log2"], seed=seed % 1000)
        cache.write_params(*network_params(rng, case["log2"]))
        state["cache"] = cache
        state["features"], state["targets"] = network_batch(rng, case["rows"])
    return state


# ---------------------------------------------------------------------------
# One pass


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("render", "cached"):
        r = state["renderer"]
        r.reset()
        st = r.execute(case["spp"])
        return {"image": r.resolve() if case.get("show") else r.image(), "rays": int(st.total_rays)}
    if kind == "batch":
        b = state["batch"]
        st = b.render(rr_depth=3)
        return {"images": [b.image(k) for k in range(state["jobs"])], "rays": int(st.total_rays)}
    if kind == "queries":
        t, inst, prim, bary = state["scene"].trace_closest(state["rays"])
        occluded = state["scene"].trace_any(state["shadow"])
        return {"t": t, "inst": inst, "prim": prim, "bary": bary, "occluded": occluded}
    if kind == "device":
        s = state
        s["scene"].trace_closest_noalloc(s["rays"].data_ptr(), case["rays"], s["t"].data_ptr(), s["inst"].data_ptr(),
                                         s["prim"].data_ptr(), s["bary"].data_ptr())
        return {"t": s["t"], "inst": s["inst"], "prim": s["prim"], "bary": s["bary"]}
    if kind == "network":
        c = state["cache"]
        out = c.infer(state["features"])
        gm, gt, loss = c.gradients(state["features"], state["targets"])
        return {"out": out, "grad_mlp": gm, "grad_table": gt, "loss": loss}
    scene = state["scene"]
    scene.build_accel(two_level=bool(case["two_level"]))
    scene.build_envmap()
    pdfs, mip = scene.read_envmap()
    t, inst, prim, bary = scene.trace_closest(state["rays"])
    return {"pdfs": pdfs, "mip": mip, "t": t, "inst": inst, "prim": prim, "bary": bary}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far two correct results may differ

RAY_FLOPS = 12 * 8 * 12 + 4 * 60  # a dozen 8-wide node visits, a few triangle tests
TRI_BYTES = 36                    # three vertices
ROW_FLOPS = 2 * (48 * 64 + 64 * 64 + 64 * 3) + 16 * 8 * 8


def triangles(case):
    scene = case.get("scene", "field")
    if scene in ("cornell", "lens", "graphs") or case["kind"] == "cached":
        return 36
    shapes = 4 if scene == "instances" else case["spheres"]
    return shapes * 20 * 4 ** case["level"] + 2


def work(case):
    kind = case["kind"]
    if kind in ("render", "cached"):
        paths = case["width"] * case["height"] * case["spp"]
        vertices = 2.0 if kind == "cached" else 2.2
        shade = 4000 if case.get("scene") == "graphs" else 800
        return {"bytes": 16 * case["width"] * case["height"] + TRI_BYTES * triangles(case),
                "flops": paths * vertices * (1.6 * RAY_FLOPS + shade)}
    if kind == "batch":
        pixels = case["jobs"] * (case["edge"] / 2.0) ** 2 * 0.75
        return {"bytes": 16 * pixels + TRI_BYTES * case["jobs"] * case["triangles"] / 4.0,
                "flops": pixels * case["spp"] / 2.0 * 3.0 * (1.6 * RAY_FLOPS + 800)}
    if kind == "queries":
        return {"bytes": case["rays"] * (32 + 20 + 32 + 4) + TRI_BYTES * triangles(case),
                "flops": 2.0 * case["rays"] * RAY_FLOPS}
    if kind == "device":
        return {"bytes": case["rays"] * (32 + 20) + TRI_BYTES * triangles(case), "flops": case["rays"] * RAY_FLOPS}
    if kind == "network":
        table = 16 * 2 ** case["log2"] * 2
        return {"bytes": case["rows"] * (48 + 12 + 12) + table * (2 + 4) + 9216 * 8, "flops": 4.0 * case["rows"] * ROW_FLOPS}
    n = triangles(case)
    return {"bytes": n * (TRI_BYTES + 48 + 20) + 4 * case["env"] ** 2 * 2.34 + case["rays"] * 52,
            "flops": n * 20 * 30 + 64.0 * case["env"] ** 2 * 150 + case["rays"] * RAY_FLOPS}


def tolerance(case):
    kind = case["kind"]
    if kind in ("render", "cached", "batch"):
        # samples add into a pixel in any order, in 32 bits (two runs differ by
        # up to 4e-8, a pixel by 3.4e-7); the paths themselves follow one
        # random stream each
        return {"rel": 5e-7, "max": 5e-6}
    if kind == "network":
        # FP16 operands and FP16 table-gradient sums, in any order: two runs
        # differ by 5e-4, an entry by 0.01 of the root mean square
        return {"rel": 2e-3, "max": 0.08}
    if kind == "setup":
        return {"rel": 1e-6}  # 32-bit sums; hits are those of the queries
    # the nearest hit, ties to the smaller ids: independent of any order
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch


def exact(case, seed):
    kind = case["kind"]
    if kind == "network":
        return exact_network(case, seed)
    if kind == "device" and not case["two_level"] and case["rays"] * triangles(case) <= 1 << 34:
        return exact_hits(case, seed)
    # a render's paths and an importance map follow random streams through the
    # scene's generated shaders: no plain-torch form of useful speed.  The
    # larger ray batches take over 20 seconds exhaustively.
    return None


def exact_hits(case, seed):
    """Nearest hit of every ray against every triangle."""
    rng = np.random.default_rng([seed, 17])
    d = field(rng, case["spheres"], case["level"], env=64)
    rays = torch.from_numpy(ray_batch(rng, case["rays"], False).astype(np.float64)).cuda()
    corners = []
    for si, m, _, _ in d.entities:
        s = d.shapes[si]
        m = np.asarray(m, np.float32).astype(np.float64)
        v = s.vertices.astype(np.float64) @ m[:3, :3].T + m[:3, 3]
        corners.append(v[s.faces])
    tri = torch.from_numpy(np.concatenate(corners)).cuda()
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    # with n = e1 x e2: t = n.(a - o) / n.d, and U, V, W as triple products
    n = torch.linalg.cross(e1, e2)
    na = (n * a).sum(1)
    count = rays.shape[0]
    t_out = torch.full((count,), -1.0, dtype=torch.float64, device="cuda")
    b_out = torch.zeros((count, 2), dtype=torch.float64, device="cuda")
    b_out[:, :] = 0.0
    step = max(1, (1 << 25) // tri.shape[0])
    for i in range(0, count, step):
        r = rays[i:i + step]
        o, dr = r[:, None, 0:3], r[:, None, 4:7]
        den = (dr * n).sum(2)
        t = (na - (o * n).sum(2)) / den
        p = o + t[..., None] * dr - a
        c = torch.linalg.cross(p, e2.expand_as(p))
        nn = (n * n).sum(1)
        w1 = (c * n).sum(2) / nn
        w2 = (torch.linalg.cross(e1.expand_as(p), p) * n).sum(2) / nn
        ok = (w1 >= 0) & (w2 >= 0) & (w1 + w2 <= 1) & (t > r[:, None, 3]) & (t < r[:, None, 7])
        best, at = torch.where(ok, t, math.inf).min(1)
        hit = torch.isfinite(best)
        t_out[i:i + step] = torch.where(hit, best, -1.0)
        w1 = w1.gather(1, at[:, None])[:, 0]
        w2 = w2.gather(1, at[:, None])[:, 0]
        b_out[i:i + step, 0] = torch.where(hit, 1.0 - w1 - w2, 0.0)
        b_out[i:i + step, 1] = torch.where(hit, w1, 0.0)
    return {"t": t_out, "inst": None, "prim": None, "bary": b_out}


def exact_network(case, seed):
    """Hash-grid encoding, the 48-64-64-3 ReLU network and the gradients of
    the mean relative L2 loss (its denominator held constant)."""
    rng = np.random.default_rng([seed, 17])
    mlp, table = network_params(rng, case["log2"])
    f, target = network_batch(rng, case["rows"])
    f, target = (torch.from_numpy(x.astype(np.float64)).cuda() for x in (f, target))
    mlp = torch.from_numpy(mlp.astype(np.float64)).cuda().requires_grad_()
    tab = torch.from_numpy(table.astype(np.float64)).cuda().reshape(16, -1, 2).requires_grad_()
    size = 2 ** case["log2"]
    ratio = math.exp((math.log(2048.0) - math.log(16.0)) / 15)
    enc = []
    for level in range(16):
        res = int(math.floor(16.0 * ratio ** level + 0.5))
        x = f[:, :3] * res
        cell = x.floor().clamp(0, res - 1)
        frac = x - cell
        cell = cell.to(torch.int64)
        total = 0.0
        for k in range(8):
            bit = torch.tensor([k & 1, (k >> 1) & 1, (k >> 2) & 1], device="cuda")
            c = cell + bit
            if (res + 1) ** 3 <= size:
                idx = c[:, 0] + (res + 1) * (c[:, 1] + (res + 1) * c[:, 2])
            else:
                idx = (c[:, 0] ^ (c[:, 1] * 2654435761) ^ (c[:, 2] * 805459861)) & (size - 1)
            w = torch.where(bit == 1, frac, 1.0 - frac).prod(1)
            total = total + w[:, None] * tab[level][idx]
        enc.append(total)
    n = f.shape[0]
    x = torch.cat(enc + [f[:, 3:], torch.ones(n, 1, dtype=f.dtype, device="cuda"),
                         torch.zeros(n, 6, dtype=f.dtype, device="cuda")], 1)
    h = torch.relu(x @ mlp[:3072].reshape(48, 64))
    h = torch.relu(h @ mlp[3072:7168].reshape(64, 64))
    y = (h @ mlp[7168:].reshape(64, 32))[:, :3]
    loss = ((y - target) ** 2 / (y.detach() ** 2 + 0.01)).sum() / n
    loss.backward()
    return {"out": y.detach(), "grad_mlp": mlp.grad, "grad_table": tab.grad.reshape(-1), "loss": float(loss)}
