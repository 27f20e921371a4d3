"""What a program that renders with this framework has it do, as cases that
can be measured: tile and frame traces with every estimator, a batch of
scenes, closest-hit queries, the irradiance cube map and the post step, from
one 64x64 tile to a 1920x1080 frame of a 4M-triangle room.

A case is a dict of plain values.  ``prepare`` builds what the program has in
hand (scene, camera, guide, device images), ``run`` makes one pass through the
public entry points and returns its whole outputs.  Images are progressive:
pass k of a state traces the samples after pass k - 1's, as a viewer does.

Every output is defined bit for bit (FP32 in a stated order, integer random
streams, fixed-order training sums), so the tolerance is "exact".
"""
import functools
import math

import numpy as np
import torch

import vk_cinematic_amd as V
from vk_cinematic_amd import scenes

EST = {"parity": V.EST_PARITY, "unbiased": V.EST_UNBIASED, "nee": V.EST_NEE,
       "guided": V.EST_GUIDED, "guided_nee": V.EST_GUIDED_NEE}
RNG = {"pcg": V.RNG_PCG, "xorshift": V.RNG_XORSHIFT_PIXEL}
TX = {"double": V.TX_DOUBLE, "fast": V.TX_FAST}


def _trace(name, scene, size, width, height, spp, bounces, estimator, **more):
    c = {"name": name, "kind": "trace", "scene": scene, "size": size, "width": width,
         "height": height, "spp": spp, "bounces": bounces, "estimator": estimator,
         "rng": "pcg", "tx": "double", "train": False, "frozen_passes": 0, "host": False,
         "tile": 64}
    c.update(more)
    return c


def listed():
    return [
        # one work item of the reference's tile loop: a worker thread's call
        # for one 64x64 tile of the small scene into the host image
        _trace("tile_64_host", "config1", 3, 256, 256, 1, 3, "parity", host=True, tile=64,
               rng="xorshift"),
        # the reference app's frame at its own settings (parity estimator),
        # device-resident image
        _trace("frame_256_parity", "config1", 3, 256, 256, 4, 3, "parity"),
        # an interactive preview in an odd-sized window: equirectangular sky,
        # one sample, device transcendentals
        _trace("preview_odd", "config1_equirect", 3, 333, 187, 1, 4, "unbiased", tx="fast",
               tile=50),
        # a still of the 1M-triangle room lit through its opening
        _trace("box_512_plain", "box", 7, 512, 512, 2, 6, "unbiased"),
        # the headline frame: 4M triangles, 1080p, one sample per pass
        _trace("room_1080p_plain", "room", 14, 1920, 1080, 1, 6, "unbiased"),
        # next-event estimation with emitters and sky in a mid-sized room
        _trace("lamps_nee", "room", 7, 640, 360, 2, 6, "nee"),
        # online training of the guide: one pass renders and takes the Adam steps
        _trace("guided_train", "box", 7, 512, 512, 1, 6, "guided", tx="fast", train=True),
        # rendering with a learned guide and light samples
        _trace("guided_nee_frozen", "room", 7, 960, 540, 1, 6, "guided_nee", tx="fast",
               frozen_passes=6),
        # a dataset tool's batch of scenes of uneven sizes, one graph replay
        {"name": "batch_8_scenes", "kind": "batch", "count": 8, "min_side": 64,
         "max_side": 512, "min_tris": 1e4, "max_tris": 3e5, "spp": 4, "bounces": 5},
        # incoherent closest-hit queries on device-resident rays (baking, collision)
        {"name": "closest_soup", "kind": "closest", "tris": 500_000, "rays": 1 << 21},
        # the irradiance cube map of an HDR sky at load time (host in, host out)
        {"name": "irradiance_32", "kind": "irradiance", "env_width": 1024, "env_height": 512,
         "face": 32, "tx": "double"},
        # a viewer's post step per 1080p frame: accumulate, then tone map
        {"name": "post_1080p", "kind": "post", "width": 1920, "height": 1080, "tx": "double"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace"] * 8 + ["closest"] * 2 + ["batch", "irradiance", "post"])
    if kind == "closest":
        return {"kind": "closest", "tris": _logint(rng, 500, 500_000),
                "rays": _logint(rng, 1000, 1 << 21)}
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(2, 8), "min_side": rng.randint(33, 96),
                "max_side": rng.randint(97, 512), "min_tris": 1e4, "max_tris": 3e5,
                "spp": rng.randint(1, 4), "bounces": rng.randint(2, 6)}
    if kind == "irradiance":
        w = _logint(rng, 64, 1024)
        return {"kind": "irradiance", "env_width": w, "env_height": max(2, w // 2),
                "face": rng.randint(5, 32), "tx": rng.choice(["double", "fast"])}
    if kind == "post":
        return {"kind": "post", "width": _logint(rng, 64, 1920),
                "height": _logint(rng, 64, 1080), "tx": rng.choice(["double", "fast"])}
    est = rng.choice(["parity", "unbiased", "unbiased", "nee", "guided", "guided_nee"])
    guided = est.startswith("guided")
    train = guided and rng.random() < 0.5
    scene = rng.choice(["config1", "config1_equirect", "grid", "box", "room"])
    if guided and scene.startswith("config1"):
        scene = "room"
    size = {"box": rng.randint(3, 7), "room": rng.randint(3, 8),
            "grid": _logint(rng, 5000, 200_000)}.get(scene, 3)
    c = _trace("", scene, size, _logint(rng, 48, 1280), _logint(rng, 48, 720),
               rng.randint(1, 3), rng.randint(2, 6), est,
               rng=rng.choice(["pcg", "pcg", "xorshift"]),
               tx=rng.choice(["double", "fast"]), train=train,
               frozen_passes=0 if train or not guided else 4,
               host=rng.random() < 0.25, tile=rng.choice([16, 50, 64, 128]))
    # no more rays than a third of the largest frame's (light samples, training
    # and one launch sequence per sample of the serial streams cost more each)
    while c["width"] * c["height"] * c["spp"] * c["bounces"] > 4_000_000:
        c["width"], c["height"] = c["width"] * 4 // 5, c["height"] * 4 // 5
    del c["name"]
    return c


# ------------------------------------------------------------- preparation
@functools.lru_cache(maxsize=1)
def _device():
    return V.Device(0)


class _Buffer:
    """A torch tensor on the GPU as the device image the bindings take."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


@functools.lru_cache(maxsize=8)
def _base_scene(scene, size):
    """Meshes, objects and materials without the seed's changes."""
    if scene == "config1":
        return scenes.config1(64, 64, env="cube")
    if scene == "config1_equirect":
        return scenes.config1(64, 64, env="equirect")
    if scene == "grid":
        return scenes.grid_scene(11, size, 64)
    if scene == "box":   # lit through the opening only
        return scenes.box_scene(size, 5, 64, 64, seed=4, light_fraction=0.0)
    return scenes.box_scene(size, 5, 64, 64, seed=5)   # emitters among the objects


def _scene_desc(c, seed):
    """The scene with the seed's inputs: which mesh and material each object
    takes, their sizes, and where the camera stands."""
    base = _base_scene(c["scene"], c["size"])
    r = np.random.default_rng([seed, 17])
    d = dict(base)
    objs = list(base["objects"])
    first = [i for i, o in enumerate(objs) if o[1] >= 1000 and i > 0]
    if first:
        meshes = [objs[i][0] for i in first]
        mats = [objs[i][1] for i in first]
        r.shuffle(meshes)
        r.shuffle(mats)
        for i, m, mat in zip(first, meshes, mats):
            _, _, pos, q, s = objs[i]
            k = float(r.uniform(0.85, 1.0))
            objs[i] = (m, mat, pos, q, (s[0] * k, s[1] * k, s[2] * k))
    else:
        mesh, mat, pos, q, s = objs[0]
        objs[0] = (mesh, mat, tuple(float(p + v) for p, v in zip(pos, r.uniform(-0.2, 0.2, 3))),
                   q, s)
    d["objects"] = objs
    _, _, pos, q, fd = base["camera"]
    jitter = r.uniform(-0.15, 0.15, 3)
    d["camera"] = (c["width"], c["height"],
                   tuple(float(p + j) for p, j in zip(pos, jitter)), q, fd)
    return d


def _prepare_trace(c, seed):
    dev = _device()
    scene, cam = scenes.load_gpu(dev, _scene_desc(c, seed))
    w, h = c["width"], c["height"]
    guide = None
    tiles = V.ComputeTiles(w, h, c["tile"], c["tile"])
    s = {"case": c, "scene": scene, "cam": cam, "pass": 0, "seed": seed & 0xFFFFFF}
    if c["host"]:
        s["pixels"] = np.zeros(w * h * 4, np.float32)
    else:
        s["image"] = _Buffer(torch.zeros((h, w, 4), dtype=torch.float32, device="cuda"))
    if c["estimator"].startswith("guided"):
        guide = V.Guide(dev, seed=1 + (seed & 0xFF), max_weight=10.0)
        scratch = s.get("image") or _Buffer(torch.zeros((h, w, 4), dtype=torch.float32,
                                                        device="cuda"))
        torch.cuda.synchronize()
        for k in range(c["frozen_passes"]):   # a program renders with a guide it trained
            ctx = _context(c, cam, scene, s["seed"] ^ 0x5A5A, 1, k, guide, True)
            V.path_trace_tiles_device(ctx, tiles, scratch)
    s["guide"], s["tiles"] = guide, tiles
    return s


def _context(c, cam, scene, seed, spp, offset, guide, train):
    return V.make_context(cam, scene, spp=spp, bounces=c["bounces"],
                          clamp=10.0 if c["estimator"] == "parity" else 0.0,
                          estimator=EST[c["estimator"]], rng=RNG[c["rng"]], seed=seed,
                          transcendentals=TX[c["tx"]], sample_offset=offset, guide=guide,
                          train=train)


def _prepare_batch(c, seed):
    dev = _device()
    r = np.random.default_rng([seed, 23])
    shapes = np.random.default_rng([c["count"], c["min_side"], c["max_side"]])
    items, images = [], []
    for k in range(c["count"]):
        tris = float(np.exp(shapes.uniform(np.log(c["min_tris"]), np.log(c["max_tris"]))))
        side = int(shapes.integers(c["min_side"], c["max_side"] + 1))
        desc = scenes.grid_scene(int(r.integers(1, 1 << 20)), tris, side)
        scene, cam = scenes.load_gpu(dev, desc)
        img = _Buffer(torch.zeros((side, side, 4), dtype=torch.float32, device="cuda"))
        items.append((cam, scene, img))
        images.append(img.tensor)
    torch.cuda.synchronize()
    batch = V.Batch(dev, items, spp=c["spp"], bounces=c["bounces"], seed=seed & 0xFFFFFF)
    return {"case": c, "batch": batch, "images": images}


def _rays(n, seed):
    r = np.random.default_rng([seed, 29])
    o = r.uniform(-2.0, 2.0, size=(n, 3)).astype(np.float32)
    z = r.uniform(-1.0, 1.0, size=n)
    ph = r.uniform(0.0, 2.0 * np.pi, size=n)
    q = np.sqrt(np.maximum(0.0, 1.0 - z * z))
    d = np.stack([q * np.cos(ph), q * np.sin(ph), z], axis=1).astype(np.float32)
    return o, d


def _soup(c, seed):
    # larger triangles in smaller soups: about the same cover of the cube
    mu = -5.0 + 0.5 * math.log(1e6 / c["tris"])
    return V.gen_triangle_soup(c["tris"], seed=1 + (seed & 0xFFFFFF), mu=mu, sigma=0.5)


def _prepare_closest(c, seed):
    scene = V.Scene(_device())
    verts, idx = scenes.soup_mesh(_soup(c, seed))
    mesh = scene.create_mesh(verts, idx, False)
    scene.add_object(mesh, 0, (0.0, 0.0, 0.0))
    scene.build()
    o, d = _rays(c["rays"], seed)
    cols = [torch.from_numpy(np.ascontiguousarray(a[:, k])).cuda() for a in (o, d)
            for k in range(3)]
    n = c["rays"]
    return {"case": c, "scene": scene, "mesh": mesh, "cols": cols,
            "prim": torch.zeros(n, dtype=torch.int32, device="cuda"),
            "tuv": torch.zeros((3, n), dtype=torch.float32, device="cuda")}


def _hdr_sky(c, seed):
    r = np.random.default_rng([seed, 31])
    z = r.uniform(0.2, 0.9)
    ph = r.uniform(0.0, 2.0 * np.pi)
    q = math.sqrt(1.0 - z * z)
    sky = V.gen_sky_equirect(c["env_width"], c["env_height"],
                             sun=(q * math.cos(ph), z, q * math.sin(ph)))
    img = sky.reshape(c["env_height"], c["env_width"], 4)
    return np.ascontiguousarray(img * r.uniform(0.5, 2.0, size=(1, 1, 4)).astype(np.float32))


def _post_images(c, seed):
    """A running mean and a new frame: mostly dim HDR values, some far above
    white (noise of a path tracer)."""
    g = torch.Generator().manual_seed(seed)
    n = c["width"] * c["height"]
    imgs = []
    for scale in (0.8, 1.5):
        x = torch.randn((n, 4), generator=g) * scale - 1.5
        imgs.append(torch.exp(x).float())
    return imgs


def _prepare_post(c, seed):
    mean, frame = (x.cuda() for x in _post_images(c, seed))
    out = torch.zeros((mean.shape[0], 4), dtype=torch.uint8, device="cuda")
    return {"case": c, "dev": _device(), "start": mean, "mean": _Buffer(mean.clone()),
            "frame": _Buffer(frame), "out": out}


def prepare(case, seed):
    return {"trace": _prepare_trace, "batch": _prepare_batch, "closest": _prepare_closest,
            "irradiance": lambda c, s: {"case": c, "dev": _device(), "sky": _hdr_sky(c, s)},
            "post": _prepare_post}[case["kind"]](case, seed)


# --------------------------------------------------------------------- run
def run(s):
    c = s["case"]
    if c["kind"] == "trace":
        ctx = _context(c, s["cam"], s["scene"], s["seed"], c["spp"],
                       s["pass"] * c["spp"], s["guide"], c["train"])
        s["pass"] += 1
        if c["host"]:
            # the tile loop's call for a single tile; else the whole queue
            if c["tile"] == 64:
                V.sp_PathTraceTile(ctx, s["tiles"][len(s["tiles"]) // 2], s["pixels"])
            else:
                V.path_trace_tiles(ctx, s["tiles"], s["pixels"])
            out = [s["pixels"]]
        else:
            V.path_trace_tiles_device(ctx, s["tiles"], s["image"])
            out = [s["image"].tensor]
        if c["train"]:
            out.append(s["guide"].params())   # the updated weights
        return out
    if c["kind"] == "batch":
        s["batch"].run()
        return list(s["images"])
    if c["kind"] == "closest":
        n = c["rays"]
        t, u, v = (s["tuv"][k].data_ptr() for k in range(3))
        V.check(V.lib().spg_intersect_closest_device(
            s["scene"].handle, s["mesh"], *[x.data_ptr() for x in s["cols"]], n,
            s["prim"].data_ptr(), t, u, v, None))
        return {"prim": s["prim"], "tuv": s["tuv"]}
    if c["kind"] == "irradiance":
        faces, _ = s["dev"].create_irradiance_cubemap(s["sky"], c["face"], c["face"],
                                                      transcendentals=TX[c["tx"]])
        return faces
    n = c["width"] * c["height"]
    s["dev"].accumulate(s["mean"], s["frame"], n, 3, 1)
    V.check(V.lib().spg_tonemap_device(s["dev"].handle, s["mean"].ptr, n, 1.0, TX[c["tx"]],
                                       s["out"].data_ptr()))
    return {"mean": s["mean"].tensor, "rgba8": s["out"]}


# -------------------------------------------------------------------- work
def _triangles(c):
    if c["scene"].startswith("config1"):
        return 1282
    return c["size"] if c["scene"] == "grid" else c["size"] * c["size"] * 20480


def work(case):
    """Bytes: the outputs written and the inputs a pass has to read (of a
    scene: a 64-byte shading record and a triangle's vertices per surface hit,
    no more than the scene holds).  Operations: per ray the boxes and
    triangles of a walk down a balanced four-wide tree, per hit the shading,
    per guided hit the network."""
    c = case
    if c["kind"] == "trace" or c["kind"] == "batch":
        if c["kind"] == "trace":
            w, h = (min(64, c["width"]), min(64, c["height"])) \
                if c["host"] and c["tile"] == 64 else (c["width"], c["height"])
            pixels, tris = w * h, _triangles(c)
            closed = c["scene"] in ("box", "room")
            est = c["estimator"]
        else:
            side = (c["min_side"] + c["max_side"]) / 2
            pixels, tris = c["count"] * side * side, 60_000 * c["count"]
            closed, est = False, "unbiased"
        paths = pixels * c["spp"]
        rays = paths * (0.9 * c["bounces"] if closed else min(c["bounces"], 2.0))
        hits = rays * (0.95 if closed else 0.6)
        if "nee" in est:
            rays += 0.6 * hits
        depth = max(1.0, math.log(tris / 4.0, 4.0))
        flops = rays * (depth * 4 * 18 + 4 * 45) + hits * 300
        if est.startswith("guided"):
            flops += hits * 38_912
            if c["train"]:
                flops += 4 * 16384 * 3 * 38_912
        return {"bytes": 16 * pixels + min(hits * 100, tris * 100), "flops": flops}
    if c["kind"] == "closest":
        n, t = c["rays"], c["tris"]
        depth = max(1.0, math.log(max(t, 8) / 4.0, 4.0))
        return {"bytes": 40 * n + min(36 * t, 144 * n), "flops": n * (depth * 4 * 18 + 4 * 45)}
    if c["kind"] == "irradiance":
        texels = 6 * c["face"] ** 2
        return {"bytes": 16 * c["env_width"] * c["env_height"] + 16 * texels,
                "flops": texels * 1008 * 120}
    n = c["width"] * c["height"]
    return {"bytes": n * (32 + 16 + 4), "flops": n * 60}


def tolerance(case):
    return "exact"


# ------------------------------------------------------- 64-bit references
def _exact_closest(c, seed):
    """Brute force over all triangles in float64 (front faces only)."""
    if c["rays"] * c["tris"] > 1 << 34:
        return None
    tri = torch.from_numpy(np.asarray(_soup(c, seed), np.float32)).double().cuda()
    tri = tri.reshape(-1, 3, 3)
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    o, d = (torch.from_numpy(x).double().cuda() for x in _rays(c["rays"], seed))
    n = c["rays"]
    out = torch.zeros((3, n), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 23) // c["tris"])
    for i in range(0, n, step):
        oi, di = o[i:i + step, None], d[i:i + step, None]
        T = oi - a[None]
        p = torch.linalg.cross(di.expand_as(T), e2[None].expand_as(T))
        q = torch.linalg.cross(T, e1[None].expand_as(T))
        det = 1.0 / (p * e1).sum(-1)
        t, u = det * (q * e2).sum(-1), det * (p * T).sum(-1)
        v = det * (q * di).sum(-1)
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & ((di * nrm).sum(-1) < 0) & (t > 0)
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, k = t.min(dim=1)
        hit = torch.isfinite(best)
        k = k[:, None]
        out[0, i:i + step] = torch.where(hit, best, torch.full_like(best, -1.0))
        out[1, i:i + step] = torch.where(hit, u.gather(1, k)[:, 0], torch.zeros_like(best))
        out[2, i:i + step] = torch.where(hit, v.gather(1, k)[:, 0], torch.zeros_like(best))
    return {"prim": None, "tuv": out}


def _exact_irradiance(c, seed):
    img = _hdr_sky(c, seed).astype(np.float64)
    h, w = img.shape[:2]
    one, grid = np.float32(0.1), []
    for end in (np.float32(2.0) * np.float32(math.pi), np.float32(0.5) * np.float32(math.pi)):
        x, vals = np.float32(0.0), []
        while x < end:
            vals.append(x)
            x = np.float32(x + one)
        grid.append(np.array(vals, np.float64))
    phi, theta = (g.ravel() for g in np.meshgrid(grid[0], grid[1], indexing="ij"))
    ld = np.stack([np.sin(theta) * np.cos(phi), np.cos(theta), np.sin(theta) * np.sin(phi)])
    basis = [((1, 0, 0), (0, 1, 0), (0, 0, -1)), ((-1, 0, 0), (0, 1, 0), (0, 0, 1)),
             ((0, 1, 0), (0, 0, -1), (1, 0, 0)), ((0, -1, 0), (0, 0, 1), (1, 0, 0)),
             ((0, 0, 1), (0, 1, 0), (1, 0, 0)), ((0, 0, -1), (0, 1, 0), (-1, 0, 0))]
    f = c["face"]
    out = np.ones((6, f, f, 4))

    def unit(v):
        return v / np.linalg.norm(v, axis=-1, keepdims=True)

    for face, (fwd, up, right) in enumerate(np.array(b, np.float64) for b in basis):
        for y in range(f):
            fx = np.arange(f) / f * 2.0 - 1.0
            fy = (1.0 - y / f) * 2.0 - 1.0
            n = unit(fwd + right * fx[:, None] + up * fy)
            t = unit(np.cross(up, n))
            b = unit(np.cross(n, t))
            wd = n[:, None] * ld[1][None, :, None] + t[:, None] * ld[0][None, :, None] \
                + b[:, None] * ld[2][None, :, None]
            inc = np.arctan2(np.hypot(wd[..., 0], wd[..., 2]), wd[..., 1])
            az = np.arctan2(wd[..., 2], wd[..., 0])
            az = np.where(az < 0, az + 2 * math.pi, az)
            px = np.maximum(az / (2 * math.pi) * w - 0.5, 0.0)
            py = np.maximum((1.0 - (np.cos(inc) * 0.5 + 0.5)) * h - 0.5, 0.0)
            x0, y0 = np.minimum(np.floor(px), w - 1), np.minimum(np.floor(py), h - 1)
            gx, gy = (px - x0)[..., None], (py - y0)[..., None]
            x0, y0 = x0.astype(int), y0.astype(int)
            x1, y1 = np.minimum(x0 + 1, w - 1), np.minimum(y0 + 1, h - 1)
            top = img[y0, x0, :3] * (1 - gx) + img[y0, x1, :3] * gx
            bot = img[y1, x0, :3] * (1 - gx) + img[y1, x1, :3] * gx
            L = np.clip(top * (1 - gy) + bot * gy, 0.0, 10.0)
            k = (np.cos(theta) * np.sin(theta))[None, :, None]
            out[face, y, :, :3] = math.pi * (L * k).sum(axis=1) / len(phi)
    return out


def exact(case, seed):
    """In 64 bits what has such a value.  A traced image has none: its paths
    fork wherever a ray grazes an edge, so a 64-bit render of the same random
    numbers is another sample of the same integral (the tests hold the images
    to the CPU restatement bit for bit instead)."""
    if case["kind"] == "closest":
        return _exact_closest(case, seed)
    if case["kind"] == "irradiance":
        return _exact_irradiance(case, seed)
    if case["kind"] == "post":
        mean, frame = (x.double() for x in _post_images(case, seed))
        m = (mean * 3.0 + frame) / 4.0
        m[:, 3] = 1.0
        return {"mean": m, "rgba8": None}
    return None
