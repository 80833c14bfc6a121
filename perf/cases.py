"""Performance cases of the render path, over the work its users give it.

A case is one call (or one small group of calls) of a public entry point on
scenes of a stated size. `prepare` builds what a program holds before the call
(a context, uploaded meshes and textures, output buffers, the arguments of a
batch, a captured graph, a server); `run` is the call; `exact` is the depth
image of the same frames in 64-bit arithmetic, independent of the library.

Fields of a case:
  call    draw      Context.draw: the synchronous drop-in, pixels in host arrays
          device    Context.draw_device: one asynchronous frame in device memory
          noalloc   Context.draw_device_noalloc
          batch     Context.submit_batch: `frames` frames in one launch
          graph     BatchGraph.launch: the same, replayed from captured graphs
          present   Context.present_draw / present_wait, two frames in flight
          serve     Server.submit / Server.wait: `frames` requests, pixels on the host
  scene   sphere    one displaced sphere of `faces` triangles, camera `eye` from its centre
          inside    the same turned inside out, camera within: near plane, large triangles
          instances `objects` objects in a 20^3 box around the camera, `faces` in all
          mixed     per frame one sphere, from `faces_min` to `faces` triangles, at the
                    four resolutions 320x240 .. 1920x1080
          requests  per frame 1..8 objects drawn from `meshes` resident meshes of
                    `faces` triangles in all, camera on a shell r in [2, 6], at
                    640x360, 1280x720 or 1920x1080
  texture side of the (square) texture, 0 for none; flat, overlays: options.
"""
import math

import numpy as np
import torch

from gorender_amd import _lib, scenes
from gorender_amd.device import BatchGraph, Context
from gorender_amd.scenes import MeshData, SceneData, TextureData
from gorender_amd.serve import PreparedRequest, Server

MIXED_SIZES = [(320, 240), (640, 360), (1280, 720), (1920, 1080)]
REQUEST_SIZES = [(640, 360), (1280, 720), (1920, 1080)]


def _case(name, call, scene, faces, width=0, height=0, frames=1, objects=1, meshes=1,
          faces_min=0, texture=16, eye=1.2, flat=False, overlays=False):
    c = dict(call=call, scene=scene, faces=faces, width=width, height=height, frames=frames,
             eye=eye, objects=objects, meshes=meshes, faces_min=faces_min, texture=texture, flat=flat,
             overlays=overlays)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The drop-in Draw of a small model into the caller's arrays: latency.
        _case("draw_5k_360p", "draw", "sphere", 5_120, 640, 360, texture=0, eye=3.0),
        # A thumbnail of a tiny flat-shaded model, odd sizes: launch cost alone.
        _case("device_300_odd", "device", "sphere", 300, 333, 217, texture=17, eye=2.5,
              flat=True),
        # One interactive frame at a time of the headline scene.
        _case("device_200k_720p", "device", "sphere", 200_000, 1280, 720),
        # A frame inside someone else's captured or allocation-free loop.
        _case("noalloc_40k_720p", "noalloc", "sphere", 40_000, 1280, 720, eye=2.0),
        # A large scene of many objects, half of them flat, one frame per call.
        _case("instances_1m_1080p", "batch", "instances", 1_000_000, 1920, 1080, objects=64,
              meshes=16, texture=64),
        # The camera inside a room: large clipped triangles, full cover.
        _case("inside_20k_1080p", "device", "inside", 20_000, 1919, 1079, texture=100,
              flat=True),
        # The debug view: edges, vertices, tile borders, crosshair.
        _case("overlays_20k_720p", "device", "sphere", 20_000, 1280, 720, eye=2.0,
              overlays=True),
        # Offline rendering of an animation: many frames of one scene per launch.
        _case("batch_32x200k_720p", "batch", "sphere", 200_000, 1280, 720, frames=32),
        # Many uneven frames of different models per launch, replayed.
        _case("graph_64_mixed", "graph", "mixed", 500_000, frames=64, faces_min=1_000),
        # A batch of independent requests over resident dense meshes.
        _case("requests_8x4m", "batch", "requests", 4_000_000, frames=8, meshes=16,
              texture=256),
        # The same through the serving loop, pixels delivered to the host.
        _case("serve_8x2m", "serve", "requests", 2_000_000, frames=8, meshes=8, texture=256),
        # The window loop: two frames in flight, colour delivered to the host.
        _case("present_2x200k_720p", "present", "sphere", 200_000, 1280, 720, frames=2),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def size():
        w = rng.randint(160, 1920)
        return w, max(90, min(1080, int(w * rng.uniform(0.5, 0.8))))

    tex = rng.choice([0, 16, 17, 64, 100, 256])
    kind = rng.choice(["draw", "device", "device", "noalloc", "inside", "overlays", "instances",
                       "batch", "batch", "mixed", "requests", "requests"])
    w, h = size()
    eye = round(rng.uniform(1.15, 4.0), 3)
    flat = rng.random() < 0.3
    if kind == "noalloc":
        return _case("", "noalloc", "sphere", logint(100, 60_000), w, h, texture=tex, eye=eye,
                     flat=flat)
    if kind == "inside":
        return _case("", rng.choice(["device", "draw"]), "inside", logint(500, 60_000), w, h,
                     texture=tex, flat=flat)
    if kind == "overlays":
        return _case("", "device", "sphere", logint(300, 40_000), w, h, texture=tex,
                     eye=max(eye, 1.5), overlays=True)
    if kind == "instances":
        n = rng.randint(8, 64)
        return _case("", "batch", "instances", logint(50_000, 1_000_000), w, h, objects=n,
                     meshes=rng.randint(4, 16), texture=tex)
    if kind == "batch":
        n = rng.randint(2, 32)
        return _case("", rng.choice(["batch", "graph"]), "sphere", logint(1_000, 200_000), w, h,
                     frames=n, texture=tex, eye=eye, flat=flat)
    if kind == "mixed":
        return _case("", rng.choice(["batch", "graph"]), "mixed", logint(50_000, 500_000),
                     frames=rng.randint(4, 48), faces_min=1_000, texture=tex, eye=eye)
    if kind == "requests":
        n = rng.randint(8, 16)
        return _case("", rng.choice(["batch", "batch", "serve"]), "requests",
                     logint(300_000, 250_000 * n), frames=rng.randint(2, 8), meshes=n,
                     texture=tex)
    return _case("", kind, "sphere", logint(300, 500_000), w, h, texture=tex, eye=eye,
                 flat=flat)


# ---------------------------------------------------------------------------
# Scenes of a case (sizes from the case, everything else from the seed)
# ---------------------------------------------------------------------------

def _grid(faces):
    """Rows and columns of a lat-long grid of about `faces` triangles (5:8)."""
    nlat = max(2, int(round(math.sqrt(faces / 3.2))))
    return nlat, max(3, int(round(faces / 2 / nlat)))


def _mesh_faces(case):
    """Faces asked for of each mesh of a case."""
    if case["scene"] == "mixed":
        lo, hi, n = case["faces_min"], case["faces"], case["frames"]
        return [int(lo * (hi / lo) ** (((k * 37) % n) / max(1, n - 1))) for k in range(n)]
    n = case["meshes"]
    if case["scene"] in ("instances", "requests"):  # a 1:16 range of sizes, `faces` in all
        uses = -(-case["objects"] // n) if case["scene"] == "instances" else 1
        share = [16.0 ** (k / max(1, n - 1)) for k in range(n)]
        return [max(12, int(case["faces"] * s / sum(share) / uses)) for s in share]
    return [case["faces"]]


def _frame_size(case, k):
    if case["scene"] == "mixed":
        return MIXED_SIZES[(k * 3 + k // 4) % 4]
    if case["scene"] == "requests":
        return REQUEST_SIZES[k % 3]
    return case["width"], case["height"]


def _frame_objects(case, k):
    """Meshes of the objects of frame k."""
    if case["scene"] == "mixed":
        return [k]
    if case["scene"] == "instances":
        return [j % case["meshes"] for j in range(case["objects"])]
    if case["scene"] == "requests":
        return [(5 * k + 3 * j) % case["meshes"] for j in range(1 + (3 * k + 2) % 8)]
    return [0]


def _rotation(rng):
    q = rng.normal(size=4)
    x, y, z, w = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def _world(rotation, scale=1.0, move=(0.0, 0.0, 0.0)):
    m = np.eye(4)
    m[:3, :3] = rotation * scale
    m[:3, 3] = move
    return m.astype(np.float32)


def _scenes(case, seed):
    rng = np.random.default_rng([seed, 0x6F72656E])
    meshes, textures = [], []
    side = case["texture"]
    for k, f in enumerate(_mesh_faces(case)):
        m = scenes.latlong_sphere(*_grid(f), scenes.SplitMix64(int(rng.integers(1 << 62))))
        if case["scene"] == "inside":
            m.vertex_normals[:, :3] *= -1
            m.vertex_indices = np.ascontiguousarray(m.vertex_indices[:, ::-1])
            m.normal_indices = np.ascontiguousarray(m.normal_indices[:, ::-1])
            m.uvs = np.ascontiguousarray(m.uvs[:, ::-1])
        if case["scene"] == "instances" and k % 2:
            m = MeshData(m.vertices, m.vertex_indices, uvs=m.uvs)  # no normals: flat
        if side and (case["scene"] != "mixed" or k % 2):
            kind = _lib.GR_TEXTURE_IMAGE if side & (side - 1) else _lib.GR_TEXTURE_IMAGE_FAST
            textures.append(TextureData(kind, side, side, rgba=rng.integers(
                0, 256, (side, side, 4), dtype=np.uint8)))
            scenes.with_texture(m, len(textures) - 1)
        meshes.append(m)
    flags = _lib.GR_DEFAULT_FLAGS
    if case["flat"]:
        flags |= _lib.GR_FLAT_SHADING
    if case["overlays"]:
        flags |= (_lib.GR_SHOW_EDGES | _lib.GR_SHOW_VERTICES | _lib.GR_SHOW_TILE_BOUNDS
                  | _lib.GR_SHOW_CROSSHAIR)
    out = []
    turn = _rotation(rng)
    for k in range(case["frames"]):
        w, h = _frame_size(case, k)
        fr = scenes.FrameData(w, h, flags=flags,
                              znear=0.1 if case["scene"] == "inside" else 0.0)
        eye, look, up = (0.0, 0.0, case["eye"]), (0.0, 0.0, -1.0), (0, 1, 0)
        if case["scene"] == "inside":
            eye = tuple(rng.uniform(-0.3, 0.3, 3))
        elif case["scene"] == "instances":
            eye = (0.0, 0.0, 0.0)
        elif case["scene"] == "requests":
            d = rng.normal(size=3)
            d /= np.linalg.norm(d)
            eye, look = tuple(d * rng.uniform(2.0, 6.0)), tuple(-d)
            up = (0, 1, 0) if abs(d[1]) < 0.99 else (1, 0, 0)
        objs = []
        for mi in _frame_objects(case, k):
            if case["scene"] == "instances":
                world = _world(_rotation(rng), rng.uniform(0.5, 3.0), rng.uniform(-10, 10, 3))
            elif case["scene"] == "requests":
                world = _world(_rotation(rng), rng.uniform(0.4, 1.2), rng.uniform(-1.5, 1.5, 3))
            elif case["scene"] == "mixed":
                world = _world(_rotation(rng))
            else:  # an animation: a hundredth of a radian a frame
                c, s = math.cos(0.01 * k), math.sin(0.01 * k)
                world = _world(np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]]) @ turn)
            objs.append(scenes.camera_object(fr, mi, eye, look, up, world=world))
        out.append(SceneData(fr, meshes, textures, objs))
    return out


# ---------------------------------------------------------------------------
# What is measured
# ---------------------------------------------------------------------------

class _State:
    pass


_shared = []


def _one_stream():
    """The stream of the allocation-free draws: they share one fixed array per
    GPU, so a program with several contexts keeps them on one stream."""
    if not _shared:
        _shared.append(torch.cuda.Stream())
    return _shared[0].cuda_stream


def prepare(case, seed):
    st = _State()
    st.call, st.scenes = case["call"], _scenes(case, seed)
    st.ctx = Context(0)
    if st.call == "noalloc":
        st.ctx.set_stream(_one_stream())
    st.handles, _ = st.ctx.upload_scene(st.scenes[0])
    if case["scene"] in ("requests", "instances"):
        # Dense batches list more (triangle, tile) references than the default.
        st.ctx.set_config(refs_capacity=1 << 24)
    n = [s.frame.width * s.frame.height for s in st.scenes]
    if st.call in ("device", "noalloc", "batch", "graph"):
        st.rgba = torch.empty((sum(n), 4), dtype=torch.uint8, device="cuda")
        st.depth = torch.empty(sum(n), dtype=torch.float32, device="cuda")
        at = np.concatenate([[0], np.cumsum(n)[:-1]])
        st.outputs = [(st.rgba.data_ptr() + 4 * int(a), st.depth.data_ptr() + 4 * int(a))
                      for a in at]
    if st.call in ("batch", "graph"):
        st.prepared = st.ctx.prepare_batch(st.scenes, [st.handles] * len(n), st.outputs)
    if st.call == "graph":
        st.graph = BatchGraph(st.ctx, st.prepared)
    if st.call == "serve":
        st.requests = [PreparedRequest(s, st.handles) for s in st.scenes]
        st.server = Server(st.ctx)
    return st


def run(st):
    if st.call == "draw":
        rgba, depth, stats = st.ctx.draw(st.scenes[0], st.handles)
        return {"rgba": rgba, "depth": depth, "stats": stats}
    if st.call == "present":
        for s in st.scenes:
            st.ctx.present_draw(s, st.handles, with_depth=False)
        return {"rgba": [st.ctx.present_wait(s.frame.width, s.frame.height)[0]
                         for s in st.scenes]}
    if st.call == "serve":
        tickets = [st.server.submit(r) for r in st.requests]
        done = [st.server.wait(t) for t in tickets]
        return {"rgba": [r.rgba for r in done], "depth": [r.depth for r in done]}
    if st.call == "device":
        st.ctx.draw_device(st.scenes[0], st.handles, *st.outputs[0])
    elif st.call == "noalloc":
        st.ctx.draw_device_noalloc(st.scenes[0], st.handles, *st.outputs[0])
    elif st.call == "batch":
        st.ctx.submit_batch(st.prepared)
    else:
        st.graph.launch()
    return {"rgba": st.rgba, "depth": st.depth}


def work(case):
    """Bytes: every mesh drawn (positions, normals, texture coordinates,
    indices) and texture once, every pixel's colour and depth once. Operations:
    the transform of every vertex of every object, and per pixel the
    barycentrics, three interpolations and the colour."""
    grids = [_grid(f) for f in _mesh_faces(case)]
    verts = [(a + 1) * (b + 1) for a, b in grids]
    faces = [2 * a * b for a, b in grids]
    drawn = [_frame_objects(case, k) for k in range(case["frames"])]
    pixels = sum(w * h for w, h in (_frame_size(case, k) for k in range(case["frames"])))
    used = {m for d in drawn for m in d}
    side = case["texture"]
    per_vertex = 24 + (8 if side else 0)
    size = sum(verts[m] * per_vertex + faces[m] * 12 + side * side * 4 for m in used)
    out = 4 if case["call"] == "present" else 8
    return {"bytes": size + pixels * out,
            "flops": 28 * sum(verts[m] for d in drawn for m in d) + 60 * pixels}


# ---------------------------------------------------------------------------
# The depth image in 64 bits
# ---------------------------------------------------------------------------

# What the path decides on 32-bit coordinates (facing, inside a plane, the whole
# pixel position of a vertex) is decided so here too, operation by operation;
# every value is carried beside it in 64 bits.

def _dot4(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3]


def _transform(rows, v):
    return torch.stack([_dot4(rows[i], v.unbind(-1)) for i in range(len(rows))], -1)


def _cut(A, B, point, normal):
    u, q = (B - A).unbind(-1), (A - A.new_tensor(point)).unbind(-1)
    f = -_dot4(normal, q) / _dot4(normal, u)
    return A + torch.stack(u, -1) * f[..., None]


def _clip(tri, tri32, planes):
    """Triangles [n, 3, 4] against the planes, in 64 and in 32 bits: the fans."""
    n, dev = len(tri), tri.device
    slot = torch.arange(12, device=dev)
    count = torch.full((n,), 3, device=dev)
    P = tri.new_zeros((n, 12, 4))
    Q = tri32.new_zeros((n, 12, 4))
    P[:, :3], Q[:, :3] = tri, tri32
    for point, normal in planes:
        inside = _dot4((Q - Q.new_tensor(point)).unbind(-1), normal) <= 0
        nxt = torch.where(slot + 1 < count[:, None], slot + 1, 0)
        live = slot < count[:, None]
        ib, ia = inside & live, torch.gather(inside, 1, nxt) & live
        adds = (ia != ib).long() + ia.long()
        at = adds.cumsum(1) - adds
        nxt = nxt[:, :, None].expand(-1, -1, 4)
        new = []
        for R in (P, Q):
            A = torch.gather(R, 1, nxt)
            out = R.new_zeros((n, 14, 4))
            for mask, where, val in ((ia != ib, at, _cut(A, R, point, normal)),
                                     (ia, at + (ia & ~ib).long(), A)):
                r, k = torch.nonzero(mask, as_tuple=True)
                out[r, where[r, k]] = val[r, k]
            new.append(out[:, :12])
        (P, Q), count = new, adds.sum(1)
    return [torch.cat([R[count >= k + 2][:, [0, k, k + 1]] for k in range(1, 9)])
            for R in (P, Q)]


def _exact_depth(scene, dev):
    fr = scene.frame
    W, H = fr.width, fr.height
    screen = np.asarray(fr.screen, np.float64).tolist()
    depth = torch.full((W * H,), -1.0, dtype=torch.float64, device=dev)
    # (point, normal) in draw order; inside where (q - point) . normal <= 0
    planes = [((-1, 0, 0, 1), (1, 0, 0, 1)), ((1, 0, 0, 1), (-1, 0, 0, 1)),
              ((0, -1, 0, 1), (0, 1, 0, 1)), ((0, 1, 0, 1), (0, -1, 0, 1)),
              ((0, 0, float(np.float32(fr.znear)), 1), (0, 0, -1, 0)),
              ((0, 0, float(np.float32(fr.zfar)), 1), (0, 0, 1, 0))]
    for o in scene.objects:
        m = scene.meshes[o.mesh]
        faces = torch.tensor(m.vertex_indices.astype(np.int64), device=dev)
        v32 = torch.tensor(m.vertices, device=dev)
        mvp = o.mvp.astype(np.float64).tolist()
        t32 = _transform(mvp, v32)[faces]
        t = _transform(mvp, v32.double())[faces]
        if fr.flags & _lib.GR_BACKFACE_CULLING:
            (ax, ay, az), (bx, by, bz) = ((t32[:, k, :3] - t32[:, 0, :3]).unbind(-1)
                                          for k in (1, 2))
            x, y, z = t32[:, 0, :3].unbind(-1)
            front = ((ay * bz - az * by) * -x + (az * bx - ax * bz) * -y
                     + (ax * by - ay * bx) * -z) > 0
            t, t32 = t[front], t32[front]
        ins = torch.stack([_dot4((t32 - t32.new_tensor(p)).unbind(-1), n) <= 0
                           for p, n in planes])
        whole = ins.all(2).all(0)
        maybe = ~whole & ins.any(2).all(0)
        cut, cut32 = _clip(t[maybe], t32[maybe], planes)
        w = torch.cat([t[whole], cut])[..., 3]
        t32 = torch.cat([t32[whole], cut32])
        s = t32 / t32[..., 3:]
        X, Y = _transform(screen[:2], s).trunc().long().unbind(-1)
        x0, x1 = X.amin(1).clamp(min=0), X.amax(1).clamp(max=W - 1)
        y0, y1 = Y.amin(1).clamp(min=0), Y.amax(1).clamp(max=H - 1)
        area = (x1 - x0 + 1).clamp(min=0) * (y1 - y0 + 1).clamp(min=0)
        ends = area.cumsum(0)
        start = 0
        while start < len(area):  # a few million (triangle, pixel) pairs at a time
            base = int(ends[start - 1]) if start else 0
            stop = max(start + 1, int(torch.searchsorted(ends, base + (1 << 22), right=True)))
            tri = torch.repeat_interleave(torch.arange(start, min(stop, len(area)), device=dev),
                                          area[start:stop])
            k = torch.arange(len(tri), device=dev) - (ends[tri] - area[tri] - base)
            bw = x1[tri] - x0[tri] + 1
            px, py = x0[tri] + k % bw, y0[tri] + k // bw
            e = []
            for a, b in ((0, 1), (1, 2), (2, 0)):
                dx, dy = Y[:, a] - Y[:, b], X[:, b] - X[:, a]
                c = X[:, a] * Y[:, b] - X[:, b] * Y[:, a]
                c = c - (~((dy > 0) | ((dy == 0) & (dx > 0)))).long()
                e.append(dx[tri] * px + dy[tri] * py + c[tri])
            hit = (e[0] < 0) & (e[1] < 0) & (e[2] < 0)
            tri, px, py = tri[hit], px[hit], py[hit]
            e01, e12, e20 = (f[hit].double() for f in e)
            al, be = e12 / (e01 + e12 + e20), e20 / (e01 + e12 + e20)
            zr = -(al / w[tri, 0] + be / w[tri, 1] + (1 - al - be) / w[tri, 2])
            depth.scatter_reduce_(0, py * W + px, zr, "amax")
            start = stop
    return depth


def exact(case, seed):
    if case["call"] == "present":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    done = [_exact_depth(s, dev) for s in _scenes(case, seed)]
    if case["call"] == "draw":
        return {"rgba": None, "depth": done[0].reshape(case["height"], case["width"]),
                "stats": None}
    if case["call"] == "serve":
        return {"rgba": None, "depth": [d.reshape(_frame_size(case, k)[::-1])
                                        for k, d in enumerate(done)]}
    return {"rgba": None, "depth": torch.cat(done)}
