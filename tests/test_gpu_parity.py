"""GPU parity: the HIP render path against the CPU oracle, through the C ABI.

Bar: colour and depth buffers bit-identical to the oracle (which restates the
reference's sequential draw, renderer.go:466-474), and identical counters
(TPF renderer.go:436-441, binned triangles, covered fragments, front faces).
"""
import numpy as np
import pytest

from gorender_amd import _lib
from gorender_amd import scenes as S
from oracle import refcpu

from parity import assert_same
from scene_cases import all_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,builder", all_cases(), ids=[c[0] for c in all_cases()])
def test_case(ctx, name, builder):
    scene = builder()
    want = refcpu.draw(scene)
    got = ctx.draw(scene)
    assert_same(scene, got, want)


@pytest.mark.parametrize("tw,th", [(8, 8), (16, 16), (32, 16), (64, 64), (8, 64), (64, 8)])
def test_tile_shapes(ctx, tw, th):
    """The image does not depend on the raster tile shape."""
    import scene_cases as C
    scene = C.sphere(w=150, h=110, eye=(0, 0, 1.25), nlat=30, nlon=50)
    want = refcpu.draw(scene)
    old = ctx.config()
    try:
        ctx.set_config(tile_w=tw, tile_h=th)
        got = ctx.draw(scene)
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h)
    assert_same(scene, got, want)


def test_config1_both_variants(ctx):
    for variant in ("ref", "cfg"):
        scene = S.config1(variant)
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


def test_config2_full(ctx):
    """Headline frame: 200,000 triangles, 1280x720, textured, side-plane clipping."""
    scene = S.config2()
    assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


def test_refs_capacity_retry(ctx):
    """A tiny tile-list capacity is grown and the frame redrawn (same output)."""
    import scene_cases as C
    scene = C.sphere(w=200, h=120, eye=(0, 0, 1.3), nlat=20, nlon=30)
    want = refcpu.draw(scene)
    old = ctx.config()
    try:
        ctx.set_config(refs_capacity=1024)
        got = ctx.draw(scene)
    finally:
        ctx.set_config(refs_capacity=old.refs_capacity)
    assert_same(scene, got, want)


def test_repeat_is_deterministic(ctx):
    scene = S.config1()
    mh, _ = ctx.upload_scene(scene)
    a = ctx.draw(scene, mh)
    b = ctx.draw(scene, mh)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1].view(np.uint32),
                                                         b[1].view(np.uint32))


def test_ref_tiles_one(ctx):
    """TPF on the sequential renderer's single tile equals the binned count."""
    scene = S.config1()
    scene.frame.ref_tiles = 1
    got = ctx.draw(scene)
    want = refcpu.draw(scene)
    assert_same(scene, got, want)
    assert got[2]["tpf"] == got[2]["triangles"]


def test_batch_equals_single(ctx):
    """gr_draw_batch of several uneven frames == each frame drawn alone."""
    import scene_cases as C
    frames = [C.sphere(seed=11, w=64, h=48), C.overlapping_objects(w=100, h=70),
              C.cube_scene(w=33, h=65), C.clip_space_soup(n=200, seed=9)]
    handles = [ctx.upload_scene(s)[0] for s in frames]
    outs = []
    for s in frames:
        rg, dp = ctx.frame_buffers(s.frame.width, s.frame.height)
        rg.fill(0xA5)  # every pixel must be written by the draw
        dp.fill(0x5A)
        outs.append((rg, dp))
    ctx.draw_batch(frames, handles, [(o[0].ptr, o[1].ptr) for o in outs])
    ctx.synchronize()
    stats = ctx.last_stats()
    for k, s in enumerate(frames):
        want = refcpu.draw(s)
        h, w = s.frame.height, s.frame.width
        got = (outs[k][0].to_numpy(np.uint8, (h, w, 4)),
               outs[k][1].to_numpy(np.float32, (h, w)), stats[k])
        assert_same(s, got, want)


def test_errors(ctx):
    """Reference panics become status codes (renderer.go:318-330; mesh.go:29)."""
    bad = S.MeshData(np.zeros((3, 4), np.float32), np.array([[0, 1, 3]], np.int32))
    with pytest.raises(_lib.GorenderError) as e:
        ctx.upload_mesh(bad)
    assert e.value.status == _lib.GR_ERR_INDEX_OUT_OF_RANGE
    empty = S.MeshData(np.zeros((0, 4), np.float32), np.zeros((0, 3), np.int32))
    with pytest.raises(_lib.GorenderError):
        ctx.upload_mesh(empty)
    # Gouraud shading with a normal index out of range (obj.go:77-89 v//vn faces)
    v = np.array([[0, 0, 0, 1], [1, 0, 0, 1], [0, 1, 0, 1]], np.float32)
    m = S.MeshData(v, np.array([[0, 1, 2]], np.int32), v.copy(),
                   np.array([[0, 1, -1]], np.int32))
    h = ctx.upload_mesh(m)
    fr = S.FrameData(32, 32)
    scene = S.SceneData(fr, [m], [], [S.camera_object(fr, 0, (0, 0, 3), (0, 0, -1))])
    with pytest.raises(_lib.GorenderError) as e:
        ctx.draw(scene, [h])
    assert e.value.status == _lib.GR_ERR_INDEX_OUT_OF_RANGE
    # ... but flat shading never reads the normal indices, as in the reference
    scene.frame.flags |= _lib.GR_FLAT_SHADING
    ctx.draw(scene, [h])
    # Overlay lines of unclipped geometry far off screen would walk billions of
    # pixels in the reference; the GPU path reports them as unsupported and the
    # context stays usable.
    import scene_cases as C
    wide = C.clip_space_soup(flags=C.no(_lib.GR_FRUSTUM_CLIPPING) | _lib.GR_SHOW_EDGES, seed=7,
                             w_range=(-1e-4, 1e-4))
    with pytest.raises(_lib.GorenderError) as e:
        ctx.draw(wide)
    assert e.value.status == _lib.GR_ERR_UNSUPPORTED
    ctx.draw(scene, [h])
    with pytest.raises(_lib.GorenderError) as e:
        ctx.draw(scene, [h + 1000])
    assert e.value.status == _lib.GR_ERR_INVALID_HANDLE


@pytest.mark.parametrize("flags,ref_tiles,size", [
    (_lib.GR_SHOW_CROSSHAIR, 16, (160, 96)),
    (_lib.GR_SHOW_TILE_BOUNDS, 16, (77, 53)),
    (_lib.GR_SHOW_TILE_BOUNDS | _lib.GR_SHOW_CROSSHAIR, 1, (64, 48)),
    (_lib.GR_SHOW_TILE_BOUNDS | _lib.GR_SHOW_CROSSHAIR | _lib.GR_SHOW_EDGES, 16, (120, 90)),
    (_lib.GR_SHOW_TILE_BOUNDS | _lib.GR_SHOW_CROSSHAIR, 16, (5, 7)),
])
def test_decorations(ctx, flags, ref_tiles, size):
    """Tile borders and crosshair (renderer.go:422-434,476-480;
    rasterizer.go:209-217) over the drawn frame, as the oracle draws them."""
    import scene_cases as C
    scene = C.sphere(w=size[0], h=size[1], eye=(0, 0, 2.4), flags=C.ALL | flags)
    scene.frame.ref_tiles = ref_tiles
    assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


@pytest.mark.parametrize("ref_tiles,size", [
    (16, (513, 259)), (16, (256, 65)), (1, (320, 129)), (16, (1, 9)), (1, (70, 1)),
])
def test_decorations_line_lengths(ctx, ref_tiles, size):
    """Lines of one pixel, of whole and of broken 64-pixel runs, and borders
    whose start lies past the frame's edge."""
    import scene_cases as C
    scene = C.sphere(w=size[0], h=size[1], eye=(0, 0, 2.4),
                     flags=C.ALL | _lib.GR_SHOW_TILE_BOUNDS | _lib.GR_SHOW_CROSSHAIR)
    scene.frame.ref_tiles = ref_tiles
    assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


@pytest.mark.parametrize("size", [(512, 256), (505, 249), (520, 256), (8, 8), (1, 1)])
@pytest.mark.parametrize("grid,eye", [((3, 5), 1.1), ((60, 90), 1.3), ((60, 90), 6.0)])
def test_tile_counting(ctx, size, grid, eye):
    """Frames of exactly 2,048 tiles, one row and one column short of it, past
    it and of one tile, with triangles of hundreds of tiles, of a few and of
    less than one."""
    import scene_cases as C
    scene = C.sphere(w=size[0], h=size[1], eye=(0, 0, eye), nlat=grid[0], nlon=grid[1])
    old = ctx.config()
    ctx.set_config(tile_w=8, tile_h=8)
    try:
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h)


@pytest.mark.parametrize("size", [(8200, 16), (8192, 9), (16, 8200)])
def test_binning_windows(ctx, size):
    """Triangles spanning more tiles than one binning window holds, in a row of
    1,025 tiles (two windows), of 1,024, and in a column."""
    import scene_cases as C
    scene = C.sphere(w=size[0], h=size[1], eye=(0, 0, 1.1), nlat=3, nlon=5)
    old = ctx.config()
    ctx.set_config(tile_w=8, tile_h=8)
    try:
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h)


@pytest.mark.parametrize("objects", [63, 64, 65, 130])
def test_many_objects(ctx, objects):
    """Frames of up to one, and of more than one, wave's worth of objects, some
    of several face blocks."""
    import scene_cases as C
    scene = C.sphere(w=120, h=90, eye=(0, 0, 3.0))
    big = S.latlong_sphere(20, 32, S.SplitMix64(5))
    scene.meshes.append(S.with_texture(big, 0))
    base = scene.objects[0]
    scene.objects = []
    for k in range(objects):
        world = S.world_matrix(scale=(0.2, 0.2, 0.2), rotation=(0.1 * k, 0.2 * k, 0),
                               translation=((k % 11 - 5) * 0.2, (k // 11 - 5) * 0.2, 0.1 * (k % 3)))
        scene.objects.append(S.ObjectData(1 if k % 5 == 0 else 0, S.mvp_matrix(
            base.mvp, S.world_matrix(), world), world))
    assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


def test_face_stage_forms(ctx):
    """The same frames alone (face blocks of four waves) and in a batch of over
    4,096 face blocks (of one wave): survivors on every wave, blocks of broken
    length, faces for the full clipper past a block's own records."""
    import scene_cases as C
    cases = [C.clip_space_soup(n=700, seed=31), C.inside_sphere(), C.cube_scene(),
             C.sphere(w=200, h=120, eye=(0, 0, 1.4), nlat=23, nlon=37),
             C.sphere(w=90, h=70, flags=C.no(_lib.GR_BACKFACE_CULLING), nlat=16, nlon=24)]
    # A million faces out of view: blocks that emit nothing.
    pad = C.sphere(w=16, h=16, nlat=600, nlon=900)
    pad.objects = [S.camera_object(pad.frame, 0, (100.0, 0, 0), (1, 0, 0))]
    frames = cases + [pad]
    handles = [ctx.upload_scene(s)[0] for s in frames]
    outs = [ctx.frame_buffers(s.frame.width, s.frame.height) for s in frames]
    ctx.draw_batch(frames, handles, [(o[0].ptr, o[1].ptr) for o in outs])
    ctx.synchronize()
    stats = ctx.last_stats()
    for k, s in enumerate(cases):
        want = refcpu.draw(s)
        assert_same(s, ctx.draw(s, handles[k]), want)
        h, w = s.frame.height, s.frame.width
        got = (outs[k][0].to_numpy(np.uint8, (h, w, 4)), outs[k][1].to_numpy(np.float32, (h, w)),
               stats[k])
        assert_same(s, got, want)
    for rg, dp in outs:
        rg.free()
        dp.free()
    for hs in handles:
        for h in hs:
            ctx.destroy_mesh(h)


@pytest.mark.parametrize("split", [64, 100, 512])
@pytest.mark.parametrize("eye,grid", [(1.2, (40, 64)), (4.0, (90, 144))])
def test_split_sizes(ctx, split, eye, grid):
    """A frame alone (its lists in parts of at most 64 entries) and in a batch
    of over 4,096 tiles (parts of tile_split): the same frame and statistics,
    for lists of one part, of whole parts and of broken ones."""
    import scene_cases as C
    scene = C.sphere(w=160, h=128, eye=(0, 0, eye), nlat=grid[0], nlon=grid[1])
    pad = C.sphere(w=2048, h=2112)
    pad.objects = []
    frames = [scene, pad]
    handles = [ctx.upload_scene(s)[0] for s in frames]
    outs = [ctx.frame_buffers(s.frame.width, s.frame.height) for s in frames]
    want = refcpu.draw(scene)
    old = ctx.config()
    ctx.set_config(tile_split=split)
    try:
        alone = ctx.draw(scene, handles[0])
        ctx.draw_batch(frames, handles, [(o[0].ptr, o[1].ptr) for o in outs])
        ctx.synchronize()
        stats = ctx.last_stats()[0]
    finally:
        ctx.set_config(tile_split=old.tile_split)
    assert_same(scene, alone, want)
    got = (outs[0][0].to_numpy(np.uint8, (128, 160, 4)),
           outs[0][1].to_numpy(np.float32, (128, 160)), stats)
    assert_same(scene, got, want)
    assert stats == alone[2]
    for rg, dp in outs:
        rg.free()
        dp.free()


@pytest.mark.parametrize("far", [60000.0, 65531.0, 65532.0, 65540.0])
def test_overlays_far_vertices(ctx, far):
    """Unclipped edges and vertex dots up to and past the coordinates that take
    32-bit steps, on every side of the frame."""
    w, h = 64, 48
    px = np.array([[10, 5], [far, 9], [30, 40], [20, 20], [-far + 60, 11], [33, 2],
                   [7, 7], [9, far], [50, 30], [40, 12], [22, -far + 70], [3, 44]], np.float64)
    v = np.ones((12, 4), np.float32)
    v[:, 0], v[:, 1] = (px[:, 0] - w / 2) / (w / 2), (px[:, 1] - h / 2) / (h / 2)
    v[:, 2] = 0.5
    flags = _lib.GR_SHOW_FACES | _lib.GR_SHOW_EDGES | _lib.GR_SHOW_VERTICES
    f = np.arange(12, dtype=np.int32).reshape(4, 3)
    eye = np.eye(4, dtype=np.float32)
    scene = S.SceneData(S.FrameData(w, h, flags=flags), [S.MeshData(v, f)], [],
                        [S.ObjectData(0, eye, eye)], name=f"far-{far}")
    assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


def test_frames_sharing_objects(ctx):
    """Frames of a batch that name the same range of its object array."""
    import scene_cases as C
    scene = C.sphere(w=96, h=64)
    handles = ctx.upload_scene(scene)[0]
    outs = [ctx.frame_buffers(96, 64) for _ in range(9)]
    frames, _, objs, total = ctx.prepare_batch(
        [scene] * 9, [handles] * 9, [(o[0].ptr, o[1].ptr) for o in outs])
    for f in frames:
        f.first_object = 0
    ctx.submit_batch((frames, 9, objs, 1))
    ctx.synchronize()
    want = refcpu.draw(scene)
    for rg, dp in outs:
        assert np.array_equal(rg.to_numpy(np.uint8, (64, 96, 4)), want[0])
        assert np.array_equal(dp.to_numpy(np.uint32, (64, 96)), want[1].view(np.uint32))
        rg.free()
        dp.free()


def test_decorations_batched(ctx):
    """Decorated and plain frames in one batch into shared buffers: each frame
    keeps only its own decorations, and a following draw into the same
    buffers is not painted over."""
    import scene_cases as C
    frames = [C.sphere(w=96, h=64, seed=s, flags=C.ALL | f) for s, f in
              ((21, _lib.GR_SHOW_CROSSHAIR), (22, 0),
               (23, _lib.GR_SHOW_TILE_BOUNDS | _lib.GR_SHOW_CROSSHAIR))]
    handles = [ctx.upload_scene(s)[0] for s in frames]
    outs = [ctx.frame_buffers(96, 64) for _ in frames]
    ctx.draw_batch(frames, handles, [(o[0].ptr, o[1].ptr) for o in outs])
    # The undecorated frame again into the first frame's buffers, right after.
    ctx.draw_batch(frames[1:2], handles[1:2], [(outs[0][0].ptr, outs[0][1].ptr)])
    ctx.synchronize()
    for k, src in ((0, 1), (1, 1), (2, 2)):
        want = refcpu.draw(frames[src])
        got = outs[k][0].to_numpy(np.uint8, (64, 96, 4))
        assert np.array_equal(got, want[0]), f"buffers {k} differ from frame {src}"
    for rg, dp in outs:
        rg.free()
        dp.free()


def test_fog(ctx):
    """gr_fog (FrameBuffer.Fog, rasterizer.go:185-207) over a GPU frame equals
    the oracle's fog over the oracle's frame; the depths span keep, blend and
    fog colour (the background's -1 included)."""
    import scene_cases as C
    scene = C.sphere(w=120, h=90, eye=(0, 0, 2.4))
    want_rgba, want_depth, _ = refcpu.draw(scene)
    d = want_depth[want_depth > 0]
    start, end = float(np.quantile(d, 0.7)), float(np.quantile(d, 0.2))
    want = refcpu.fog(want_rgba, want_depth, start, end, (100, 120, 140, 255))
    h, w = 90, 120
    handles = ctx.upload_scene(scene)[0]
    rg, dp = ctx.frame_buffers(w, h)
    ctx.draw_device(scene, handles, rg.ptr, dp.ptr)
    ctx.fog(rg, dp, w, h, start, end, (100, 120, 140, 255))
    ctx.synchronize()
    got = rg.to_numpy(np.uint8, (h, w, 4))
    assert np.array_equal(got, want)
    assert (got != want_rgba).any(axis=-1).sum() > 1000
    rg.free()
    dp.free()


def test_subpixel_triangles(ctx):
    """A dense sphere far from the camera: most triangles fall between pixel
    centres, and those whose box is at most 2x2 pixels with no covered pixel
    stay out of the tile lists. The image and the counters still equal the
    oracle's, and the lists hold fewer entries than there are triangles."""
    import scene_cases as C
    scene = C.sphere(w=160, h=96, eye=(0, 0, 14.0), nlat=100, nlon=160)
    got = ctx.draw(scene)
    assert_same(scene, got, refcpu.draw(scene))
    st = got[2]
    assert st["refs"] < st["triangles"], st


def _straddling_fans(n=512, seed=9):
    """n triangles given in clip space (identity matrices), each crossing the
    x = -w, x = w and y = w planes: every face reaches the clipper and reserves
    the largest fan, 7 records, so each 256-face block needs 1,792 records and
    takes all but its first 320 from the overflow pools."""
    rng = S.SplitMix64(S.SEED_BASE + 700 + seed)
    # Inside the clip volume is w < 0, |x|, |y| <= -w and znear <= z <= zfar.
    base = np.array([[-2.0, -0.2, 0.5, -1.0], [0.0, 2.0, 0.5, -1.0], [2.0, -0.1, 0.5, -1.0]])
    jit = (rng.uniform(n * 12).reshape(n, 3, 4) - 0.5) * np.array([0.4, 0.4, 0.2, 0.0])
    v4 = (base[None] + jit).reshape(3 * n, 4).astype(np.float32)
    f = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    nrm = np.tile(np.array([[0.0, 0.0, 1.0, 1.0]], np.float32), (3 * n, 1))
    uvs = (rng.uniform(6 * n).reshape(n, 3, 2)).astype(np.float32)
    m = S.MeshData(v4, f, nrm, f.copy(), uvs)
    t = S.random_texture(rng, 8, 8)
    S.with_texture(m, 0)
    fr = S.FrameData(96, 72, flags=_lib.GR_DEFAULT_FLAGS & ~_lib.GR_BACKFACE_CULLING)
    eye = np.eye(4, dtype=np.float32)
    return S.SceneData(fr, [m], [t], [S.ObjectData(0, eye, eye)], name="straddling-fans")


def test_overflow_records(ctx):
    """Faces that all reach the clipper: most of their records come from the
    overflow pools. Equal to the oracle at the default capacity, and with a
    capacity so small that the pools run out (the batch reports it, the
    capacity grows and the frame is drawn again)."""
    scene = _straddling_fans()
    want = refcpu.draw(scene)
    assert want[2]["triangles"] > 0
    assert_same(scene, ctx.draw(scene), want)
    old = ctx.config()
    try:
        ctx.set_config(refs_capacity=1024)
        got = ctx.draw(scene)
        assert ctx.config().refs_capacity > 1024
    finally:
        ctx.set_config(refs_capacity=old.refs_capacity)
    assert_same(scene, got, want)


@pytest.mark.parametrize("side,kind,scale,stretch,step", [
    ((64, 16), 2, 1.0, 1.0, 1), ((16, 64), 2, 3.5, 40.0, 7), ((1, 1), 2, 1.0, 5.0, 333),
    ((100, 37), 1, 1.0, 1.0, 10), ((100, 37), 1, 2.5, -9.0, 2), ((1, 3), 1, 1.0, 2000.0, 64),
    ((17, 17), 1, 1.0, 3e5, 3), ((17, 17), 1, 1024.0, 1.0, 2**31 - 1), ((17, 17), 1, 1025.0, 1.0, 0),
    ((64, 64), 2, 1e-13, 1e20, -5), ((17, 17), 1, 0.0, 1e30, 65), ((17, 17), 1, -2.0, 1e-30, 64),
    ((64, 64), 2, 1.0, 1e30, 63), ((17, 17), 1, 1.0, float("inf"), 16), ((64, 64), 2, 1.0, 0.0, 32)])
def test_shading_forms(ctx, side, kind, scale, stretch, step):
    """Texture sides, scales and coordinates on both sides of the shortened
    quotient, remainder and index, and steps of the dot grid."""
    import scene_cases as C
    scene = C.sphere(w=200, h=130, eye=(0, 0, 1.6), nlat=14, nlon=22)
    w, h = side
    rgba = np.random.default_rng(5).integers(0, 256, (h, w, 4), dtype=np.uint8)
    scene.textures[:] = [S.TextureData(kind, w, h, scale, rgba=rgba)] * len(scene.textures)
    mesh = scene.meshes[0]
    with np.errstate(invalid="ignore"):
        mesh.uvs = (np.asarray(mesh.uvs) * np.float32(stretch)).astype(np.float32)
    scene.frame.dot_step = step
    with np.errstate(invalid="ignore"):
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))


@pytest.mark.parametrize("grid,eye,tile", [
    ((100, 160), 4.5, (32, 32)), ((100, 160), 2.2, (8, 64)), ((100, 160), 3.0, (64, 64)),
    ((200, 320), 9.0, (16, 16)), ((200, 320), 5.0, (64, 8))])
def test_dense_batches(ctx, grid, eye, tile):
    """Batches that take the dense raster, at several tile shapes: chunks of
    small boxes, of mixed ones, and of boxes cut by their tile."""
    import scene_cases as C
    scene = C.sphere(w=331, h=245, eye=(0.02, 0.01, eye), nlat=grid[0], nlon=grid[1])
    want = refcpu.draw(scene)
    tiles = -(-331 // tile[0]) * -(-245 // tile[1])
    old = ctx.config()
    try:
        ctx.set_config(tile_w=tile[0], tile_h=tile[1], refs_capacity=1 << 23)
        handles = ctx.upload_scene(scene)[0]
        n = 4096 // tiles + 1
        outs = [ctx.frame_buffers(331, 245) for _ in range(n)]
        ctx.draw_batch([scene] * n, [handles] * n, [(o[0].ptr, o[1].ptr) for o in outs])
        ctx.synchronize()
        stats = ctx.last_stats()
        for k, (rg, dp) in enumerate(outs):
            assert np.array_equal(rg.to_numpy(np.uint8, (245, 331, 4)), want[0]), k
            assert np.array_equal(dp.to_numpy(np.uint32, (245, 331)), want[1].view(np.uint32)), k
            assert stats[k]["fragments_covered"] == want[2]["fragments_covered"]
            rg.free()
            dp.free()
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h, refs_capacity=old.refs_capacity)


def _soup(n, w, h, px, seed=1):
    """n triangles of about px pixels at random places, drawn in no order of place."""
    rng = np.random.default_rng(seed)
    c = rng.uniform([2, 2], [w - 2, h - 2], (n, 1, 2))
    a = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0, 2 * np.pi / 3, 4 * np.pi / 3])
    p = np.clip(c + px * np.stack([np.cos(a), np.sin(a)], -1), 0, [w - 1, h - 1]).reshape(-1, 2)
    v = np.ones((3 * n, 4), np.float32)
    v[:, 0], v[:, 1] = (p[:, 0] - w / 2) / (w / 2), (p[:, 1] - h / 2) / (h / 2)
    v[:, 2] = 0.5 + 0.4 * np.sin(np.arange(3 * n))
    # Both windings: about half of the faces cover pixels whichever side counts.
    f = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    f[::2] = f[::2, ::-1]
    eye = np.eye(4, dtype=np.float32)
    return S.SceneData(S.FrameData(w, h, flags=_lib.GR_SHOW_FACES), [S.MeshData(v, f)], [],
                       [S.ObjectData(0, eye, eye)], name=f"soup-{n}-{px}")


@pytest.mark.parametrize("size", [(256, 256), (520, 257), (1041, 1033)])
@pytest.mark.parametrize("n,px", [(40, 3), (300, 14), (300, 15), (700, 40), (1300, 200), (9000, 6)])
def test_binning_scattered_triangles(ctx, size, n, px):
    """Face blocks whose triangles lie all over the frame, in one binning window
    (1,024 tiles), a few and many: placed by references or through the windows,
    boxes on either side of what a lane places by itself, few and many of them."""
    scene = _soup(n, *size, px)
    old = ctx.config()
    ctx.set_config(tile_w=8, tile_h=8, refs_capacity=1 << 22)
    try:
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h, refs_capacity=old.refs_capacity)


def test_binning_cost_follows_the_references(ctx):
    """Small triangles all over a frame of 129,600 tiles: placing their few thousand
    references takes less than the raster of the frame (it took five times as long
    when every block went through all windows of the frame)."""
    scene = _soup(20000, 3840, 2160, 8)
    old = ctx.config()
    ctx.set_config(tile_w=8, tile_h=8, pipelines=1)
    try:
        handles = ctx.upload_scene(scene)[0]
        rg, dp = ctx.frame_buffers(3840, 2160)
        best = {}
        ctx.set_kernel_timing(True)
        for _ in range(6):
            ctx.reset_kernel_times()
            ctx.draw_device(scene, handles, rg.ptr, dp.ptr)
            ctx.synchronize()
            for k, (ms, _) in ctx.kernel_times().items():
                best[k] = min(best.get(k, 1e9), ms)
        assert best["k_bin_fill"] < best["k_raster"], best
        rg.free()
        dp.free()
    finally:
        ctx.set_kernel_timing(False)
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h, pipelines=old.pipelines)


@pytest.mark.parametrize("n,px,tile", [(6000, 40, 8), (2500, 90, 16), (9000, 12, 8), (3000, 60, 64)])
def test_split_shares(ctx, n, px, tile):
    """Lists of over 64 entries in every tile, about as long as a share of the
    launch's entries (some are left whole), alone and beside frames that leave one
    frame's lists above the share of the batch or put them below it."""
    scene = _soup(n, 512, 512, px)
    light = _soup(200, 512, 512, 20, seed=3)
    heavy = _soup(9000, 256, 256, 60, seed=4)
    want = [refcpu.draw(s) for s in (scene, light, heavy)]
    old = ctx.config()
    ctx.set_config(tile_w=tile, tile_h=tile, refs_capacity=1 << 23)
    try:
        handles = [ctx.upload_scene(s)[0] for s in (scene, light, heavy)]
        assert_same(scene, ctx.draw(scene, handles[0]), want[0])
        for batch in ([0, 1], [0, 2], [1, 2, 0]) if tile > 8 else ([1], [2]):
            frames = [(scene, light, heavy)[k] for k in batch]
            outs = [ctx.frame_buffers(s.frame.width, s.frame.height) for s in frames]
            ctx.draw_batch(frames, [handles[k] for k in batch], [(o[0].ptr, o[1].ptr) for o in outs])
            ctx.synchronize()
            stats = ctx.last_stats()
            for j, k in enumerate(batch):
                h, w = frames[j].frame.height, frames[j].frame.width
                got = (outs[j][0].to_numpy(np.uint8, (h, w, 4)),
                       outs[j][1].to_numpy(np.float32, (h, w)), stats[j])
                assert_same(frames[j], got, want[k])
                for b in outs[j]:
                    b.free()
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h, refs_capacity=old.refs_capacity)


@pytest.mark.parametrize("size", [(512, 256), (520, 256)])
@pytest.mark.parametrize("grid", [(190, 258), (191, 259)])
def test_face_stage_forms_by_tiles(ctx, size, grid):
    """383 and 387 face blocks, either side of the four-wave form's limit in frames
    of more than 2,048 tiles, in a frame of 2,048 and in one of more."""
    import scene_cases as C
    scene = C.sphere(w=size[0], h=size[1], eye=(0, 0, 2.6), nlat=grid[0], nlon=grid[1])
    blocks = -(-len(scene.meshes[0].vertex_indices) // 256)
    assert (blocks <= 384) == (grid[0] == 190)
    old = ctx.config()
    ctx.set_config(tile_w=8, tile_h=8)
    try:
        assert_same(scene, ctx.draw(scene), refcpu.draw(scene))
    finally:
        ctx.set_config(tile_w=old.tile_w, tile_h=old.tile_h)


@pytest.mark.parametrize("size", [(16384, 9), (9, 16384), (8191, 65)])
def test_overlays_long_lines(ctx, size):
    """Edges of tens of thousands of steps whose float32 positions drift by many
    pixels, shallow and steep, across wide and tall frames and far beside them."""
    w, h = size
    far = 45000.0
    px = np.array([[-far, 3], [5000, h - 2], [w / 2, -far],
                   [w / 3, far], [w + 20000.0, h / 2], [-20000.0, 2],
                   [-40000, -40000], [3000, 4000], [w - 3, h - 3],
                   [-32768, 32768], [32000, 49221], [w / 2, h / 2]], np.float64)
    v = np.ones((12, 4), np.float32)
    v[:, 0], v[:, 1] = (px[:, 0] - w / 2) / (w / 2), (px[:, 1] - h / 2) / (h / 2)
    v[:, 2] = 0.5
    flags = _lib.GR_SHOW_FACES | _lib.GR_SHOW_EDGES | _lib.GR_SHOW_VERTICES
    f = np.arange(12, dtype=np.int32).reshape(4, 3)
    eye = np.eye(4, dtype=np.float32)
    scene = S.SceneData(S.FrameData(w, h, flags=flags), [S.MeshData(v, f)], [],
                        [S.ObjectData(0, eye, eye)], name=f"long-{w}")
    want = refcpu.draw(scene)
    assert (want[0][..., :3] == 0).all(-1).sum() > 50  # edge pixels in the frame
    assert_same(scene, ctx.draw(scene), want)
