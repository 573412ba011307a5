"""The traversal at the edges of its slab test and triangle set-up: direction
components that are zero, on and beside flat boxes; instances scaled far up
and down, mirrored and far from the origin (the bias o / d large beside the
boxes, divisions outside the range of the shared reciprocal).  Closest-hit
ids and tie flags are bit-exact against the oracle, and the wavefront and
per-sample schedules agree bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (left, up, forward): components of the directions that are exactly zero
FRAMES = {
    "free": ((1, 0, 0), (0, 1, 0), (0, 0, -1)),
    "x0": ((0, 0, 0), (0, 1, 0), (0, 0, -1)),
    "y0": ((1, 0, 0), (0, 0, 0), (0, 0, -1)),
    "along_z": ((0, 0, 0), (0, 0, 0), (0, 0, -1)),
    "along_x": ((0, 0, 0), (0, 0, 0), (1, 0, 0)),
    "minus_y": ((0, 0, 0), (0, 0, 0), (0, -1, 0)),
    "tiny_x": ((1e-25, 0, 0), (0, 1, 0), (0, 0, -1)),
}


def _scene(wl, scale, shift):
    """A floor on y = 0, boxes standing on it and a sphere, as instances of
    meshes at unit size, scaled by `scale` and moved by `shift`; one mirrored."""
    d = wl.SceneDesc()
    d.materials.append(("pbr", dict(base_color=(0.7, 0.6, 0.5, 1.0), metallic=0.3, roughness=0.4)))
    d.materials.append(("om_nk",) + wl.rng_om(1))
    for v, f, uv in (wl.plane(6, 6, 3.0, 0.0), wl.grid_box(3, (0.5, 0.5, 0.5))):
        d.meshes.append({"vertices": v, "faces": f, "mat_id": 0, "uvs": [uv]})
    v, f = wl.icosphere(2, 0.6)
    d.meshes.append({"vertices": v, "faces": f, "mat_id": 1})

    def put(t, mesh, sc=(1, 1, 1), axis=(0, 1, 0), angle=0.0):
        t = tuple(scale * x + y for x, y in zip(t, shift))
        d.instances.append((wl.trs(t, axis, angle, tuple(scale * x for x in sc)), mesh))

    put((0, 0, 0), 0)
    put((0.0, 0.5, -1.0), 1)
    put((1.2, 0.5, 0.0), 1, sc=(-1, 1, 1))
    put((-1.1, 0.7, 0.2), 2, axis=(1, 1, 0), angle=0.7)
    put((0.3, 0.6, 1.0), 2, sc=(0.2, 0.4, 1e-3))
    d.lights.append((tuple(scale * x + y for x, y in zip((2.0, 3.0, 2.0), shift)), (40.0 * scale,) * 3, -1.0))
    d.background = ("const", (0.2, 0.3, 0.4))
    return d


def _camera(pkg, frame, scale, shift, w=37, h=29):
    cam = pkg.Camera(w, h, yfov=50.0)
    x, y, z = FRAMES[frame]
    # Off the meshes' planes of symmetry: there a whole frame of rays with x = 0
    # runs along shared edges, where the oracle's own boxes (padded by 1e-6) may
    # leave out one of two faces hit at the same t (test_rays_along_shared_edges).
    x0, y0 = 0.0137, 0.0 if frame == "y0" else 0.5071
    at = {"along_x": (-4.0, y0, -1.0 + x0), "minus_y": (x0, 4.0, -1.0)}.get(frame, (x0, y0, 4.0))
    cam.set_viewpoint(tuple(scale * a + b for a, b in zip(at, shift)), x, y, z)
    return cam


PLACES = [(1.0, (0, 0, 0)), (1e-4, (0, 0, 0)), (3e5, (0, 0, 0)), (1.0, (4096.0, -512.0, 20000.0)), (1e-20, (0, 0, 0))]


@pytest.mark.parametrize("place", range(len(PLACES)))
@pytest.mark.parametrize("frame", list(FRAMES))
def test_ids_match_the_oracle(pkg, wl, ref, frame, place):
    scale, shift = PLACES[place]
    d = _scene(wl, scale, shift)
    d.lights.clear()
    d.fc_subject = "ipid"
    cam = _camera(pkg, frame, scale, shift)
    s = pkg.Scene()
    d.apply(s, pkg.pbr_desc)
    r = pkg.Renderer(pkg.default_params(seed=3))
    r.set_scene(s)
    _, ids, tie = r.render_fc(cam)
    rs = ref.Scene()
    d.apply(rs, ref.pbr_desc)
    _, rids, rtie = rs.render_fc(ref.default_params(seed=3), cam.desc())
    assert np.array_equal(ids, rids)
    assert np.array_equal(tie, rtie)
    if frame == "free" and scale > 1e-10:
        assert (ids[0] >= 0).mean() > 0.2   # the view does hit geometry


@pytest.mark.parametrize("build", ["host", "device"])
@pytest.mark.parametrize("place", [0, 1, 2, 3])
@pytest.mark.parametrize("frame", ["x0", "y0", "along_z", "along_x", "minus_y"])
def test_rays_along_shared_edges(pkg, wl, ref, frame, place, build):
    """A camera on the meshes' planes of symmetry: rays run along edges that
    two faces share, and along flat boxes' planes.  Both faces have to be
    seen: ids and tie flags are those of a loop over all triangles."""
    import ctypes as C
    scale, shift = PLACES[place]
    d = _scene(wl, scale, shift)
    d.lights.clear()
    d.fc_subject = "ipid"
    w, h, seed = 23, 17, 3
    cam = pkg.Camera(w, h, yfov=50.0)
    at = {"along_x": (-4.0, 0.5, -1.0), "minus_y": (0.0, 4.0, -1.0)}.get(frame, (0.0, 0.0 if frame == "y0" else 0.5, 4.0))
    cam.set_viewpoint(tuple(scale * a + b for a, b in zip(at, shift)), *FRAMES[frame])
    s = pkg.Scene()
    s.set_build_mode(pkg.BUILD_DEVICE_LBVH if build == "device" else pkg.BUILD_HOST_SAH)
    d.apply(s, pkg.pbr_desc)
    r = pkg.Renderer(pkg.default_params(seed=seed))
    r.set_scene(s)
    _, ids, tie = r.render_fc(cam)
    rs = ref.Scene()
    d.apply(rs, ref.pbr_desc)
    lib, desc = ref.lib(), ref.CameraDesc.from_buffer_copy(cam.desc())
    want, wtie = np.full((2, h, w), -1), np.zeros((h, w), int)
    for p in range(w * h):   # the pass's ray of every pixel: jitter from the camera stream, origin off the position by its ulps
        bits, o, dv = (C.c_uint32 * 4)(), np.zeros(3, np.float32), np.zeros(3, np.float32)
        lib.ref_philox4x32_10((C.c_uint32 * 4)(0, 0, p, 0), (C.c_uint32 * 2)(seed, 0), bits)
        lib.ref_camera_ray(C.byref(desc), p % w, p // w, lib.ref_u01(bits[0]), lib.ref_u01(bits[1]), ref.ptr(o), ref.ptr(dv))
        o = o + np.float32(3 * 2.0**-23) * max(np.float32(1), np.abs(o).max()) * dv
        hit = rs.closest_hit(o, dv, bvh=False)[0]
        if hit:
            want[:, p // w, p % w], wtie[p // w, p % w] = (hit[4], hit[3]), hit[5]
    base = np.cumsum([0] + [len(m["faces"]) for m in d.meshes])
    ids = ids.reshape(4, h, w)
    got = np.where(ids[0] >= 0, ids[0] - base[np.maximum(ids[1], 0)], -1)
    assert np.array_equal(got, want[0]) and np.array_equal(ids[3], want[1])
    assert np.array_equal(np.asarray(tie).reshape(h, w), wtie)
    assert (got >= 0).mean() > 0.2


@pytest.mark.parametrize("place", [0, 1, 3])
@pytest.mark.parametrize("frame", ["free", "x0", "y0"])
def test_schedules_agree(pkg, wl, frame, place):
    scale, shift = PLACES[place]
    d = _scene(wl, scale, shift)
    cam = _camera(pkg, frame, scale, shift)
    s = pkg.Scene()
    d.apply(s, pkg.pbr_desc)
    films = []
    for sched in (pkg.SCHEDULE_WAVEFRONT, pkg.SCHEDULE_PER_SAMPLE):
        r = pkg.Renderer(pkg.default_params(samples_per_pixel=3, camera_bounces=4, light_bounces=3, max_path_length=5, seed=9))
        r.set_scene(s)
        r.set_schedule(sched)
        films.append(r.render(cam))
        assert r.stats()["stack_overflows"] == 0
    assert np.array_equal(films[0], films[1])


@pytest.mark.parametrize("keep", [0, 1, 33, 64])
@pytest.mark.parametrize("size", [(1, 1), (63, 1), (64, 1), (65, 1), (129, 3)])
def test_refill_at_the_edges_of_a_list(pkg, wl, keep, size):
    """The refilling traversal at queue lengths around a wave's 64 entries, and
    at several lists per wave (few workgroups), banded and not: every entry is
    traced once, so films and ray counts equal the per-sample schedule's."""
    desc, view = wl.mixed_test_scene(hdr=True, lights=True)
    view.width, view.height = size
    s = pkg.Scene()
    desc.apply(s, pkg.pbr_desc)
    cam = pkg.Camera(view.width, view.height, view.position, view.forward, view.up, view.yfov)
    params = dict(samples_per_pixel=1, camera_bounces=5, light_bounces=3, max_path_length=6, seed=21, extensions=pkg.EXT_HDRI_NEE)
    ref = pkg.Renderer(pkg.default_params(**params))
    ref.set_scene(s)
    ref.set_schedule(pkg.SCHEDULE_PER_SAMPLE)
    want, st = ref.render(cam), ref.stats()
    for tuning in (dict(), dict(trace_blocks_per_cu=1, xcd_bands=1), dict(xcd_bands=16)):
        r = pkg.Renderer(pkg.default_params(**params))
        r.set_scene(s)
        r.set_tuning(trace_keep=keep, **tuning)
        assert np.array_equal(r.render(cam), want)
        for k in ("rays", "camera_rays", "light_rays", "shadow_rays"):
            assert r.stats()[k] == st[k], k


@pytest.mark.parametrize("build", ["host", "device"])
@pytest.mark.parametrize("place", [0, 1, 3])
def test_turned_instances(pkg, wl, ref, place, build):
    """Instance boxes come from several boxes of a mesh, each turned by the
    instance's matrix: meshes of one leaf, of one triangle, far from their own
    origin, plates that lie back in a plane of the world, turned, sheared and
    mirrored.  Ids and tie flags are the oracle's, under both builders."""
    scale, shift = PLACES[place]
    d = wl.SceneDesc()
    d.materials.append(("pbr", dict(base_color=(0.7, 0.6, 0.5, 1.0), metallic=0.3, roughness=0.4)))
    tri = np.array([[-0.6, -0.4, 0.1], [0.7, -0.3, -0.2], [0.05, 0.65, 0.15]], np.float32)
    d.meshes.append({"vertices": tri, "faces": np.array([[0, 1, 2]], np.uint32), "mat_id": 0})
    v, f, _ = wl.plane(6, 6, 0.8, 0.0)
    c, q = np.cos(0.6), np.sin(0.6)
    turn = np.array([[c, -q, 0], [q, c, 0], [0, 0, 1]])   # the plate at 0.6 rad about z
    d.meshes.append({"vertices": (v @ turn.T).astype(np.float32), "faces": f, "mat_id": 0})
    v, f, _ = wl.grid_box(4, (0.9, 0.1, 0.05))
    d.meshes.append({"vertices": v, "faces": f, "mat_id": 0})
    v, f = wl.icosphere(3, 0.5)
    d.meshes.append({"vertices": (v + np.array([30.0, 0.0, -20.0], np.float32)).astype(np.float32), "faces": f, "mat_id": 0})
    rng = np.random.default_rng(5)
    for i in range(40):
        a = wl.trs((0, 0, 0), rng.normal(size=3), rng.uniform(0, 6.3), rng.uniform(0.3, 1.2, 3) * rng.choice([-1, 1], 3))
        m = np.array(a, np.float64).reshape(-1, 4)
        if i % 5 == 4:
            m[:3, :3] = m[:3, :3] @ np.array([[1, 0.7, 0], [0, 1, -0.4], [0, 0, 1]])
        if i % 4 == 1 and i < 20:   # the plates, turned back into y = const
            m[:3, :3] = turn.T
        at = rng.uniform(-1.8, 1.8, 3)
        if i % 4 == 3:
            at = at - m[:3, :3] @ np.array([30.0, 0.0, -20.0])
        m[:3, :3] *= scale
        m[:3, 3] = scale * at + np.array(shift)
        d.instances.append((np.asarray(m, np.float32).reshape(np.shape(a)), i % 4))
    d.fc_subject = "ipid"
    cam = _camera(pkg, "free", scale, shift, 97, 83)
    s = pkg.Scene()
    s.set_build_mode(pkg.BUILD_DEVICE_LBVH if build == "device" else pkg.BUILD_HOST_SAH)
    d.apply(s, pkg.pbr_desc)
    r = pkg.Renderer(pkg.default_params(seed=3))
    r.set_scene(s)
    _, ids, tie = r.render_fc(cam)
    rs = ref.Scene()
    d.apply(rs, ref.pbr_desc)
    _, rids, rtie = rs.render_fc(ref.default_params(seed=3), cam.desc())
    assert np.array_equal(ids, rids)
    assert np.array_equal(tie, rtie)
    assert (ids[0] >= 0).mean() > 0.2


def _inside(value):
    """What a program can pass for a place: none of it is refused."""
    return {"inf_x": (np.inf, 0.0, 0.0), "nan": (np.nan,) * 3, "inf": (np.inf, -np.inf, np.inf), "minus_inf": (-np.inf,) * 3}[value]


ODD = ["flat", "flatter", "point", "far"] + [f"{k}_{v}" for k in ("instance", "light", "camera") for v in ("inf_x", "nan", "inf", "minus_inf")]


@pytest.mark.parametrize("build", ["host", "device"])
@pytest.mark.parametrize("odd", ODD)
def test_rays_that_cull_on_no_axis(pkg, wl, ref, odd, build):
    """Instances of a singular matrix (their inverse is inf and NaN), of a
    scale beyond the slab test's range, and instances, lights and cameras at
    places that are not finite: the box test may cull on no axis, so empty
    child slots are taken for hit.  Ids are the oracle's; rounds, film tiles,
    wave packets and the allocation-free render give the per-sample schedule's
    film."""
    import torch
    d = _scene(wl, 1.0, (0, 0, 0))
    cam = _camera(pkg, "free", 1.0, (0, 0, 0))
    kind, _, value = odd.partition("_")
    rng = np.random.default_rng(6)
    for k in range(6):   # turned plates, boxes and spheres, each under the odd matrix
        at = rng.uniform(-1.0, 1.0, 3) + (0.0, 0.6, 0.0)
        scale = {"flat": (1, 1, 0), "flatter": (0, 1, 0), "point": (0, 0, 0), "far": (1e32, 1e32, 1e32)}.get(kind, (0.3, 0.3, 0.3))
        m = np.array(wl.trs(tuple(at), rng.normal(size=3), 0.7 + k, scale), np.float32)
        if kind == "instance":
            m.reshape(-1, 4)[:3, 3] = _inside(value)
        d.instances.append((m, k % 3))
    if kind == "light":
        d.lights.append((_inside(value), (40.0,) * 3, -1.0))
    if kind == "camera":
        cam.set_viewpoint(_inside(value), (1, 0, 0), (0, 1, 0), (0, 0, -1))
    d.fc_subject = "ipid"
    s = pkg.Scene()
    s.set_build_mode(pkg.BUILD_DEVICE_LBVH if build == "device" else pkg.BUILD_HOST_SAH)
    d.apply(s, pkg.pbr_desc)
    params = dict(samples_per_pixel=2, camera_bounces=4, light_bounces=3, max_path_length=5, seed=9)
    print(f"odd case {odd} {build}", flush=True)
    r = pkg.Renderer(pkg.default_params(seed=3))
    r.set_scene(s)
    _, ids, tie = r.render_fc(cam)
    rs = ref.Scene()
    d.apply(rs, ref.pbr_desc)
    _, rids, rtie = rs.render_fc(ref.default_params(seed=3), cam.desc())
    assert np.array_equal(ids, rids) and np.array_equal(tie, rtie)
    if kind != "camera":
        assert (ids[0] >= 0).mean() > 0.2
    one = pkg.Renderer(pkg.default_params(**params))
    one.set_scene(s)
    one.set_schedule(pkg.SCHEDULE_PER_SAMPLE)
    want = one.render(cam)
    assert one.stats()["stack_overflows"] == 0
    for tuning in (dict(), dict(tail_round=1), dict(tail_round=2), dict(traversal=2), dict(sort_rays=2)):
        r = pkg.Renderer(pkg.default_params(**params))
        r.set_scene(s)
        if tuning:
            r.set_tuning(**tuning)
        assert np.array_equal(r.render(cam), want, equal_nan=True), tuning
    film = torch.empty(cam.desc().height, cam.desc().width, 4, device="cuda")
    torch.cuda.synchronize()   # the film's allocation, before a stream that does not wait for torch's
    one.render_noalloc(cam, film.data_ptr())
    torch.cuda.synchronize()
    assert np.array_equal(film.cpu().numpy().reshape(want.shape), want, equal_nan=True)


@pytest.mark.parametrize("build", ["host", "device"])
@pytest.mark.parametrize("away", [250.0, 262.0, 4e3, 3e5, 2e6])
def test_meshes_far_from_their_origin(pkg, wl, ref, away, build):
    """Meshes on either side of the distance (256 times their size) from which
    their boxes are relative to a pivot, turned and scaled, among meshes about
    their origin: the oracle's ids, one film in every schedule, and about as
    many node visits as for the same mesh about its origin."""
    v, f = wl.icosphere(3, 0.5)
    at = np.float32([away, -0.25 * away, 0.5 * away])
    far = (v + at).astype(np.float32)
    rng = np.random.default_rng(8)
    places = [(rng.normal(size=3), rng.uniform(0, 6.3), rng.uniform(0.4, 1.0, 3), rng.uniform(-1.5, 1.5, 3)) for _ in range(16)]

    def scene(moved):
        d = wl.SceneDesc()
        d.materials.append(("pbr", dict(base_color=(0.7, 0.6, 0.5, 1.0), metallic=0.3, roughness=0.4)))
        d.meshes.append({"vertices": far if moved else (far - at).astype(np.float32), "faces": f, "mat_id": 0})
        d.meshes.append({"vertices": v, "faces": f, "mat_id": 0})
        for k, (axis, angle, size, place) in enumerate(places):
            m = np.array(wl.trs((0, 0, 0), axis, angle, size), np.float64).reshape(4, 4)
            m[:3, 3] = place - (m[:3, :3] @ at.astype(np.float64) if moved and k % 2 == 0 else 0.0)
            d.instances.append((m.astype(np.float32), k % 2))
        d.lights.append(((2.0, 3.0, 2.0), (40.0,) * 3, -1.0))
        d.background = ("const", (0.2, 0.3, 0.4))
        d.fc_subject = "ipid"
        s = pkg.Scene()
        s.set_build_mode(pkg.BUILD_DEVICE_LBVH if build == "device" else pkg.BUILD_HOST_SAH)
        d.apply(s, pkg.pbr_desc)
        return d, s

    cam = _camera(pkg, "free", 1.0, (0, 0, 0), 97, 83)
    d, s = scene(True)
    r = pkg.Renderer(pkg.default_params(seed=3))
    r.set_scene(s)
    _, ids, tie = r.render_fc(cam)
    visits = r.stats()["nodes_visited"]
    rs = ref.Scene()
    d.apply(rs, ref.pbr_desc)
    _, rids, rtie = rs.render_fc(ref.default_params(seed=3), cam.desc())
    assert np.array_equal(ids, rids) and np.array_equal(tie, rtie)
    assert (ids[0] >= 0).mean() > 0.2
    _, near = scene(False)
    r.set_scene(near)
    r.render_fc(cam)
    if away < 1e5:   # farther off, the instances' boxes carry the rounding of their own transforms
        assert visits <= 1.2 * r.stats()["nodes_visited"]
    params = dict(samples_per_pixel=2, camera_bounces=4, light_bounces=3, max_path_length=5, seed=9)
    one = pkg.Renderer(pkg.default_params(**params))
    one.set_scene(s)
    one.set_schedule(pkg.SCHEDULE_PER_SAMPLE)
    want = one.render(cam)
    for tuning in (dict(), dict(tail_round=1), dict(traversal=2)):
        r = pkg.Renderer(pkg.default_params(**params))
        r.set_scene(s)
        if tuning:
            r.set_tuning(**tuning)
        assert np.array_equal(r.render(cam), want), tuning
