"""Tiny and ragged films (1 x 1, one row, one column, odd sizes) through the
wavefront and per-sample schedules, the false-colour pass and the post pass:
far fewer samples than one traversal grid holds, and post windows that fall
off every edge.  Bars as in the full-size parity tests: films of the two
schedules bit-identical, ids and tie flags bit-exact against the oracle,
radiance per pixel within 1e-3 relative, post floats within 2 ulp."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 7), (13, 1), (3, 5), (2, 2)]
PARAMS = dict(samples_per_pixel=3, camera_bounces=4, light_bounces=3, max_path_length=5, seed=21)


def _scene(pkg, wl, w, h):
    desc, view = wl.mixed_test_scene(hdr=True, lights=True)
    s = pkg.Scene()
    desc.apply(s, pkg.pbr_desc)
    # a narrow field of view on the middle of the scene, so the few pixels see geometry
    cam = pkg.Camera(w, h, view.position, view.forward, view.up, 12.0)
    return desc, s, cam


@pytest.mark.parametrize("w,h", SIZES)
def test_small_film_radiance(pkg, wl, ref, w, h):
    print(f"small film {w}x{h}", flush=True)
    desc, s, cam = _scene(pkg, wl, w, h)
    films = []
    for sched in (pkg.SCHEDULE_WAVEFRONT, pkg.SCHEDULE_PER_SAMPLE):
        r = pkg.Renderer(pkg.default_params(**PARAMS))
        r.set_scene(s)
        r.set_schedule(sched)
        films.append(r.render(cam).copy())
        assert r.stats()["samples"] == w * h * PARAMS["samples_per_pixel"]
    assert films[0].shape == (h, w, 4)
    assert np.array_equal(films[0], films[1])
    rs = ref.Scene()
    desc.apply(rs, ref.pbr_desc)
    rimg = rs.render(ref.default_params(**PARAMS), cam.desc(), threads=4)[0]
    a, b = films[0][..., :3].astype(np.float64), rimg[..., :3].astype(np.float64)
    assert np.all(np.isfinite(a))
    err = np.abs(a - b) / np.maximum(np.abs(b), 1e-3)
    assert err.max() < 1e-3, err.max()
    for denoise in (False, True):
        f, _ = r.post(cam, gamma=0.5, denoise=denoise)
        rf, _ = ref.post(films[1], gamma=0.5, denoise=denoise)
        ulp = np.abs(f.view(np.int32).astype(np.int64) - rf.view(np.int32).astype(np.int64))
        assert ulp.max() <= 2, (denoise, ulp.max())


@pytest.mark.parametrize("w,h", SIZES)
def test_small_film_ids(pkg, wl, ref, w, h):
    print(f"small film ids {w}x{h}", flush=True)
    desc, _, _ = _scene(pkg, wl, w, h)
    desc.fc_subject = "pid"
    desc.background = None
    s = pkg.Scene()
    desc.apply(s, pkg.pbr_desc)
    _, _, cam = _scene(pkg, wl, w, h)
    r = pkg.Renderer(pkg.default_params(seed=7))
    r.set_scene(s)
    film, ids, tie = r.render_fc(cam)
    rs = ref.Scene()
    desc.apply(rs, ref.pbr_desc)
    rfilm, rids, rtie = rs.render_fc(ref.default_params(seed=7), cam.desc())
    assert np.array_equal(ids, rids) and np.array_equal(tie, rtie) and np.array_equal(film, rfilm)


@pytest.mark.parametrize("ext", [0, 1, 2])
@pytest.mark.parametrize("lights", [False, True])
def test_default_schedule_at_the_tile_limit(pkg, wl, lights, ext):
    """With the default tuning a render of at most 2^18 samples is one launch
    over film tiles, a larger one ray-queue rounds: on both sides of the limit
    film and ray counts equal those of the rounds (any tuning set) bit for bit,
    also when one renderer goes from one to the other and back."""
    desc, view = wl.mixed_test_scene(hdr=True, lights=lights, masked=True)
    s = pkg.Scene()
    desc.apply(s, pkg.pbr_desc)
    params = dict(samples_per_pixel=4, camera_bounces=3, light_bounces=2, max_path_length=4, seed=5, extensions=ext)
    r, q = pkg.Renderer(pkg.default_params(**params)), pkg.Renderer(pkg.default_params(**params))
    q.set_tuning(tail_round=1)
    for x in (r, q):
        x.set_scene(s)
    for w, h in ((256, 256), (257, 256), (37, 5)):
        cam = pkg.Camera(w, h, view.position, view.forward, view.up, view.yfov)
        assert np.array_equal(r.render(cam), q.render(cam))
        a, b = r.stats(), q.stats()
        for k in ("samples", "rays", "camera_rays", "light_rays", "shadow_rays", "stack_overflows"):
            assert a[k] == b[k], k
        assert (a["trace_launches"] == 1) == (w * h * 4 <= 1 << 18)


@pytest.mark.parametrize("chunk", [0, 1 << 18])
def test_refused_however_few_samples(pkg, wl, chunk):
    """Samples x connections per vertex past 32 bits are refused, on the tile launch of small renders as in rounds."""
    _, s, cam = _scene(pkg, wl, 512, 512)
    for vertices, refused in ((1 << 14, True), (64, False)):
        r = pkg.Renderer(pkg.default_params(samples_per_pixel=1, camera_bounces=2, light_bounces=vertices - 1, max_path_length=vertices))
        r.set_scene(s)
        if chunk:
            r.set_tuning(chunk_samples=chunk)
        if refused:
            with pytest.raises(RuntimeError, match="too many samples per pixel"):
                r.render(cam)
        else:
            r.render(cam)


@pytest.mark.parametrize("size,spp,tiles", [((8, 8), 64, True), ((8, 8), 65, False), ((1, 1), 64, True), ((1, 1), 4096, False),
                                            ((64, 64), 64, True), ((4, 4), 3000, False), ((512, 512), 1, True), ((513, 512), 1, False)])
def test_many_samples_on_few_pixels(pkg, wl, size, spp, tiles):
    """The tile launch takes a pixel's samples 64 at a time in one wave, so it
    is for up to 64 samples a pixel (and 2^18 in all); either way the film is
    the per-sample schedule's."""
    desc, s, cam = _scene(pkg, wl, *size)
    params = dict(samples_per_pixel=spp, camera_bounces=4, light_bounces=2, max_path_length=5, seed=5)
    r, q = pkg.Renderer(pkg.default_params(**params)), pkg.Renderer(pkg.default_params(**params))
    q.set_schedule(pkg.SCHEDULE_PER_SAMPLE)
    for x in (r, q):
        x.set_scene(s)
    assert np.array_equal(r.render(cam), q.render(cam))
    assert (r.stats()["trace_launches"] == 1) == tiles
