"""The traversal's own code (path_device.h) on the CPU, one lane at a time,
under AddressSanitizer (tests/hostsim/trav_host.cpp): rays whose box test
culls on no axis -- non-finite, tiny, into flattened instances -- must neither
leave the node and instance arrays nor hit anything that a loop over all
triangles does not, and ordinary rays must hit what that loop hits."""
import os
import pathlib
import re
import shutil
import struct
import subprocess

import numpy as np
import pytest

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE.parent / "openmaterial-validation_amd" / "csrc"
CLANG = "/opt/rocm/llvm/bin/clang++"
FAR = np.float32(np.finfo(np.float32).max)


@pytest.fixture(scope="module")
def trav(tmp_path_factory):
    if not os.path.exists(CLANG) or not shutil.which("g++"):
        pytest.skip("clang++ or g++ is missing")
    out = tmp_path_factory.mktemp("trav")
    # device assembly -> C++: the two comparators of the child sort; the empty
    # statements (optimiser barriers) go
    src = (CSRC / "path_device.h").read_text()
    src, n = re.subn(r'asm\("v_(min|max)_f64[^;]*;',
                     r"double da, db; __builtin_memcpy(&da, &a, 8); __builtin_memcpy(&db, &b, 8); da = \1F64(da, db); "
                     r"__builtin_memcpy(&r, &da, 8);", src)
    assert n == 2
    src = re.sub(r'asm (?:volatile)?\(""[^;]*;|asm\(""[^;]*;', ";", src)
    src = src.replace('"../../include/omv.h"', f'"{HERE.parent / "include" / "omv.h"}"')
    (out / "path_device_host.h").write_text(src)
    subprocess.run([CLANG, "-std=c++17", "-O1", "-g", "-ffp-contract=off", "-mfma", "-fsanitize=address", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{CSRC}", f'-DPATH_DEVICE="{out / "path_device_host.h"}"',
                    str(HERE / "hostsim" / "trav_host.cpp"), str(CSRC / "bvh.cpp"), "-o", str(out / "trav")], check=True)

    def run(meshes, insts, rays):
        """(hit instance, primitive, t bits, node visits, the loop's instance, primitive, t bits) per ray."""
        msg = [struct.pack("i", len(meshes))]
        for v, f in meshes:
            msg += [struct.pack("ii", len(v), len(f)), np.ascontiguousarray(v, np.float32).tobytes(), np.ascontiguousarray(f, np.int32).tobytes()]
        msg.append(struct.pack("i", len(insts)))
        for m, mesh in insts:
            msg += [struct.pack("i", mesh), np.ascontiguousarray(m[:3], np.float32).tobytes(), inverse(m).tobytes()]
        msg += [struct.pack("i", len(rays)), np.ascontiguousarray(rays, np.float32).tobytes()]
        r = subprocess.run([str(out / "trav")], input=b"".join(msg), capture_output=True, timeout=120)
        assert r.returncode == 0, r.stderr.decode()[-3000:]
        return np.array([line.split() for line in r.stdout.decode().splitlines()], np.int64)

    return run


def inverse(m):
    """World to object, as the scene makes it: double, rounded; inf and NaN where m is singular."""
    with np.errstate(all="ignore"):
        a, b, c, _, d, e, f, _, g, h, i, _ = np.asarray(m[:3], np.float32).astype(np.float64).ravel()
        t = np.asarray(m[:3, 3], np.float32).astype(np.float64)
        A, B, C = e * i - f * h, -(d * i - f * g), d * h - e * g
        r = np.float64(1.0) / (a * A + b * B + c * C)
        n = np.array([[A * r, -(b * i - c * h) * r, (b * f - c * e) * r], [B * r, (a * i - c * g) * r, -(a * f - c * d) * r],
                      [C * r, -(a * h - b * g) * r, (a * e - b * d) * r]])
        return np.concatenate([n, -(n @ t)[:, None]], 1).astype(np.float32)


def turned(rng, scale, shift):
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    m = np.eye(4)
    m[:3, :3] = q * np.asarray(scale, np.float64)
    m[:3, 3] = shift
    return m


def scene(wl, rng, extra=()):
    v, f = wl.icosphere(2, 0.7)
    tri = np.array([[-0.6, -0.4, 0.1], [0.7, -0.3, -0.2], [0.05, 0.65, 0.15]], np.float32)
    insts = [(turned(rng, (1, 1, 1), rng.uniform(-2, 2, 3)), k % 2) for k in range(7)]
    return [(v, f), (tri, np.array([[0, 1, 2]]))], insts + list(extra)


def rays(rng, n=400):
    o = rng.uniform(-4, 4, (n, 3))
    d = rng.uniform(-2, 2, (n, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, d, np.zeros((n, 1)), np.full((n, 1), FAR)], 1).astype(np.float32)


def check(got, hits=None):
    assert np.array_equal(got[:, :3], got[:, 4:])
    if hits is not None:
        assert hits[0] <= (got[:, 0] >= 0).mean() <= hits[1]


def test_ordinary_rays(trav, wl):
    rng = np.random.default_rng(1)
    check(trav(*scene(wl, rng), rays(rng)), (0.1, 1.0))


@pytest.mark.parametrize("flat", [(1, 1, 0), (1, 0, 1), (0, 1, 1), (0, 0, 1), (0, 0, 0)])
@pytest.mark.parametrize("mesh", [0, 1])
def test_flattened_instances(trav, wl, flat, mesh):
    """A singular matrix has an inverse of inf and NaN rows: the object ray culls on no axis."""
    rng = np.random.default_rng(2)
    extra = [(turned(rng, flat, rng.uniform(-1, 1, 3)), mesh) for _ in range(6)]
    check(trav(*scene(wl, rng, extra), rays(rng)), (0.1, 1.0))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("axes", [(0,), (1, 2), (0, 1, 2)])
def test_non_finite_rays_and_places(trav, wl, value, axes):
    rng = np.random.default_rng(3)
    meshes, insts = scene(wl, rng)
    for first in (0, 3):   # the origin's, then the direction's components
        r = rays(rng)
        for a in axes:
            r[:, first + a] = value
        check(trav(meshes, insts, r), (0.0, 0.0))
    r = rays(rng)
    r[:200, 6] = value if value > 0 else np.nan   # the interval's ends
    r[200:, 7] = np.nan
    check(trav(meshes, insts, r), (0.0, 0.0))
    shift = np.zeros(3)
    shift[list(axes)] = value
    check(trav(meshes, insts + [(turned(rng, (1, 1, 1), shift), 0)], rays(rng)), (0.1, 1.0))


@pytest.mark.parametrize("size", [1e-36, 1e-31, 1e-29, 1e29, 1e33, 1e36])
def test_tiny_and_huge_directions(trav, wl, size):
    """Instances scaled so far that every component of the object direction is below or above the slab test's range."""
    rng = np.random.default_rng(4)
    meshes, insts = scene(wl, rng)
    extra = [(turned(rng, (size,) * 3, np.zeros(3)), k % 2) for k in range(3)]
    check(trav(meshes, insts + extra, rays(rng)), (0.1, 1.0))


@pytest.mark.parametrize("zero", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2)])
@pytest.mark.parametrize("place", ["free", "edge", "flat", "far"])
def test_zero_components_cull(trav, wl, zero, place):
    """A ray with components of exactly 0 (either sign) hits what it has to,
    on the very edge of boxes too, and visits no more than a ray that is
    turned away from the axis by 1e-4."""
    rng = np.random.default_rng(5)
    v, f = wl.icosphere(4, 0.7)
    n, q = 400, 24
    g = np.linspace(-1, 1, q, dtype=np.float32)
    plate = np.stack(np.meshgrid(g, np.zeros(1, np.float32), g, indexing="ij"), -1).reshape(-1, 3)
    i = (np.arange(q - 1)[:, None] * q + np.arange(q - 1)).ravel()
    pf = np.concatenate([np.stack([i, i + 1, i + q], 1), np.stack([i + 1, i + q + 1, i + q], 1)])
    meshes, m = [(v, f), (plate, pf)], np.eye(4)
    m[:3, 3] = {"far": (7e4, -2e4, 3e3)}.get(place, (0, 0, 0))
    target = rng.uniform(-0.6, 0.6, (n, 3))
    if place == "edge":
        target = np.where(rng.random((n, 3)) < 0.5, 0.7 * rng.choice([-1, 0, 1], (n, 3)), target)
    d = rng.normal(size=(n, 3))
    d[:, list(zero)] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[: n // 2, list(zero)] = -0.0
    o = np.float32(m[:3, 3]) + (target - 3.0 * d)
    if place == "flat":   # along and beside a plate on y = 0, among its vertices' planes
        o[:, 1] = np.float32(m[1, 3]) + rng.choice([0.0, 1e-7, -1e-7, 1e-30, -1e-40], n)
    r = np.concatenate([o, d, np.zeros((n, 1)), np.full((n, 1), FAR)], 1).astype(np.float32)
    insts = [(m, 1 if place == "flat" else 0)]
    got = trav(meshes, insts, r)
    check(got)
    if place in ("free", "far"):
        assert (got[:, 0] >= 0).mean() > 0.3
        turn = r.copy()
        turn[:, 3:6] += np.where(turn[:, 3:6] == 0, np.float32(1e-4), 0)
        assert got[:, 3].mean() <= 1.2 * trav(meshes, insts, turn)[:, 3].mean() + 2


@pytest.mark.parametrize("away", [0.0, 1e3, 1e5, 1e6])
def test_meshes_far_from_their_origin(trav, wl, away):
    """A mesh moved away in its own coordinates and back by its instance: the
    slab test's slack goes with the size of the mesh, not with the distance,
    so a ray visits hardly more nodes than for the mesh in place."""
    rng = np.random.default_rng(6)
    v, f = wl.icosphere(4, 0.7)
    at = np.float32([away, -0.5 * away, 0.25 * away])
    far = v + at
    m, back = np.eye(4), np.eye(4)
    back[:3, 3] = -at.astype(np.float64)
    r = rays(rng, 300)
    r[:, :3] *= 0.5
    d = -r[:, :3] + rng.uniform(-0.6, 0.6, (len(r), 3))
    r[:, 3:6] = d / np.linalg.norm(d, axis=1, keepdims=True)
    got = trav([(far, f)], [(back, 0)], r)
    check(got, (0.3, 1.0))
    # the mesh that rounding has made of it, in place
    near = trav([(far - at, f)], [(m, 0)], r)
    assert got[:, 3].mean() <= 1.2 * near[:, 3].mean() + 1
