"""Closest and any hits of unusual rays against the binary traversal (the reference's
order, node by node) and the CPU oracle, bit for bit.

The traversal's box test is conservative arithmetic around a clamped reciprocal
direction, with the reference's own slab test for rays outside its range: rays along
an axis, inside a plane that holds vertices, with tiny or huge components, from far
away, without a direction or with NaNs have to find the hits of the reference's order.
"""
import numpy as np
import pytest

import oracle as O
import pbrtm

pytestmark = pytest.mark.gpu

SCENES = {
    "soup": lambda: pbrtm.gen_soup(4000, seed=21, mu=-3.0),
    # an axis-aligned grid of quads: flat boxes, vertices shared by planes and rays
    "grid": lambda: _grid(),
    # small triangles far from the origin: planes known to few bits
    "offset": lambda: (pbrtm.gen_soup(4000, seed=22, mu=-3.0) + np.float32(4096.0)).astype(np.float32),
    "leaf": lambda: pbrtm.gen_soup(1, seed=23, mu=-1.0),
}


def _grid():
    tris = []
    k = np.linspace(0, 1, 9)
    for a in range(3):
        for x in (0.0, 0.5, 1.0):
            for i in range(8):
                for j in range(8):
                    q = np.array([[x, k[i], k[j]], [x, k[i + 1], k[j]], [x, k[i + 1], k[j + 1]], [x, k[i], k[j + 1]]])
                    q = np.roll(q, a, axis=1)
                    tris += [q[[0, 1, 2]], q[[0, 2, 3]]]
    return np.array(tris, np.float32)


def _rays(form, tri, n, rng):
    lo, hi = tri.min(axis=(0, 1)).astype(np.float64), tri.max(axis=(0, 1)).astype(np.float64)
    span = hi - lo
    o = lo + rng.uniform(-0.5, 1.5, (n, 3)) * span
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    t_max = np.full(n, np.inf)
    vert = tri.reshape(-1, 3)[rng.integers(0, 3 * len(tri), n)].astype(np.float64)
    axis = rng.integers(0, 3, n)
    rows = np.arange(n)
    if form == "axis":  # along +-x, y, z with signed zeros, half of them through vertex coordinates
        d = np.where(rng.random((n, 3)) < 0.5, -0.0, 0.0)
        d[rows, axis] = rng.choice([-1.0, 1.0], n)
        o[::2] = vert[::2]
        o[rows, axis] = np.where(d[rows, axis] > 0, lo.min() - 1, hi.max() + 1)
    elif form == "plane":  # one zero component, inside the plane of a vertex
        d[rows, axis] = np.where(rng.random(n) < 0.5, -0.0, 0.0)
        o[rows, axis] = vert[rows, axis]
    elif form == "tiny":  # components whose reciprocal is huge, denormal or overflows
        d[rows, axis] = rng.choice([1e-12, -1e-25, 1e-30, -1e-38, 1e-42], n)
        o[::2, :] = vert[::2]
    elif form == "scaled":  # unnormalised directions
        d *= 10.0 ** rng.uniform(-12, 12, (n, 1))
    elif form == "far":  # far origins, aimed at a vertex
        o = vert + d * 10.0 ** rng.uniform(1, 6, (n, 1))
        d = vert - o
    elif form == "vertex":  # at shared vertices and edges: ties
        o = vert + d * span.max()
        d = vert - o
    elif form == "short":  # a finite interval
        t_max = rng.uniform(0.01, 0.7, n)
    elif form == "none":  # no direction, or NaN, or infinite
        bad = rng.integers(0, 4, n)
        d[bad == 0] = 0.0
        d[bad == 1, 0] = np.nan
        d[bad == 2, 1] = np.nan
        d[bad == 3, 2] = np.inf
    rays = np.zeros((n, 8), np.float32)
    with np.errstate(over="ignore", under="ignore"):
        rays[:, 0:3] = o
        rays[:, 3] = t_max
        rays[:, 4:7] = d
    return rays


def _same(a, b):
    """Bit equality, any NaN for any NaN."""
    return bool(((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all())


@pytest.mark.parametrize("form", ["axis", "plane", "tiny", "scaled", "far", "vertex", "short", "none"])
@pytest.mark.parametrize("scene", sorted(SCENES))
def test_ray_forms(ctx, scene, form):
    tri = SCENES[scene]()
    bvh, ref = ctx.build(tri), O.OracleBvh(tri)
    rng = np.random.default_rng(len(form) * 31 + len(scene))
    for n in (3, 4001):
        rays = _rays(form, tri, n, rng)
        print(f"{scene} {form} {n} rays", flush=True)
        for any_hit in (False, True):
            prim, t, bary = bvh.intersect(rays, any_hit=any_hit)
            wants = [bvh.intersect(rays, any_hit=any_hit, binary=True)]
            if scene != "grid":  # coplanar faces tie, and the oracle's order inside a leaf is its own
                wants.append(ref.intersect(rays, any_hit=any_hit)[:3])
            for op, ot, ob in wants:
                assert np.array_equal(prim, op), (any_hit, int((prim != op).sum()))
                if not any_hit:
                    hit = op != pbrtm.NO_HIT
                    assert _same(t[hit], ot[hit])
                    assert _same(bary[hit], ob[hit])
    bvh.free()


@pytest.mark.parametrize("form", ["axis", "tiny", "far", "none"])
def test_ray_forms_noalloc(ctx, form):
    """The same rays through the entry point without allocation."""
    from test_zz_no_alloc import DeviceArray

    tri = SCENES["grid"]()
    bvh = ctx.build(tri)
    n = 4001
    rays = _rays(form, tri, n, np.random.default_rng(len(form)))
    print(f"noalloc {form}", flush=True)
    dev = DeviceArray(rays.shape, np.float32, rays)
    out = [DeviceArray((n,), np.uint32), DeviceArray((n,), np.float32), DeviceArray((n, 3), np.float32)]
    for any_hit in (False, True):
        bvh.intersect_noalloc(dev, *out, any_hit=any_hit)
        prim, t, bary = (a.numpy() for a in out)
        op, ot, ob = bvh.intersect(rays, any_hit=any_hit, binary=True)
        assert np.array_equal(prim, op)
        if not any_hit:
            hit = op != pbrtm.NO_HIT
            assert _same(t[hit], ot[hit]) and _same(bary[hit], ob[hit])
    for a in (dev, *out):
        a.free()
    bvh.free()


def test_short_directions_take_as_long_as_others(ctx):
    """Rays on both sides of the range of the conservative box test (directions shorter than
    2^-20 take the reference's own test): a queue of them takes at most twice the time."""
    import time

    from test_zz_no_alloc import DeviceArray

    n = 230_400
    bvh = ctx.build(pbrtm.gen_soup(1_000_000, seed=41))
    rng = np.random.default_rng(41)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    prim, took = DeviceArray((n,), np.uint32), {}
    for length in (2.0 ** -18, 2.0 ** -24):
        rays = np.zeros((n, 8), np.float32)
        rays[:, 0:3] = np.random.default_rng(42).uniform(size=(n, 3))
        rays[:, 3] = np.inf
        rays[:, 4:7] = d * length
        dev, times = DeviceArray(rays.shape, np.float32, rays), []
        for _ in range(12):
            t0 = time.perf_counter()
            bvh.intersect(dev, device_ptrs=True, prim=prim)
            times.append(time.perf_counter() - t0)
        took[length] = float(np.median(times[2:]))
        print(f"directions of length {length:.3g}: {took[length] * 1e6:.0f} us", flush=True)
        dev.free()
    prim.free()
    bvh.free()
    assert took[2.0 ** -24] <= 2 * took[2.0 ** -18], took


@pytest.mark.parametrize("form,scale,offset", [
    ("axis", 2.0 ** -30, 0), ("axis", 2.0 ** 40, 0), ("axis", 1, 4096), ("short", 2.0 ** -30, 0),
    ("short", 2.0 ** 40, 0), ("short", 1, 4096), ("short", 1, 16384)])
def test_work_does_not_depend_on_the_scene_s_place(ctx, form, scale, offset):
    """The same rays into the same triangles, scaled or moved: a ray visits as many nodes and
    tests as many triangles. (In small and large scenes rays along an axis once entered every
    box, far from the world's origin all rays the boxes around their own.)"""
    base = pbrtm.gen_soup(100_000, seed=51, mu=-5.0)
    counts = []
    for s, o in ((1.0, 0.0), (scale, offset)):
        tri = (base.astype(np.float64) * s + o).astype(np.float32)
        bvh = ctx.build(tri)
        rays = _rays(form, base, 2000, np.random.default_rng(52))
        rays[:, 0:3] = (rays[:, 0:3].astype(np.float64) * s + o).astype(np.float32)
        rays[:, 3] *= np.float32(s)
        stats = np.zeros(3, np.uint64)
        bvh.intersect(rays, stats=stats)
        counts.append(stats[[0, 2]] / len(rays))
        bvh.free()
    print(f"{form} scale {scale} offset {offset}: visits and tests per ray {counts[0]} -> {counts[1]}", flush=True)
    assert counts[1][0] <= 1.1 * counts[0][0] and counts[1][1] <= 1.3 * counts[0][1]


@pytest.mark.parametrize("distance", [20.0, 2000.0, 40000.0])
def test_work_from_far_away(ctx, distance):
    """Rays into 200,000 triangles from `distance` extents away find the hits of the reference's
    order and test about as many triangles. (An allowance that grows with the distance once
    had them test seven times as many at 30,000 extents.)"""
    tri = pbrtm.gen_soup(200_000, seed=61, mu=-5.0)
    lo, hi = tri.min(axis=(0, 1)).astype(np.float64), tri.max(axis=(0, 1)).astype(np.float64)
    rng = np.random.default_rng(62)
    eye = (lo + hi) / 2 + distance * (hi - lo).max() * np.array([0.3, 0.5, -0.81])
    d = rng.uniform(lo, hi, (4000, 3)) - eye
    rays = np.zeros((4000, 8), np.float32)
    rays[:, 0:3], rays[:, 3] = eye, np.inf
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    bvh = ctx.build(tri)
    tests, out = [], []
    for binary in (True, False):
        stats = np.zeros(3, np.uint64)
        out.append(bvh.intersect(rays, stats=stats, binary=binary))
        tests.append(stats[2] / len(rays))
    bvh.free()
    print(f"distance {distance}: tests per ray {tests[0]:.1f} binary, {tests[1]:.1f} wide", flush=True)
    assert np.array_equal(out[0][0], out[1][0]) and _same(out[0][1], out[1][1]) and _same(out[0][2], out[1][2])
    assert tests[1] <= 1.5 * tests[0]
