"""Ray queues at the edges of the traversal's rows against the binary traversal: one ray,
row lengths that change (multiples of the 1024 waves the rows are spread over), the first
queues with full rows, more rays than one row of every wave, inactive rays in between. On
256 compute units with 6 workgroups of 4 waves, one row of every wave is 393,216 rays; with
four of them or more a wave is dealt a second row before it asks for others, which takes
1,572,864 active rays: the last size has about 1,967,000."""
import numpy as np
import pytest

import pbrtm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2049, 65535, 65537, 400_003, 1_200_001, 2_458_765])
def test_row_edges(ctx, n):
    print(f"{n} rays", flush=True)
    bvh = ctx.build(pbrtm.gen_soup(5000, seed=31, mu=-3.0))
    rng = np.random.default_rng(n)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-0.3, 1.3, (n, 3))
    rays[:, 4:7] = rng.normal(size=(n, 3))
    rays[:, 3] = np.where(rng.random(n) < 0.2, 0.0, np.inf)
    rays[0, 3] = np.inf
    for any_hit in (False, True):
        got = bvh.intersect(rays, any_hit=any_hit)
        want = bvh.intersect(rays, any_hit=any_hit, binary=True)
        for g, w in zip(got, want):
            assert np.array_equal(g.view(np.uint32), w.view(np.uint32))
    bvh.free()


@pytest.mark.parametrize("integrator", ["path", "megakernelpath", "ambientocclusion", "surfacenormal"])
@pytest.mark.parametrize("pool", [1, 255, 257, 5000])
def test_pool_sizes(ctx, pool, integrator):
    """Film of a pool that refills many times, in ragged workgroups, against one that never does
    (the megakernel integrators add samples in sample order, one sample per pixel has no order)."""
    from pbrtm import scenes

    w, h = (9, 7) if pool == 1 else (53, 37)
    print(f"{integrator} pool {pool}", flush=True)
    scene = ctx.scene(scenes.cornell34(w, h))
    a, aux, st = scene.render(spp=1, max_depth=4, pool_size=pool, integrator=integrator)
    b, bux, _ = scene.render(spp=1, max_depth=4, integrator=integrator)
    assert st["paths"] == w * h and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.array_equal(aux.view(np.uint32), bux.view(np.uint32))
    scene.free()


@pytest.mark.parametrize("spp,pool", [(9, 0), (9, 700), (16, 1), (49, 300), (64, 0), (64, 97), (81, 300)])
def test_film_order(ctx, spp, pool):
    """Film sums in (round, sample) order on both sides of the per-lane film's sample limit, with
    pools that finish a pixel's samples in and out of order, against the oracle."""
    import oracle as O
    from pbrtm import scenes

    w, h = (5, 3) if pool == 1 else (13, 7)
    print(f"{spp} spp, pool {pool}", flush=True)
    sc = scenes.cornell34(w, h, spp=spp, max_depth=6)
    scene = ctx.scene(sc)
    rgb, aux, _ = scene.render(spp=spp, max_depth=6, pool_size=pool)
    orgb, oaux, _ = O.render(sc, threads=8, pool_size=pool) if pool else O.render(sc, threads=8)
    assert np.array_equal(rgb.view(np.uint32), orgb.view(np.uint32))
    assert np.array_equal(aux.view(np.uint32), oaux.view(np.uint32))
    scene.free()


@pytest.mark.parametrize("n", [360_000, 1_210_000])
def test_cheap_rays_do_not_wait_for_each_other(ctx, n):
    """Rays past a single triangle, a node each: the call is a few launches and the queue's
    traffic (the binary traversal, without a queue, takes 29 and 40 us, this one 42 and 71; 102
    and 260 us when all waves asked one counter for their rows)."""
    import time

    from test_zz_no_alloc import DeviceArray

    bvh = ctx.build(np.array([[[0.4, 0.4, 0], [0.6, 0.4, 0], [0.5, 0.6, 0]]], np.float32))
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:2] = np.random.default_rng(1).uniform(size=(n, 2))
    rays[:, 2], rays[:, 3], rays[:, 6] = 1.0, np.inf, -1.0
    dev, prim, took = DeviceArray(rays.shape, np.float32, rays), DeviceArray((n,), np.uint32), {}
    for binary in (False, True):
        times = []
        for _ in range(40):
            t0 = time.perf_counter()
            bvh.intersect(dev, device_ptrs=True, prim=prim, binary=binary)
            times.append(time.perf_counter() - t0)
        took[binary] = float(np.median(times[10:]))
    print(f"{n} rays: {took[False] * 1e6:.0f} us, binary {took[True] * 1e6:.0f} us", flush=True)
    dev.free()
    prim.free()
    bvh.free()
    assert took[False] <= 2.5 * took[True]
