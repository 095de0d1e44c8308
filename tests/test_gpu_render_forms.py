"""Unusual rays in the traversal's instances that only renders reach, against the oracle, bit for
bit: the one with analytic primitives (which fetches the ray's direction again for them) and the
one with a tree per ray (a batch), through cameras that are far away, or whose field of view is
so narrow that the primary rays' other two components are tiny, aimed at walls, a mirror, a
sphere and an edge of boxes."""
import numpy as np
import pytest

import oracle as O
import scenes

pytestmark = pytest.mark.gpu

VIEWS = {  # eye, look, field of view in degrees
    "mirror": ((278.0, 273.0, -800.0), (278.0, 273.0, 0.0), 1e-12),
    "far": ((278.0, 273.0, -8e5), (278.0, 273.0, 0.0), 0.03),
    "wall": ((420.0, 400.0, -800.0), (420.0, 400.0, 0.0), 1e-12),
    "sphere": ((70.0, 45.0, -800.0), (70.0, 45.0, 0.0), 1e-9),
    "edge": ((290.0, 165.0, -800.0), (290.0, 165.0, 65.0), 1e-5),
    "down": ((300.0, 540.0, 290.0), (300.0, 0.0, 290.0), 1e-12),  # off the light's diagonal: no tie
}
SPP, DEPTH = 4, 5


def view(make, name):
    eye, look, fov = VIEWS[name]
    sc = make(19, 13, spp=SPP, max_depth=DEPTH)
    sc.update(eye=eye, look=look, fov=fov, up=(0.0, 0.0, 1.0) if name == "down" else sc["up"])
    return sc


def same(a, b):
    """Bit equality, any NaN for any NaN."""
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    return bool(((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all())


@pytest.mark.parametrize("name", sorted(VIEWS))
@pytest.mark.parametrize("make", [scenes.cornell34, scenes.shapes_room], ids=["triangles", "shapes"])
def test_views(ctx, make, name):
    sc = view(make, name)
    scene = ctx.scene(sc)
    try:
        for integrator in ("path", "ambientocclusion", "surfacenormal"):
            print(f"{make.__name__} {name} {integrator}", flush=True)
            rgb, aux, st = scene.render(spp=SPP, max_depth=DEPTH, integrator=integrator)
            if integrator == "path":
                orgb, oaux, ost = O.render(sc, threads=16)
                assert (st["rays"], st["shadow_rays"]) == (ost["rays"], ost["shadow_rays"])
            else:
                orgb, oaux, _ = O.render_megakernel(sc, integrator, threads=16)
            assert same(rgb, orgb) and same(aux, oaux), integrator
    finally:
        scene.free()


def test_views_in_a_batch(ctx):
    jobs = [view(make, name) for make in (scenes.cornell34, scenes.shapes_room) for name in sorted(VIEWS)]
    handles = [ctx.scene(sc) for sc in jobs]
    try:
        for part in (slice(0, len(VIEWS)), slice(None)):  # triangles only, then with analytic primitives
            print(f"batch of {len(jobs[part])}", flush=True)
            films, _, _, _ = ctx.render_batch([(h, SPP, DEPTH, 0) for h in handles[part]], pool_size=1500)
            for sc, film in zip(jobs[part], films):
                assert same(film, O.render(sc, threads=16)[0]), (sc["eye"], sc["fov"])
    finally:
        for h in handles:
            h.free()
