"""Albedo derivatives of scenes with more than one kind of material, against the oracle's
FP64 replay: conductors and dielectrics among the diffuse materials (their rows are zero, and
the replay orders its slots by material), black albedos, and grey ones, whose columns of the
RGB-to-spectrum table no scene set-up computes: the first gradient here finds them missing on
the device, unless a test before this file filled them, and the host adds them."""
import numpy as np
import pytest

import oracle as O
import pbrtm
import scenes
from test_gpu_grad import close, log

pytestmark = pytest.mark.gpu


def mixed_scene(seed):
    """cornell_emitters with every third albedo grey, two black, and a conductor, a rough
    conductor, a dielectric and a rough dielectric."""
    sc = scenes.cornell_emitters(32, 32, spp=16, max_depth=5)
    alb = np.random.default_rng(seed).uniform(0.1, 0.9, sc["albedo"].shape).astype(np.float32)
    alb[::3] = alb[::3, :1]
    alb[[4, 11]] = 0.0
    mats = [{"type": "diffuse", "rgb": tuple(float(v) for v in a)} for a in alb]
    mats[7] = {"type": "conductor", "metal": "Cu", "roughness": 0.0, "remap": False}
    mats[13] = {"type": "conductor", "metal": "Al", "roughness": 0.2, "remap": True}
    mats[23] = {"type": "dielectric", "eta": 1.5, "roughness": 0.0}
    mats[28] = {"type": "dielectric", "eta": "glass-BK7", "roughness": 0.3}
    sc.update(materials=mats)
    return sc, alb


def brighter(sc):
    mats = [dict(m, rgb=tuple(min(0.99, 1.07 * v + 0.01) for v in m["rgb"])) if m["type"] == "diffuse" else m
            for m in sc["materials"]]
    return dict(sc, materials=mats)


@pytest.mark.parametrize("pool", [0, 777])
def test_mixed_materials(ctx, pool):
    sc, alb = mixed_scene(5 + pool)
    target, _, _ = O.render(brighter(sc), threads=16)
    kw = {"pool_size": pool} if pool else {}
    loss_o, d_rgb_o, d_scale_o, film_o = O.render_grad(sc, target, threads=16, **kw)
    log(f"pool {pool}: oracle done")
    s = ctx.scene(sc)
    try:
        loss, d_alb, d_sc, film, _ = s.render_grad(target, spp=sc["spp"], max_depth=sc["max_depth"], **kw)
        _, again, _, _, _ = s.render_grad(target, spp=sc["spp"], max_depth=sc["max_depth"], **kw)
    finally:
        s.free()
    assert np.array_equal(film.view(np.uint32), film_o.view(np.uint32))
    assert abs(loss - loss_o) <= 1e-9 * loss_o
    assert np.isfinite(d_alb).all()
    zero = [m for m, mat in enumerate(sc["materials"]) if mat["type"] != "diffuse"] + [4, 11]
    assert (d_alb[zero] == 0).all() and (again[zero] == 0).all()
    grey = np.arange(0, len(alb), 3)
    assert np.count_nonzero(d_alb[grey]) > len(grey)
    close(d_alb, d_rgb_o, 2e-3, "d_albedo")
    close(again, d_rgb_o, 2e-3, "d_albedo again")
    close(d_sc, d_scale_o, 2e-3, "d_scale")
