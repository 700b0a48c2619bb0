"""The one-box volume tracker against the general volume kernels: a launch
with ``samples_per_thread`` > 0 takes the general kernels, and both trace the
same samples. Images differ only by the order in which a pixel's samples are
added (at most 64 float32 additions, each rounding to 2^-24 of the sum), the
gradients by the order of the scatter-adds and the scatter log's fixed point.
A path whose decisions differed would move a pixel by 1e-2 of it."""
import numpy as np
import pytest
import torch

import recursive_control_variates_amd as rcv
from conftest import announce
from recursive_control_variates_amd.transform import T

pytestmark = pytest.mark.gpu

SIGMA = "box.interior_medium.sigma_t.data"
ALBEDO = "box.interior_medium.albedo.data"

# (name, (nz, ny, nx), albedo grid, supergrid factor, shape and medium
# transforms, integrator properties, spp, samples per thread)
UNIT = (T.translate([0.5, 0.5, 0.5]).scale(0.5), T.scale(1.0))
ODD = (T.translate([0.4, 0.55, 0.5]).rotate([0.2, 1.0, 0.3], 25).scale([0.45, 0.3, 0.5]),
       T.translate([-0.3, -0.1, -0.2]).scale([1.3, 1.2, 1.5]))
INNER = (T.translate([0.5, 0.5, 0.5]).scale(0.5), T.translate([0.2, 0.25, 0.1]).scale([0.6, 0.5, 0.7]))
CASES = [
    ("unit", (16, 16, 16), False, 0, UNIT, dict(max_depth=8, rr_depth=8), 16, 4),
    ("ragged", (7, 13, 5), False, 0, UNIT, dict(max_depth=6, rr_depth=2), 9, 9),
    ("narrow", (3, 1, 2), False, 0, UNIT, dict(max_depth=5, rr_depth=5, hide_emitters=True), 8, 2),
    ("rotated", (12, 10, 9), False, 0, ODD, dict(max_depth=8, rr_depth=4), 12, 3),
    ("inner", (9, 8, 10), True, 0, INNER, dict(max_depth=7, rr_depth=7), 8, 8),
    ("albedo", (10, 11, 12), True, 0, UNIT, dict(max_depth=9, rr_depth=3), 16, 16),
    ("supergrid", (17, 16, 15), False, 4, UNIT, dict(max_depth=8, rr_depth=8), 16, 4),
    ("supergrid albedo", (9, 17, 12), True, 8, ODD, dict(max_depth=8, rr_depth=8), 8, 8),
    ("deep", (8, 8, 8), False, 0, UNIT, dict(max_depth=64, rr_depth=64), 4, 1),
    ("unbounded", (8, 8, 8), False, 0, UNIT, dict(max_depth=-1, rr_depth=5), 8, 4),
    # sigma_t = majorant everywhere: every shadow ray ends at its first collision
    ("uniform", (8, 8, 8), False, 0, UNIT, dict(max_depth=8, rr_depth=8), 8, 4),
    ("single scattering", (8, 8, 8), False, 0, UNIT, dict(max_depth=1, rr_depth=5), 8, 4),
]


def _scene(case, w=37, h=23):
    name, n, albedo_grid, factor, (shape_tf, grid_tf), props, spp, spt = case
    scale = {"deep": 40.0, "uniform": 20.0}.get(name, 8.0)
    rng = np.random.default_rng(sum(map(ord, name)))
    grid = rng.uniform(0.0, 1.0, n + (1,)).astype(np.float32)
    if name == "uniform":
        grid[:] = 0.1
    albedo = ({"type": "gridvolume", "data": rng.uniform(0.3, 0.95, n + (3,)).astype(np.float32), "to_world": grid_tf}
              if albedo_grid else {"type": "rgb", "value": (0.9, 0.97, 0.8) if name != "deep" else (0.99, 1.0, 0.98)})
    medium = {"type": "heterogeneous", "sigma_t": {"type": "gridvolume", "data": grid, "to_world": grid_tf},
              "albedo": albedo, "scale": scale, "majorant_resolution_factor": factor}
    sc = rcv.load_dict({
        "type": "scene",
        "box": {"type": "cube", "bsdf": {"type": "null"}, "to_world": shape_tf,
                "interior": {"type": "twostatemedium", "old": medium, "new": medium, "incoming": medium}},
        "env": {"type": "constant", "radiance": {"type": "rgb", "value": (1.0, 0.7, 1.4)}},
        "sensor": {"type": "perspective", "fov": 35.0,
                   "to_world": T.look_at(origin=[0.6, 0.8, 2.8], target=[0.5, 0.5, 0.5], up=[0, 1, 0]),
                   "film": {"type": "hdrfilm", "width": w, "height": h, "rfilter": {"type": "box"}},
                   "sampler": {"type": "independent", "sample_count": spp}}})
    p = rcv.traverse(sc)
    for key in [SIGMA] + ([ALBEDO] if albedo_grid else []):
        x = p[key].detach()
        new = x.clone() if name == "uniform" else (x * torch.from_numpy(rng.uniform(0.9, 1.05, x.shape).astype(np.float32)).cuda()).clamp(max=1.0)
        p[key] = new.requires_grad_(True)
    p.update()
    gimg = torch.from_numpy(rng.uniform(-0.5, 1.5, (h, w, 3)).astype(np.float32)).cuda()
    gimg[3:5] = 0.0
    tangents = {k: torch.from_numpy(rng.uniform(-1, 1, tuple(t.shape)).astype(np.float32)).cuda()
                for k, t in p.differentiable()}
    integ = rcv.load_dict(dict(props, type="twostateprbvolpath"))
    return sc, p, integ, gimg, tangents, spp, spt


@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0])
def test_box_tracker_equals_general_kernels(cuda, case):
    announce(f"one-box tracker vs general kernels ({case[0]})")
    sc, p, integ, gimg, tangents, spp, spt = _scene(case)
    out = []
    for s in (0, spt):
        integ.samples_per_thread = s
        plain = integ.render(sc, 0, 11, spp)
        old, new = integ.render_twostates(sc, 0, 12, spp)
        fwd = integ.render_forward(sc, p, 0, 13, spp, tangents=tangents)
        grads = integ.adjoint(sc, p, gimg, 0, 14, spp)
        out.append(([x.double().cpu().numpy() for x in (plain, old, new)], fwd.double().cpu().numpy(),
                    {k: g.double().cpu().numpy() for k, g in grads.items()}))
    (imgs, fwd, grads), (imgs0, fwd0, grads0) = out
    for a, b in zip(imgs, imgs0):
        assert np.abs(b).max() > 0 or case[5].get("hide_emitters")
        np.testing.assert_allclose(a, b, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(fwd, fwd0, rtol=1e-4, atol=1e-5 * max(np.abs(fwd0).max(), 1e-6))
    for k in grads0:
        scale = np.abs(grads0[k]).max()
        assert scale > 0, k
        assert np.allclose(grads[k], grads0[k], rtol=1e-4, atol=1e-5 * scale), (k, np.abs(grads[k] - grads0[k]).max())


def test_box_tracker_empty_and_masked(cuda):
    # a medium of zero density scatters nothing; an image gradient of zeros
    # has no work for the adjoint
    announce("one-box tracker: zero density, zero image gradient")
    sc, p, integ, gimg, _, spp, spt = _scene(CASES[0])
    img = integ.render(sc, 0, 3, spp)
    g = integ.adjoint(sc, p, torch.zeros_like(gimg), 0, 4, spp)[SIGMA]
    assert float(g.abs().max()) == 0.0 and float(img.max()) > 0
    p[SIGMA] = torch.zeros_like(p[SIGMA].detach())
    p.update()
    p.update()
    img = integ.render(sc, 0, 3, spp)
    env = torch.tensor([1.0, 0.7, 1.4], device="cuda")
    np.testing.assert_allclose(img.cpu().numpy(), env.expand_as(img).cpu().numpy(), rtol=1e-5)


@pytest.mark.parametrize("many_pixels", [False, True])
def test_batched_box_jobs_equal_single_launches(cuda, monkeypatch, many_pixels):
    # first iteration of a batch of every feature mask (old = new = initial
    # value), one job plain: images and gradients of the single launches with
    # the same seeds; with many pixels the renders' units are whole pixels
    from recursive_control_variates_amd.batch import BatchOptimizer, JobSpec
    from recursive_control_variates_amd.rendering import sample_tea_32
    announce(f"batched one-box jobs vs single launches (many_pixels={many_pixels})")
    w, h = (760, 240) if many_pixels else (37, 23)
    specs, want = [], []
    for i, k in enumerate([0, 3, 4, 6, 7]):
        sc, p, integ, _, _, spp, _ = _scene(CASES[k], w, h)
        init = p[SIGMA].detach().clone()
        for _ in range(2):
            for key in p.keys():
                p[key] = p[key].detach().clone().requires_grad_(key == SIGMA)
            p.update()
        seed = 100 + i
        img = (integ.render(sc, 0, seed, spp) if i == 1 else integ.render_twostates(sc, 0, seed, spp)[1])
        ref = torch.full_like(img, 0.4)
        g = integ.adjoint(sc, p, 2.0 * (img - ref) / img.numel(), 0, sample_tea_32(seed, 1)[0], spp)[SIGMA]
        want.append((img.cpu().numpy(), g.cpu().numpy()))
        specs.append(JobSpec(scene=sc, key=SIGMA, init=init, img_ref=ref, method="baseline" if i == 1 else "cv_ps",
                             integrator=dict(CASES[k][5], type="twostateprbvolpath"), loss="L2", spp=spp, seed=seed))
    batch = BatchOptimizer(specs, use_graph=False)
    batch.step(1)
    batch.synchronize()
    for j, (img, g) in enumerate(want):
        np.testing.assert_allclose(batch.image(j).cpu().numpy(), img, rtol=1e-5, atol=1e-6)
        got = batch.jobs[j].grad.cpu().numpy()
        assert np.allclose(got, g, rtol=1e-4, atol=1e-5 * np.abs(g).max()), (j, np.abs(got - g).max())
    batch.close()
