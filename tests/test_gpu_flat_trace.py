"""Ray tracing of small scenes over all their primitives (flat_trace) against
the BVH: the same scene with a mesh hidden inside one of its spheres has too
many primitives for it. Both find the same hits, so images are equal; a ray
through an edge to within rounding may take either side in a different BVH
(two of a million), so one pixel may differ."""
import numpy as np
import pytest
import torch

import recursive_control_variates_amd as rcv
from conftest import announce
from helpers import cam
from recursive_control_variates_amd import scenes
from recursive_control_variates_amd.transform import T

pytestmark = pytest.mark.gpu


def _hidden(center, n=40):
    rng = np.random.default_rng(0)
    v = np.asarray(center) + rng.uniform(-0.05, 0.05, (3 * n, 3))
    return {"type": "mesh", "vertices": v.astype(np.float32), "faces": np.arange(3 * n).reshape(n, 3),
            "bsdf": {"type": "diffuse", "reflectance": {"type": "rgb", "value": 0.5}}}


def _tri(pts, albedo):
    return {"type": "mesh", "vertices": np.asarray(pts, np.float32), "faces": np.arange(len(pts)).reshape(-1, 3),
            "bsdf": {"type": "diffuse", "reflectance": {"type": "rgb", "value": albedo}}}


def _mixed(n_single):
    """Floor, light, three spheres, a tetrahedron and single triangles."""
    d = {"type": "scene",
         "floor": {"type": "rectangle", "to_world": T.rotate([1, 0, 0], -90).scale(3.0),
                   "bsdf": {"type": "diffuse", "reflectance": {"type": "bitmap",
                                                                 "data": scenes.texture_target(8, 3)}}},
         "light": {"type": "rectangle", "to_world": T.translate([0.3, 2.5, 0]).rotate([1, 0.2, 0], 80).scale(0.6),
                   "bsdf": {"type": "diffuse", "reflectance": {"type": "rgb", "value": 0.0}},
                   "emitter": {"type": "area", "radiance": {"type": "rgb", "value": 6.0}}},
         "sensor": cam((0.5, 1.2, 4.0), (0, 0.5, 0), fov=45, w=40, h=30, spp=16)}
    for i, c in enumerate([(-0.9, 0.4, 0.1), (0.8, 0.45, -0.6), (0.2, 0.3, 0.9)]):
        d[f"sphere{i}"] = {"type": "sphere", "center": list(c), "radius": 0.3,
                           "bsdf": {"type": "diffuse", "reflectance": {"type": "rgb", "value": 0.6 + 0.1 * i}}}
    a, b, c, e = (-0.2, 0.05, -0.5), (0.4, 0.05, -0.4), (0.1, 0.05, 0.2), (0.1, 0.9, -0.2)
    d["tetra"] = _tri([a, b, e, b, c, e, c, a, e, a, c, b], (0.3, 0.7, 0.5))
    rng = np.random.default_rng(5)
    for k in range(n_single):
        p = rng.uniform([-1.5, 0.2, -1.5], [1.5, 1.6, 0.5])
        d[f"tri{k}"] = _tri([p, p + rng.uniform(-0.4, 0.4, 3), p + rng.uniform(-0.4, 0.4, 3)], 0.4)
    return d


SCENES = {
    "cornell": lambda: (scenes.cornell_scene_dict(scenes.texture_target(16, 2), twostate=False, film_res=40, spp=16),
                        (0.35, -0.7, 0.2), "prb"),
    "triangles": lambda: (_mixed(4), (-0.9, 0.4, 0.1), "prb"),
    "at the limit": lambda: (_mixed(10), (-0.9, 0.4, 0.1), "prb"),
    "past the limit": lambda: (_mixed(11), (-0.9, 0.4, 0.1), "prb"),
    "shadow rays with a range": lambda: (_mixed(4), (-0.9, 0.4, 0.1), "prbvolpath"),
}


@pytest.mark.parametrize("name", list(SCENES))
def test_flat_trace_finds_the_bvh_hits(cuda, name):
    announce(f"flat trace vs BVH ({name})")
    imgs = []
    for hidden in (False, True):
        d, center, kind = SCENES[name]()
        if hidden:
            d["hidden"] = _hidden(center)
        sc = rcv.load_dict(d)
        integ = rcv.load_dict({"type": kind, "max_depth": 6, "rr_depth": 4})
        imgs.append(integ.render(sc, 0, 9, 16).cpu().numpy())
    a, b = imgs
    assert b.max() > 0
    off = (np.abs(a - b) > 1e-5 * np.abs(b) + 1e-6).any(axis=-1).sum()
    assert off <= 1, off


@pytest.mark.parametrize("name", ["cornell", "triangles"])
def test_flat_trace_of_axis_parallel_and_edge_rays(cuda, name):
    # an orthogonal view straight at the scene: no jitter can be asked for, so
    # a tiny field of view makes every ray nearly parallel to the walls
    announce(f"flat trace, nearly axis-parallel rays ({name})")
    imgs = []
    for hidden in (False, True):
        d, center, kind = SCENES[name]()
        d["sensor"] = cam((0.0, 0.5 if name == "triangles" else 0.0, 40.0), (0, 0.5 if name == "triangles" else 0.0, 0),
                          fov=0.01, w=16, h=16, spp=8)
        if hidden:
            d["hidden"] = _hidden(center)
        sc = rcv.load_dict(d)
        imgs.append(rcv.load_dict({"type": kind, "max_depth": 3}).render(sc, 0, 4, 8).cpu().numpy())
    off = (np.abs(imgs[0] - imgs[1]) > 1e-5 * np.abs(imgs[1]) + 1e-6).any(axis=-1).sum()
    assert off <= 1, off


# Triangles whose longest edge squared is 650 to 1400 times twice their area,
# with a ray that passes an edge by a few of flat_trace's error bounds: corners,
# origin and aim. The exact test's rounding decides such rays, which differs
# from that of the plane arithmetic.
SLENDER = [
    ([(-0.574098408, -0.84156394, 0.271853179),
      (-0.662747085, -0.919269085, -0.163141653),
      (-0.662446916, -0.919084191, -0.163264483)],
     (1.30990362, -2.12933588, -0.582932115), (-0.662626272, -0.919196959, -0.163237821)),
    ([(0.888710678, -0.667799354, -0.913880408),
      (0.571613371, -0.393958598, -0.971578956),
      (0.571358919, -0.39413932, -0.971578598)],
     (0.825455368, -1.57785404, -2.64932489), (0.571582298, -0.39398066, -0.971578913)),
    ([(-0.0412372611, 0.230409771, -0.376535982),
      (-0.655070186, -0.453622699, -0.436333328),
      (-0.653996944, -0.454530478, -0.436249822)],
     (-2.47753286, 0.158143461, -2.20428133), (-0.654465049, -0.454185023, -0.436286749)),
    ([(-0.819045722, -0.0108747967, -0.633749902),
      (-1.36246324, -0.496002436, -1.31658602),
      (-1.36244345, -0.495248348, -1.31685078)],
     (0.355672807, -1.84802747, -1.72207677), (-1.3624468, -0.495381475, -1.31680382)),
    ([(-0.950862288, -0.0256499425, 0.176232278),
      (-0.389036149, -0.241063565, 0.56866312),
      (-0.389438152, -0.240668342, 0.567294121)],
     (-0.732924759, 1.57457078, 1.70631206), (-0.389320577, -0.240788209, 0.567713812)),
    ([(-0.831167579, 0.328666508, 0.910116732),
      (-1.35111499, 0.174996153, 0.382492304),
      (-1.3512727, 0.174067885, 0.382832378)],
     (0.381067455, 1.45943701, -0.869288862), (-1.35120776, 0.174449847, 0.382692501)),
]


@pytest.mark.parametrize("case", range(len(SLENDER)))
def test_flat_trace_of_slender_triangles(cuda, case):
    # a film 3e-5 wide around the aim, most of it within the rounding of the edge
    announce(f"flat trace of a slender triangle ({case})")
    corners, origin, aim = SLENDER[case]
    dist = np.linalg.norm(np.subtract(origin, aim))
    imgs = []
    for hidden in (False, True):
        d = {"type": "scene", "tri": _tri(corners, 0.4),
             "env": {"type": "constant", "radiance": {"type": "rgb", "value": 1.0}},
             "ball": {"type": "sphere", "center": [0, -1.6, 0], "radius": 0.3,
                      "bsdf": {"type": "diffuse", "reflectance": {"type": "rgb", "value": 0.5}}},
             "sensor": cam(origin, aim, fov=float(np.degrees(3e-5 / dist)), w=32, h=32, spp=16)}
        if hidden:
            d["hidden"] = _hidden((0, -1.6, 0))
        imgs.append(rcv.load_dict({"type": "prb", "max_depth": 2}).render(rcv.load_dict(d), 0, 9, 16).cpu().numpy())
    off = (np.abs(imgs[0] - imgs[1]) > 1e-5 * np.abs(imgs[1]) + 1e-6).any(axis=-1).sum()
    assert off <= 1, off
