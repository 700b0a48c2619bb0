"""The surface adjoint's vertex tape: paths with no, some and more textured
vertices than the tape holds, against forward mode on the same samples (which
replays every path): <g, J t> = <J^T g, t> per texture."""
import numpy as np
import pytest
import torch

import recursive_control_variates_amd as rcv
from conftest import announce
from helpers import furnace_box_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_depth", [1, 2, 6, 7, 8, 24])
def test_vertex_tape_is_the_transpose_of_forward_mode(cuda, max_depth):
    announce(f"surface adjoint with all walls textured, max_depth {max_depth}")
    rng = np.random.default_rng(max_depth)
    d = furnace_box_scene(radiance=0.7, w=24, h=18, spp=8)
    walls = [k for k, v in d.items() if isinstance(v, dict) and v.get("type") == "rectangle"]
    for k in walls:
        tex = rng.uniform(0.2, 0.9, (5, 7, 3)).astype(np.float32)
        d[k]["bsdf"] = {"type": "diffuse", "reflectance": {"type": "bitmap", "data": tex}}
    sc = rcv.load_dict(d)
    p = rcv.traverse(sc)
    keys = p.keys()
    assert len(keys) == 6
    for k in keys:
        p[k] = p[k].detach().clone().requires_grad_(True)
    p.update()
    integ = rcv.load_dict({"type": "prb", "max_depth": max_depth, "rr_depth": 30})
    g = torch.from_numpy(rng.uniform(0.5, 1.5, (18, 24, 3)).astype(np.float32)).cuda()
    grads = integ.adjoint(sc, p, g, 0, 5, 8)
    for k in keys:
        t = torch.from_numpy(rng.uniform(0.5, 1.0, (5, 7, 3)).astype(np.float32)).cuda()
        lhs = float((g.double() * integ.render_forward(sc, p, 0, 5, 8, tangents={k: t}).double()).sum())
        rhs = float((grads[k].double() * t.double()).sum())
        # positive terms: float32 sums of a few thousand of them each
        assert abs(lhs - rhs) <= 2e-5 * abs(lhs), (k, lhs, rhs)
        # (at depth 2 only the walls the camera sees have a derivative)
        assert lhs == 0 if max_depth == 1 else (lhs > 0 or max_depth == 2)
