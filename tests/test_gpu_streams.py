"""Calls on one scene from several streams, and captured calls replayed
beside eager ones."""
import ctypes as C

import numpy as np
import pytest
import torch

import recursive_control_variates_amd as rcv
from conftest import announce
from helpers import homogeneous_box_scene, volume_box_scene
from recursive_control_variates_amd import _native as N

pytestmark = pytest.mark.gpu

KEY = "box.interior_medium.sigma_t.data"
W, H, SPP = 40, 28, 16


def _scene(kind="grid", w=W, h=H):
    rng = np.random.default_rng(71)
    if kind == "homogeneous":
        sc, key = rcv.load_dict(homogeneous_box_scene(w=w, h=h, spp=SPP)), "box.interior_medium.sigma_t.value.value"
    else:
        grid = (0.2 + rng.uniform(0, 0.8, (20, 20, 20, 1))).astype(np.float32)
        sc, key = rcv.load_dict(volume_box_scene(grid, albedo=0.8, scale=5.0, w=w, h=h, spp=SPP)), KEY
    p = rcv.traverse(sc)
    for f in (0.9, 1.0):
        p[key] = (p[key].detach() * f).requires_grad_(True)
        p.update()
    gimg = torch.from_numpy(rng.uniform(0.5, 1.5, (h, w, 3)).astype(np.float32)).cuda()
    tangent = {key: torch.from_numpy(rng.uniform(-1, 1, tuple(p[key].shape)).astype(np.float32)).cuda()}
    return sc, p, key, gimg, tangent


def _calls(sc, p, key, gimg, tangent, kinds=("twostateprbvolpath", "volpathsimple")):
    """Name -> call of every kind at one seed."""
    prb = rcv.load_dict({"type": kinds[0], "max_depth": 8, "rr_depth": 4})
    calls = {
        "render": lambda seed: prb.render(sc, 0, seed, SPP),
        "two states": lambda seed: torch.stack(prb.render_twostates(sc, 0, seed, SPP)),
        "forward": lambda seed: prb.render_forward(sc, p, 0, seed, SPP, tangents=tangent),
        "adjoint": lambda seed: prb.adjoint(sc, p, gimg, 0, seed, SPP)[key],
    }
    if len(kinds) > 1:
        simple = rcv.load_dict({"type": kinds[1], "max_depth": 8, "rr_depth": 4})
        calls["volpathsimple adjoint"] = lambda seed: simple.adjoint(sc, p, gimg, 0, seed, SPP)[key]
    return calls


def _assert_close(name, got, want):
    # Images: the same samples, a pixel's 16 added in another order at most
    # (2^-20 of it). Gradients: up to ~10^3 terms per voxel in another order,
    # sqrt(10^3) 2^-24 = 2e-6 of the largest partial sum; 1e-4 of the largest
    # gradient with room for partial sums above the result.
    tol = 1e-4 if "adjoint" in name or name == "forward" else 1e-5
    got, want = got.double().cpu().numpy(), want.double().cpu().numpy()
    scale = np.abs(want).max()
    assert scale > 0 and np.allclose(got, want, rtol=tol, atol=tol * scale), (name, np.abs(got - want).max() / scale)


@pytest.mark.parametrize("kind", ["grid", "homogeneous"])
def test_calls_on_two_streams(cuda, kind):
    announce(f"one scene on two streams ({kind})")
    scene = _scene(kind)
    calls = _calls(*scene, kinds=("twostateprbvolpath", "volpathsimple") if kind == "grid" else ("twostateprbvolpath",))
    want = {(n, k): c(100 + k) for n, c in calls.items() for k in range(4)}
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = {}
    for n, c in calls.items():
        for k in range(4):
            with torch.cuda.stream(streams[k % 2]):
                got[n, k] = c(100 + k)
    torch.cuda.synchronize()
    for (n, k), w in want.items():
        _assert_close(n, got[n, k], w)


def test_more_streams_than_scratches(cuda):
    # 32 streams of torch's pool and the default stream: the last ones take
    # over a scratch
    announce("one scene on 40 streams")
    scene = _scene()
    calls = _calls(*scene)
    want = [calls["forward"](200 + k) for k in range(3)]
    torch.cuda.synchronize()
    got = []
    for k in range(40):
        with torch.cuda.stream(torch.cuda.Stream()):
            got.append(calls["forward"](200 + k % 3))
    torch.cuda.synchronize()
    for k, g in enumerate(got):
        _assert_close("forward", g, want[k % 3])


# (from 2^17 pixels on, captured renders take the tracker)
@pytest.mark.parametrize("name,w,h", [("render", W, H), ("two states", W, H), ("two states", 512, 257),
                                      ("forward", W, H), ("adjoint", W, H), ("volpathsimple adjoint", W, H)])
def test_replays_beside_eager_calls(cuda, name, w, h):
    # The capture is the scene's first launch on its stream; the graph is
    # replayed on another one while eager calls run on the capture's and on
    # the default stream.
    announce(f"captured {name} replayed beside eager calls ({w} x {h})")
    scene = _scene(w=w, h=h)
    call = _calls(*scene)[name]
    want = [call(300 + k) for k in range(3)]
    torch.cuda.synchronize()
    side, replays = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call(300)
    for _ in range(3):
        with torch.cuda.stream(replays):
            graph.replay()
        with torch.cuda.stream(side):
            beside = call(301)
        here = call(302)
        torch.cuda.synchronize()
        _assert_close(name, out, want[0])
        _assert_close(name, beside, want[1])
        _assert_close(name, here, want[2])


@pytest.mark.parametrize("kind", ["prbvolpath", "volpathsimple"])
def test_captured_adjoint_after_an_eager_one(cuda, kind):
    # The capture's stream has its scatter log from an eager call before; the
    # graph is replayed on another stream while eager adjoints log on that one,
    # of another scene with larger sums.
    announce(f"captured {kind} adjoint after an eager one on its stream, replayed beside others")
    name = "adjoint" if kind == "prbvolpath" else "volpathsimple adjoint"
    (a, b) = (_scene(), _scene())
    b[3].mul_(50.0)
    call, other = _calls(*a)[name], _calls(*b)[name]
    want, want_other = call(400), other(401)
    torch.cuda.synchronize()
    side, replays = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        call(402)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call(400)
    for _ in range(4):
        with torch.cuda.stream(replays):
            graph.replay()
        with torch.cuda.stream(side):
            beside = other(401)
        torch.cuda.synchronize()
        _assert_close(name, out, want)
        _assert_close(name, beside, want_other)


def test_first_call_on_a_stream_while_another_is_captured(cuda):
    # its scratch and its scatter log are allocated then, which leaves the
    # capture as it is
    announce("first adjoint on a stream while another stream is being captured")
    sc, p, key, gimg, _ = _scene()
    integ = rcv.load_dict({"type": "prbvolpath", "max_depth": 8, "rr_depth": 4})
    want = integ.adjoint(sc, p, gimg, 0, 500, SPP)[key]
    got, d, index = torch.zeros_like(want), integ.desc(), N.i32_array([sc.params[key].index])
    grads = (C.c_void_p * 1)(got.data_ptr())
    x = torch.zeros(1000, device="cuda")
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        x.add_(1.0)
        N.call("rcv_render_backward", sc.handle, C.byref(d), 0, C.c_uint32(500), SPP, C.c_void_p(gimg.data_ptr()), 1,
               index, grads, C.c_void_p(other.cuda_stream))
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert float(x.min()) == float(x.max()) == 3.0
    _assert_close("adjoint", got, want)
