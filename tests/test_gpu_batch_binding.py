"""A batch job traces its ring's states, whatever the scene had bound when
the job was added."""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import announce
from helpers import volume_box_scene
from recursive_control_variates_amd import _native as N
from recursive_control_variates_amd.batch import BatchOptimizer, JobSpec, _JobBuffers, _lib

pytestmark = pytest.mark.gpu

SIGMA = "box.interior_medium.sigma_t.data"
ALBEDO = "box.interior_medium.albedo.data"


def _buffers(key, factor):
    rng = np.random.default_rng(67)
    grid = (0.2 + rng.uniform(0, 0.8, (9, 10, 11, 1))).astype(np.float32)
    albedo = rng.uniform(0.4, 0.9, (9, 10, 11, 3)).astype(np.float32)
    d = volume_box_scene(grid, albedo={"type": "gridvolume", "data": albedo, "to_world": np.eye(4)}, scale=6.0,
                         w=24, h=16, spp=8, majorant_factor=factor)
    init = (albedo if key == ALBEDO else grid) * np.float32(0.9)
    ref = np.full((16, 24, 3), 0.4, np.float32)
    spec = JobSpec(scene=d, key=key, init=init, img_ref=ref, method="cv_ps", loss="L2", spp=8, seed=5,
                   integrator={"type": "twostateprbvolpath", "max_depth": 8, "rr_depth": 8})
    return _JobBuffers(spec, torch.device("cuda", 0))


def _bind(job, states):
    sp = job.scene.params[job.spec.key]
    sp.states = list(states)
    job.scene._bind(sp)


@pytest.mark.parametrize("key", [SIGMA, ALBEDO])
@pytest.mark.parametrize("factor", [0, 4])
def test_states_bound_after_the_job_was_added(cuda, key, factor):
    # The scene holds other states (half the values) while the job is added
    # and gets the ring's before the commit. The same samples as a batch bound
    # first: images equal up to the order of a pixel's 8 additions (2^-21 of
    # it), gradients up to the order of the scatter-adds.
    announce(f"batch job bound after it was added ({key}, supergrid factor {factor})")
    out = []
    for late in (False, True):
        job = _buffers(key, factor)
        if not late:
            batch = BatchOptimizer([job], use_graph=False)
        else:
            batch = BatchOptimizer.__new__(BatchOptimizer)
            batch.device, batch.use_graph, batch.jobs, batch.iterations = job.scene.device, False, [job], 0
            batch.stream = torch.cuda.Stream()
            batch._h = C.c_void_p()
            lib = _lib()
            other = 0.5 * job.ring[0]
            _bind(job, [other, other])
            N.check(lib.rcv_batch_create(C.byref(batch._h)), "rcv_batch_create")
            desc, index = job.native(), C.c_int32()
            N.check(lib.rcv_batch_add_job(batch._h, C.byref(desc), C.byref(index)), "rcv_batch_add_job")
            _bind(job, job.ring[:2])
            batch.stream.wait_stream(torch.cuda.current_stream())
            N.check(lib.rcv_batch_commit(batch._h, C.c_void_p(batch.stream.cuda_stream)), "rcv_batch_commit")
            batch.set_launch()
        batch.step(1)
        batch.synchronize()
        out.append([x.double().cpu().numpy() for x in (job.F, job.H, job.grad)])
        batch.close()
    for k, (a, b) in enumerate(zip(*out)):
        scale = np.abs(a).max()
        assert scale > 0
        assert np.allclose(b, a, rtol=1e-5 if k < 2 else 1e-4, atol=(1e-6 if k < 2 else 1e-4) * scale), \
            (k, np.abs(a - b).max() / scale)
