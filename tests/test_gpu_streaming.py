"""Stride loops and vector forms of the combine, the running variance and the
loss at the sizes where they change: fewer elements than a block, remainders,
unaligned buffers, several strides per thread."""
import numpy as np
import pytest
import torch

from conftest import announce
from recursive_control_variates_amd.optim import l1_loss, l2_loss
from recursive_control_variates_amd.welford import CVState, WelfordVarianceEstimator

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 4, 1023, 4096, 4099, 1024 * 256 * 4, 1024 * 256 * 4 + 4, 1024 * 256 * 4 * 2 + 37]


@pytest.mark.parametrize("n", SIZES)
def test_combine_strides_match_the_oracle(cuda, n):
    import welford_ref
    announce(f"combine and running variance over {n} elements")
    rng = np.random.default_rng(n)
    st, ref = CVState((n,), cuda), welford_ref.CVStateRef((n,))
    est, xs = WelfordVarianceEstimator(0.9, 0.99), []
    for _ in range(4):
        h, f = (rng.uniform(0.2, 1.0, n).astype(np.float32) for _ in range(2))
        st.step(torch.from_numpy(h).cuda(), torch.from_numpy(f).cuda(), 1)
        ref.step(h, f)
        est.update(torch.from_numpy(f).cuda())
        xs.append(f.astype(np.float64))
    got = st.buf.cpu().numpy()
    for k, a in enumerate(ref.arrays()):
        assert np.array_equal(got[k].view(np.uint32), a.view(np.uint32)), k
    assert st.counters.tolist()[:3] == [4, 3, 0]
    # the running variance in 64 bits
    b1, b2, m, v = float(np.float32(0.9)), float(np.float32(0.99)), np.zeros(n), np.zeros(n)
    for k, x in enumerate(xs):
        d1 = x - m / (1 - b1 ** k) if k > 0 else x
        m = b1 * m + (1 - b1) * x
        v = b2 * v + (1 - b2) * d1 * (x - m / (1 - b1 ** (k + 1)))
    assert int(est.counter[0]) == 4
    np.testing.assert_allclose(est.mean.cpu().numpy(), m, rtol=1e-6)
    np.testing.assert_allclose(est.var.cpu().numpy(), v, rtol=2e-5, atol=2e-7)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("loss", [l1_loss, l2_loss])
def test_loss_sizes_and_alignment(cuda, n, offset, loss):
    # offset 1: buffers that are not 16-byte aligned
    announce(f"{loss.__name__} over {n} elements, offset {offset}")
    rng = np.random.default_rng(n + offset)
    a, b = (rng.uniform(0.0, 1.0, n + offset).astype(np.float32) for _ in range(2))
    x = torch.from_numpy(a).cuda()[offset:].requires_grad_(True)
    y = torch.from_numpy(b).cuda()[offset:]
    out = loss(x, y)
    out.backward()
    d = a[offset:].astype(np.float64) - b[offset:].astype(np.float64)
    want = np.abs(d).mean() if loss is l1_loss else (d * d).mean()
    # float32 differences and products, sums of at most 2^13 terms per thread in tree order
    np.testing.assert_allclose(float(out.detach()), want, rtol=2e-6)
    g = np.sign(d) / n if loss is l1_loss else 2 * d / n
    np.testing.assert_allclose(x.grad.cpu().numpy(), g, rtol=1e-5, atol=3e-7 / n)
