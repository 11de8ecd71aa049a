"""The proposal network's BF16 kernels at the batch sizes where their forms
change above a few hundred spectra: the convolutions' wide tiles start at
512 (third layer) and 1024 (fourth), and the hidden layer's sums go from
splits of 4 slices to splits of 8 and 16, which the wave groups still share,
with sizes in between (5, and 22 and 32 above 4096) that one group takes alone."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# As for the small batches.  Forward: BF16 operands (2^-9) in four products,
# at most 8e-3 where all roundings agree, and the outputs cancel to about half
# of their terms.  One spectrum's gradient in two batches: five products'
# operands round to BF16 at another scale, 5 x 2^-9 = 1e-2, and a share of
# about 1e-4 of the ReLUs changes sign, 1e-2 of the gradient's norm.  A
# spectrum that a tile's end lost or doubled is an error of one.
TOL_OUT = 2e-2
TOL_GRAD = 3e-2


@pytest.mark.parametrize("n", [
    515,     # wide tiles in the third layer, splits of 4 slices
    1030,    # wide tiles in the fourth, splits of 5
    1700,    # splits of 8
    3300,    # splits of 16
    5000,    # splits of 22
    6200,    # splits of 32
])
def test_every_spectrum_counts_once(n):
    """Targets equal to the outputs leave a spectrum without gradient: with one
    spectrum's target moved away, the batch's gradient is that spectrum's
    alone, divided by the batch."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf, proposal
    rng = np.random.default_rng(n)
    k = np.arange(257) / 257.0
    radial = (np.exp(-3 * k) * np.sin(rng.uniform(5, 60, (n, 1)) * k ** 2 * 6) ** 2
              + 0.02 * rng.standard_normal((n, 257))).astype(np.float32)
    params = proposal.init_params(3)
    d = torch.from_numpy(radial).cuda()
    net, one = gctf.Net(n), gctf.Net(1)
    net.set_params(params)
    one.set_params(params)
    o = net.forward(d.data_ptr(), 257, n)
    # both ends, the middle and one spectrum of every tile of 32
    rows = sorted({*range(8), *range(n // 2, n // 2 + 8), *range(n - 8, n), *range(5, n, 32)})
    ref = O.net_forward(params.astype(np.float64), radial[rows])
    assert (np.linalg.norm(o[rows] - ref, axis=1) <= TOL_OUT * np.linalg.norm(ref, axis=1)).all()
    still = np.stack([np.exp(o[:, 0].astype(np.float64)) * 1e4, o[:, 1] * 1e3, np.rad2deg(o[:, 2]), 0 * o[:, 3]],
                     1).astype(np.float32)
    for b in (0, n // 2, n - 1):
        target = still.copy()
        target[b] = [1.5e4 + still[b, 0], 800.0, 35.0, 1.0]
        t = torch.from_numpy(target).cuda()
        loss, g = net.loss_grad(d.data_ptr(), 257, t.data_ptr(), n, want_grad=True)
        again = net.loss_grad(d.data_ptr(), 257, t.data_ptr(), n, want_grad=True)
        assert again[0] == loss and np.array_equal(again[1], g)
        loss1, g1 = one.loss_grad(d[b].data_ptr(), 257, t[b].data_ptr(), 1, want_grad=True)
        assert abs(loss * n - loss1) <= TOL_OUT * loss1, b
        for name, (ws, bs) in proposal.layer_slices().items():
            for s in (ws, bs):
                assert np.linalg.norm(g[s] * n - g1[s]) <= TOL_GRAD * np.linalg.norm(g1[s]), (b, name, s)
