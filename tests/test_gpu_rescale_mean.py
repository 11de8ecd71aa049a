"""Rescale of images whose mean is far above their contrast, as detectors
give them: the interpolated transforms of lengths without a Stockham plan may
not leak the mean into the rest."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# Of the result's norm, which the mean makes up: as for zero-mean images,
# aliasing below 1e-7 and FP32 rounding of 4e-7 to 1e-6.
TOL = 2e-6


@pytest.mark.parametrize("nx,ny,pix", [
    (1021, 1031, 0.9),    # prime sides, odd lengths
    (2047, 600, 1.1),     # least oversampling
    (3710, 1550, 0.7),    # even lengths with shared weights
    (514, 8182, 0.5),     # split columns
    (8194, 514, 0.9),     # packed half-length rows
])
def test_large_mean(nx, ny, pix):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    rng = np.random.default_rng(nx * 10007 + ny)
    img = (1000.0 + 30.0 * rng.standard_normal((ny, nx))).astype(np.float32)
    ctx = gctf.Context()
    nnx, nny, pitch, _ = ctx.rescale_setup(nx, ny, pix)
    d = torch.from_numpy(img).cuda()
    ctx.rescale(d.data_ptr(), on_device=True)

    class Dev:
        __cuda_array_interface__ = dict(shape=(nny, pitch), typestr="<f4", data=(ctx.scaled_image(), False), version=2)

    out = torch.as_tensor(Dev(), device="cuda:0").cpu().numpy().astype(np.float64)
    ref = np.asarray(O.rescale(img, pix), np.float64)[:, :nnx]
    err = np.linalg.norm(out[:, :nnx] - ref) / np.linalg.norm(ref)
    assert err <= TOL, err
    # the mean itself, a sum of the whole image's rounding errors, and no drift
    # of it along either side
    dev = out[:, :nnx] - ref
    assert abs(dev.mean()) <= TOL * abs(ref.mean())
    assert np.abs(dev.mean(0)).max() <= 2 * TOL * abs(ref.mean())
    assert np.abs(dev.mean(1)).max() <= 2 * TOL * abs(ref.mean())
