"""Rescale at the lengths where its transforms change form, against the FP64
oracle: lengths without a Stockham plan run on a power-of-two grid at least
twice as fine (gctf_fft.hpp, itp_fwd and itp_inv), with shared weights for
even lengths and one set per point for odd ones."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# The interpolation's aliasing is below 1e-7 of the result's norm and FP32
# rounding over the at most 40 rounded operations a value passes through in
# two dimensions is about sqrt(40) x 6e-8 x the twiddles' share, 4e-7 to 1e-6.
TOL = 2e-6


@pytest.mark.parametrize("nx,ny,pix", [
    (1021, 1031, 0.9),    # prime sides: odd forward lengths on 2048 points
    (2047, 600, 1.1),     # odd row just under a power of two (least oversampling); 1876 = 4 x 7 x 67
    (2049, 520, 1.0),     # just over one (most oversampling)
    (600, 2053, 1.0),     # prime height on 8192 points
    (514, 4093, 1.0),     # odd height, 4096-point halves
    (8194, 514, 0.9),     # packed half-length rows of 4097 (odd, prime factors 17 x 241) on 16384 points
    (514, 8182, 0.5),     # split columns: two 4091-point (prime) transforms on 8192 points
    (514, 8182, 1.1),     # the same height on 16384 points, rescaled height 7500 = 2^2 3 5^4
    (514, 7000, 1.1),     # 6416 = 2^4 x 401 inverse on 16384 points
    (900, 1024, 1.0),     # power-of-two forward, mixed-radix inverse columns' neighbour 852 = 4 x 3 x 71
    (9210, 514, 1.1),     # C2R rows of 8442 = 2 x 4221: odd packed length
])
def test_rescale_lengths(nx, ny, pix):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    rng = np.random.default_rng(nx * 10007 + ny)
    img = rng.standard_normal((ny, nx)).astype(np.float32)
    ctx = gctf.Context()
    nnx, nny, pitch, pixn = ctx.rescale_setup(nx, ny, pix)
    d = torch.from_numpy(img).cuda()
    ctx.rescale(d.data_ptr(), on_device=True)
    out = _read(ctx.scaled_image(), nny, pitch)
    ref = np.asarray(O.rescale(img, pix), np.float64)[:, :nnx]
    err = np.linalg.norm(out[:, :nnx] - ref) / np.linalg.norm(ref)
    assert err <= TOL, err
    assert (out[:, nnx:] == 0.0).all()


def _read(ptr, rows, pitch):
    """The padded rescaled image from its device address."""

    class Dev:
        __cuda_array_interface__ = dict(shape=(rows, pitch), typestr="<f4", data=(ptr, False), version=2)

    return torch.as_tensor(Dev(), device="cuda:0").cpu().numpy().astype(np.float64)
