"""Rescale at lengths 2^a 3^b 5^c whose transforms take each of the pass
radices, with and without a first radix of 8 (whose absence leaves the LDS
addresses of the passes unequally spaced), against the FP64 oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# As for the other lengths: FP32 rounding over at most about 40 rounded
# operations in two dimensions, 4e-7 to 1e-6.
TOL = 2e-6


@pytest.mark.parametrize("nx,ny,pix", [
    (3000, 520, 1.0),     # rows 10 10 6 5, C2R 2500 = 10 10 5 5
    (1215, 514, 1.1),     # odd rows: 9 9 5 3
    (5625, 514, 0.9),     # odd rows: 9 5 5 5 5
    (514, 7680, 1.0),     # columns 8 8 12 10, inverse 6400
    (11520, 514, 1.0),    # packed rows of 5760 = 8 8 10 9, C2R 9600
    (1440, 1536, 1.0),    # no radix 8 in the rows, columns 1536, inverse 1280
    (6480, 600, 0.8),     # rows 8 10 9 9
    (540, 4860, 0.9),     # columns with two factors of 2
    (2700, 1350, 1.08),   # rows and columns with one or two factors of 2
    (640, 15000, 0.5),    # columns on 16384 points, inverse 6250 = 2 x 5^5
])
def test_mixed_radix_lengths(nx, ny, pix):
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
