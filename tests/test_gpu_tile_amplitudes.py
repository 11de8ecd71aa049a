"""The tile amplitudes |F| are square roots rounded as IEEE single has it, for
all magnitudes.  A tile with one value A at its centre (and -A in a corner,
which the mask removes, so that the tile's mean is zero) has the transform
+-A at every point: all its butterflies add zeros, and its twiddles multiply
zeros.  The raw half spectrum of one tile is then sqrt(A A), the product and
the root each rounded once, at every pixel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tile", [256, 512, 1024])
@pytest.mark.parametrize("exponent", [0, -50, -66])    # A A normal, below 2^-96, below the least normal number
def test_amplitude_is_the_rounded_root(tile, exponent):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    rng = np.random.default_rng(tile - exponent)
    ctx = gctf.Context(tile=tile)
    nnx, nny, _, pix = ctx.rescale_setup(tile, tile, 1.3)
    ctx.setup1(300.0, 2.7, 0.07, pix)
    ctx.setup2(nnx, nny)
    for a in np.ldexp(rng.uniform(1.0, 4.0, 48), exponent).astype(np.float32):
        img = np.zeros((tile, tile), np.float32)
        img[tile // 2, tile // 2] = a
        img[0, 0] = -a
        d = torch.from_numpy(img).cuda()
        ctx.rescale(d.data_ptr(), on_device=True)
        ctx.gen_half_spectrum(ctx.scaled_image())
        raw = ctx.get_half_spect(raw=True)
        want = np.sqrt(np.float32(a * a))
        assert np.array_equal(raw, np.full_like(raw, want)), (a, want, np.unique(raw))
