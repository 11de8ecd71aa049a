"""Background removal and low-pass of the three tile sizes, whose box sums and
column transforms run in groups that end inside the half spectrum (129, 257
and 513 columns), against the FP64 oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tile", [256, 512, 1024])
@pytest.mark.parametrize("log_spect", [False, True])
@pytest.mark.parametrize("scale", [0.01, 1.0])    # below and above the gate's variance of 1: without and with low-pass
def test_background_and_lowpass(tile, log_spect, scale):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    n = 2 * tile + 6
    rng = np.random.default_rng(tile + log_spect)
    y, x = np.mgrid[:n, :n]
    img = (scale * (rng.standard_normal((n, n)) + 0.5 * np.sin(0.7 * x + 0.2 * y))).astype(np.float32)
    ctx = gctf.Context(tile=tile, log_spect=log_spect)
    nnx, nny, pitch, pix = ctx.rescale_setup(n, n, 1.3)
    d = torch.from_numpy(img).cuda()
    ctx.rescale(d.data_ptr(), on_device=True)
    ctx.setup1(300.0, 2.7, 0.07, pix)
    ctx.setup2(nnx, nny)
    ctx.gen_half_spectrum(ctx.scaled_image())
    raw = ctx.get_half_spect(raw=True).astype(np.float64)
    got = ctx.get_half_spect().astype(np.float64)
    ref = O.rm_background(raw, log_spect=int(log_spect))
    if O.gate(ref):
        ref = O.lowpass(ref)
    # sums of up to 69 x 69 values in FP32 and, low-passed, two transforms of
    # 1024: about 1e-6 of the raw spectrum, whose background cancels
    assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(raw)
