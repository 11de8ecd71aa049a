"""The flatness gate: low-pass when mean(o^2) - mean(o)^2 of the background-
removed spectrum o is at least 1 in single precision (CFindCtfBase.cpp:
171-174).  The sums behind the two means run over up to half a million pixels."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _image(tile, seed):
    n = 2 * tile + 6
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[:n, :n]
    return rng.standard_normal((n, n)) + 0.5 * np.sin(0.7 * x + 0.2 * y)


def _context(tile, log_spect=False):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    ctx = gctf.Context(tile=tile, log_spect=log_spect)
    n = 2 * tile + 6
    nnx, nny, _, pix = ctx.rescale_setup(n, n, 1.3)
    ctx.setup1(300.0, 2.7, 0.07, pix)
    ctx.setup2(nnx, nny)
    return ctx


def _spectra(ctx, img):
    """Raw half spectrum and the half spectrum after the gate."""
    d = torch.from_numpy(img.astype(np.float32)).cuda()
    ctx.rescale(d.data_ptr(), on_device=True)
    ctx.gen_half_spectrum(ctx.scaled_image())
    return ctx.get_half_spect(raw=True), ctx.get_half_spect()


def _background32(raw):
    """The background-removed spectrum in single precision, operation by
    operation as the library forms it (GRmBackground2D.cu:33-95)."""
    f = np.float32
    t, cx = raw.shape
    box = int(f(1.0 / 15.0) * f(t))
    if f(box) > f(0.3) * f(t):
        box = int(f(0.3) * f(t))
    hb = max(box // 2 * 2 + 1, 7) // 2
    rest = np.roll(raw[::-1], 1, 0)                  # row (t - y) mod t
    p = np.sqrt(np.concatenate([raw[:, :t // 2], rest[:, t // 2:0:-1]], 1))
    h = np.zeros_like(p)
    for j in range(-hb, hb + 1):
        h += np.roll(p, -j, 1)
    q = np.zeros_like(h)
    for j in range(-hb, hb + 1):
        q += np.roll(h, -j, 0)
    acc = q[:, :cx] / f((2 * hb + 1) ** 2)
    acc *= acc
    x = np.arange(cx, dtype=f) * f(0.5) / f(cx - 1)
    yc = np.arange(t) - t // 2
    fr = np.sqrt(x[None, :] * x[None, :] + (yc * yc).astype(f)[:, None] / f(t * t))
    return np.where(fr.astype(np.float64) < 0.04, f(0), raw - acc)


def _gate32(o):
    """The gate of o, its sums in 64 bits, the rest in single precision."""
    o = o.astype(np.float64)
    mean, std = np.float32(o.sum() / o.size), np.float32((o * o).sum() / o.size)
    return not std - mean * mean < np.float32(1.0)


@pytest.mark.parametrize("tile", [256, 512, 1024])
def test_gate_at_its_threshold(tile):
    """Variances in steps of 4e-8 around 1, a third of the spacing of single
    precision there: the sums' own rounding may not move the decision."""
    img = _image(tile, tile)
    ctx = _context(tile)
    raw, half = _spectra(ctx, 1e-3 * img)
    o = _background32(raw)
    assert np.array_equal(half, o)
    s0 = 1e-3 / np.sqrt(np.var(o.astype(np.float64)))
    decided = []
    for k in range(-16, 17):
        raw, half = _spectra(ctx, s0 * (1.0 + 2e-8 * k) * img)
        o = _background32(raw)
        want = _gate32(o)
        assert want == (not np.array_equal(half, o)), (k, np.var(o.astype(np.float64)) - 1.0)
        decided.append(want)
    assert any(decided) and not all(decided)


@pytest.mark.parametrize("tile", [256, 512, 1024])
@pytest.mark.parametrize("log_spect", [False, True])
def test_background_without_lowpass(tile, log_spect):
    """All three tile sizes on the side of the gate where nothing is filtered."""
    ctx = _context(tile, log_spect)
    raw, half = _spectra(ctx, 1e-3 * _image(tile, 3 * tile + log_spect))
    ref = O.rm_background(raw.astype(np.float64), log_spect=int(log_spect))
    assert O.gate(ref) == 0
    # FP32 sums of up to 69 x 69 values: below 69 x 6e-8 of the background,
    # a part of the raw spectrum
    assert np.linalg.norm(half - ref) <= 5e-6 * np.linalg.norm(raw)
