"""The 2D search's launches over batch sizes: the candidates per workgroup and
so the kernels of a stage follow from the batch size, and each transition is
made inside the next stage's launch.  A spectrum's result may not depend on
either.  The radial averages are FP32 sums in table order, bit for bit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _setup():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf
    return gctf


def _spectra(n, pix, seed, flat=()):
    """Half spectra [n][512][257] with Thon rings under noise; those in `flat`
    are zero (every CC 0: no candidate is better than the first)."""
    rng = np.random.default_rng(seed)
    ky, kx = np.meshgrid((np.arange(512) - 256) / (512 * pix), np.arange(257) / (512 * pix), indexing="ij")
    k2, th = kx * kx + ky * ky, np.arctan2(ky, kx)
    out = np.empty((n, 512, 257), np.float32)
    for i in range(n):
        df = rng.uniform(8000, 25000) + rng.uniform(100, 700) * np.cos(2 * (th - rng.uniform(-1.5, 1.5)))
        c = np.abs(np.sin(np.pi * 0.01969 * k2 * (df - 0.5 * 0.01969 ** 2 * 2.7e7 * k2) + 0.07))
        out[i] = np.exp(-20 * k2) * (c - 0.64) + 0.3 * rng.standard_normal((512, 257))
        if i in flat:
            out[i] = 0.0
    return torch.from_numpy(out).cuda()


# block sizes of the line stages at 22, 52 and 32 candidates: 1 spectrum 1,
# 3 spectra 1 to 2, 7 spectra 2 to 4, 16 spectra 4 to 8
@pytest.mark.parametrize("n", [3, 7, 16])
@pytest.mark.parametrize("phase", [0.0, 60.0, 90.0])   # without, 61 and more than 64 phase candidates
def test_result_independent_of_batch(n, phase):
    gctf = _setup()
    sp = _spectra(n, 1.2, 900 + n, flat=(1,))
    ctx = gctf.Context(ext_phase=(45.0, phase) if phase > 0.0 else (0.0, 0.0))
    ctx.setup1(300.0, 2.7, 0.07, 1.2)
    out = torch.zeros((n, 6), dtype=torch.float32, device="cuda")
    one = torch.zeros((n, 6), dtype=torch.float32, device="cuda")
    ctx.do2d_batch_static(sp.data_ptr(), n, out.data_ptr())
    for i in range(n):
        ctx.do2d_batch_static(sp[i].data_ptr(), 1, one[i].data_ptr())
    ctx.synchronize()
    assert np.array_equal(out.cpu().numpy(), one.cpu().numpy(), equal_nan=True)
    for block in (2, 16):
        c2 = gctf.Context(ext_phase=(45.0, phase) if phase > 0.0 else (0.0, 0.0))
        c2.tune(search_block=block)
        c2.setup1(300.0, 2.7, 0.07, 1.2)
        c2.do2d_batch_static(sp.data_ptr(), n, one.data_ptr())
        c2.synchronize()
        assert np.array_equal(out.cpu().numpy(), one.cpu().numpy(), equal_nan=True), block


@pytest.mark.parametrize("tile", [256, 512, 1024])
def test_radial_average_bits(tile):
    gctf = _setup()
    cx = tile // 2 + 1
    rng = np.random.default_rng(tile)
    s = rng.standard_normal((3, tile, cx)).astype(np.float32)
    ctx = gctf.Context(tile=tile)
    d = torch.from_numpy(s).cuda()
    out = torch.full((3, cx + 5), -7.0, dtype=torch.float32, device="cuda")
    ctx.radial_average(d.data_ptr(), 3, out.data_ptr(), cx + 5)
    got = out.cpu().numpy()
    assert np.all(got[:, cx:] == -7.0)
    counts, xy = O.radial_table(cx, tile)
    first = np.concatenate([[0], np.cumsum(counts)])
    for i in range(3):
        v = s[i][xy[:, 1] % tile, xy[:, 0]]
        ref = [np.add.accumulate(v[a:b])[-1] / np.float32(b - a) for a, b in zip(first[:-1], first[1:])]
        assert np.array_equal(got[i, :cx], np.array(ref, np.float32))
