"""The calls this library is measured on.

listed() holds the work a user of the library has it do, from one small
micrograph to the largest batches: the sizes are those of bench.py, of the
full-size tests (tests/test_gpu_full_configs.py) and of the smoke run.
draw() gives further calls of the same ranges.  Each case has a "kind":

  estimate  gctf_estimate_batch, the whole plain path of a few micrographs
  list      gctf_estimate_list, micrographs of different shapes and types
  session   the reference-shaped calls for one micrograph (CRescaleImage,
            CFindCtfBase::GenHalfSpectrum, GetHalfSpect), the half spectra
  spectra   gctf_radial_batch: rescale, tile spectra, background, low-pass
            and radial averages of a batch, the part every path shares
  search    gctf_do2d_batch_static: Do1D + Do2D on half spectra
  grid      gctf_grid_search_batch, the BF16 grid search
  train     one training step of the proposal network
  propose   the proposal network's forward pass

The whole calls (estimate, list) end in chains of argmax decisions; the
others return what their kernels compute.
"""
import math

import numpy as np
import torch

from gctffind_amd import gctf, proposal

DEV = "cuda:0"
PIX_WORK = 1.2          # A, the pixel size micrographs are rescaled to
LAM = proposal.gctf_wavelength(300.0)
CS = 2.7e7              # A
AMP = math.atan(0.07 / math.sqrt(1.0 - 0.07 * 0.07))


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one small micrograph, as the smoke run takes it: latency and launches
        dict(name="estimate 1 x 1024^2", kind="estimate", n=1, nx=1024, ny=1024, pix=1.2, half=False),
        # a session's mix of cameras and pixel sizes in one call
        dict(name="list 8 uneven", kind="list", n=8, pix_lo=0.5, pix_hi=1.1),
        # one 4096^2 micrograph through the reference's calls
        dict(name="session 4096^2 1.0 A", kind="session", nx=4096, ny=4096, pix=1.0, tile=512),
        # the headline workload's spectra: 32 micrographs, rescaled 1.0 -> 1.2 A
        dict(name="spectra 32 x 4096^2 1.0 A", kind="spectra", n=32, nx=4096, ny=4096, pix=1.0, half=False,
             tile=512),
        # K3 frames in float16: odd transform lengths
        dict(name="spectra 8 x 5760x4092 f16", kind="spectra", n=8, nx=5760, ny=4092, pix=0.8, half=True,
             tile=512),
        # super-resolution K3 frames, binned by 2.4
        dict(name="spectra 4 x 11520x8184 f16", kind="spectra", n=4, nx=11520, ny=8184, pix=0.5, half=True,
             tile=512),
        # a tilt series' spectra: no rescale
        dict(name="spectra 41 x 3838x3710", kind="spectra", n=41, nx=3838, ny=3710, pix=1.35, half=False,
             tile=512),
        # the search alone, on one spectrum (serving) and on a full static call
        dict(name="search 1", kind="search", n=1, pix=1.2, phase=0.0),
        dict(name="search 16", kind="search", n=16, pix=1.2, phase=0.0),
        # the BF16 grid search on its batch of 256
        dict(name="grid 256 x 4096^2", kind="grid", n=256, nx=4096, ny=4096, pix=1.0),
        # the network: a training step, and the proposals of one batch
        dict(name="train 256", kind="train", n=256),
        dict(name="propose 32", kind="propose", n=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spectra"] * 5 + ["session", "search", "search", "estimate", "list", "grid", "train", "propose"])
    if kind in ("spectra", "session", "estimate"):
        # sides from one small tile grid to super-resolution frames, even and odd
        nx, ny = _log_int(rng, 1000, 11520), _log_int(rng, 1000, 8184)
        pix = round(rng.uniform(0.5, 1.4), 3)
        tile = rng.choice([512, 512, 512, 512, 256, 1024])
        # after the rescale a side still holds a tile
        while min(nx, ny) * min(1.0, pix / PIX_WORK) < 1.1 * tile:
            nx, ny = nx * 2, ny * 2
        nx, ny = min(nx, 11520), min(ny, 8184)
        # working lengths of the column transforms: long odd heights have none
        if ny > 4096:
            ny -= ny % 2
        if nx > 4096:
            nx -= nx % 2
        if kind == "session":
            return dict(kind=kind, nx=nx, ny=ny, pix=pix, tile=tile)
        if kind == "estimate":
            return dict(kind=kind, n=rng.choice([1, 1, 2]), nx=nx, ny=ny, pix=pix, half=rng.random() < 0.5)
        n = max(1, min(_log_int(rng, 1, 64), (32 << 24) // (nx * ny)))
        return dict(kind=kind, n=n, nx=nx, ny=ny, pix=pix, half=rng.random() < 0.5, tile=tile)
    if kind == "list":
        return dict(kind=kind, n=rng.randint(2, 8), pix_lo=round(rng.uniform(0.5, 0.8), 3),
                    pix_hi=round(rng.uniform(0.9, 1.3), 3))
    if kind == "search":
        return dict(kind=kind, n=rng.randint(1, 16), pix=round(rng.uniform(1.2, 1.35), 3),
                    phase=rng.choice([0.0, 0.0, 0.0, 60.0]))
    if kind == "grid":
        return dict(kind=kind, n=rng.randint(2, 64), nx=_log_int(rng, 1200, 4096), ny=_log_int(rng, 1200, 4096),
                    pix=round(rng.uniform(1.0, 1.3), 3))
    return dict(kind=kind, n=_log_int(rng, 1, 512))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _micrographs(n, ny, nx, pix, seed, half=False, df=(5000.0, 50000.0)):
    """n synthetic micrographs [n][ny][nx] on the GPU: defocus log-uniform,
    astigmatism up to 1500 A, SNR 0.03-0.3, B 50-200 A^2."""
    rng = np.random.default_rng(seed)
    d1, d2, az, b, s = proposal.draw_params(rng, n, df_lo=df[0], df_hi=df[1])
    out = torch.empty((n, ny, nx), dtype=torch.float16 if half else torch.float32, device=DEV)
    for i in range(n):
        proposal.micrograph_batch(torch, 1, ny, nx, pix, d1[i:i + 1], d2[i:i + 1], az[i:i + 1], b[i:i + 1],
                                  s[i:i + 1], seed * 1000 + i, out=out[i:i + 1], device=DEV)
    return out


def _half_spectra(n, pix, seed):
    """n background-removed half spectra [n][512][257] as GenHalfSpectrum
    leaves them: |CTF| oscillations under an envelope, and noise."""
    rng = np.random.default_rng(seed)
    d1, d2, az, _, _ = proposal.draw_params(rng, n, df_lo=5000.0, df_hi=40000.0)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    ky = (torch.arange(512, device=DEV) - 256)[:, None] / (512.0 * pix)
    kx = torch.arange(257, device=DEV)[None, :] / (512.0 * pix)
    k2 = (kx * kx + ky * ky).to(torch.float64)
    th = torch.atan2(ky.expand_as(k2), kx.expand_as(k2)).to(torch.float64)
    out = torch.empty((n, 512, 257), dtype=torch.float32, device=DEV)
    for i in range(n):
        df = 0.5 * (d1[i] + d2[i]) + 0.5 * (d1[i] - d2[i]) * torch.cos(2.0 * (th - math.radians(az[i])))
        c = torch.sin(math.pi * LAM * k2 * (df - 0.5 * LAM * LAM * CS * k2) + AMP).abs()
        env = torch.exp(-rng.uniform(50.0, 120.0) * k2 / 4.0)
        noise = torch.randn((512, 257), generator=g, device=DEV, dtype=torch.float32)
        s = env * (c - 2.0 / math.pi) + rng.uniform(0.1, 0.5) * noise
        out[i] = torch.where(k2 * pix * pix < 0.04 ** 2, torch.zeros_like(s), s).to(torch.float32)
    return out


def _radial_rows(n, seed):
    """n radial spectra [n][257] with Thon rings, and their targets [n][4]."""
    rng = np.random.default_rng(seed)
    d1, d2, az, b, _ = proposal.draw_params(rng, n)
    k2 = (np.arange(257) / (512.0 * PIX_WORK)) ** 2
    df = 0.5 * (d1 + d2)
    c = np.abs(np.sin(math.pi * LAM * k2 * (df[:, None] - 0.5 * LAM * LAM * CS * k2) + AMP))
    r = np.exp(-b[:, None] * k2 / 4.0) * (c - 2.0 / math.pi) + 0.02 * rng.standard_normal((n, 257))
    label = rng.choice([-1.0, 0.0, 1.0], n)
    t = np.stack([df, np.abs(d1 - d2), az, label], 1)
    return (torch.from_numpy(r.astype(np.float32)).to(DEV), torch.from_numpy(t.astype(np.float32)).to(DEV))


def _list_shapes(case, seed):
    """(ny, nx, half, pix) of an uneven list: half 4096^2 float32, the rest
    K3 frames and super-resolution K3 frames in float16."""
    rng = np.random.default_rng(10 ** 6 + seed)
    kinds = [(4096, 4096, False), (4092, 5760, True), (4096, 4096, False), (8184, 11520, True)]
    return [kinds[i % 4] + (float(np.float32(rng.uniform(case["pix_lo"], case["pix_hi"]))),)
            for i in range(case["n"])]


def _params(seed):
    """Network parameters of a run in training."""
    return proposal.init_params(seed)


def prepare(case, seed):
    k = case["kind"]
    st = dict(case=case)
    if k in ("estimate", "spectra", "grid", "session"):
        n = case.get("n", 1)
        st["img"] = _micrographs(n, case["ny"], case["nx"], case["pix"], seed, case.get("half", False),
                                 df=(5000.0, 40000.0))
        st["ctx"] = ctx = gctf.Context(tile=case.get("tile", 512))
        if k == "spectra":
            st["out"] = torch.zeros((n, case["tile"] // 2 + 1), dtype=torch.float32, device=DEV)
        if k == "session":
            nnx, nny, _, pixn = ctx.rescale_setup(case["nx"], case["ny"], case["pix"])
            ctx.setup1(300.0, 2.7, 0.07, pixn)
            ctx.setup2(nnx, nny)
    elif k == "list":
        st["imgs"], st["items"] = [], []
        for i, (ny, nx, half, pix) in enumerate(_list_shapes(case, seed)):
            im = _micrographs(1, ny, nx, pix, seed * 16 + i, half, df=(5000.0, 40000.0))
            st["imgs"].append(im)
            st["items"].append(dict(data=im.data_ptr(), dtype=gctf.DTYPE_F16 if half else gctf.DTYPE_F32, nx=nx,
                                    ny=ny, pix=pix))
        st["ctx"] = gctf.Context()
    elif k == "search":
        st["spect"] = _half_spectra(case["n"], case["pix"], seed)
        st["out"] = torch.zeros((case["n"], 6), dtype=torch.float32, device=DEV)
        p = case["phase"]
        st["ctx"] = ctx = gctf.Context(ext_phase=(45.0, p) if p > 0.0 else (0.0, 0.0))
        ctx.setup1(300.0, 2.7, 0.07, case["pix"])
    else:
        st["radial"], st["target"] = _radial_rows(case["n"], seed)
        st["net"] = gctf.Net(case["n"])
        st["params"] = proposal.load_params()[0] if k == "propose" else _params(seed)
        st["net"].set_params(st["params"])
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _rows(results):
    return np.array([[r["df_min"], r["df_max"], r["azimuth"], r["ext_phase"], r["score"], r["ctf_res"]]
                     for r in results], np.float32)


def run(st):
    case = st["case"]
    k = case["kind"]
    if k == "estimate":
        return _rows(st["ctx"].estimate_batch(st["img"].data_ptr(), case["n"], case["nx"], case["ny"], case["pix"],
                                              dtype=gctf.DTYPE_F16 if case["half"] else gctf.DTYPE_F32))
    if k == "list":
        return _rows(st["ctx"].estimate_list(st["items"]))
    if k == "session":
        ctx = st["ctx"]
        ctx.rescale(st["img"].data_ptr(), on_device=True)
        ctx.gen_half_spectrum(ctx.scaled_image())
        return dict(raw=ctx.get_half_spect(raw=True), half=ctx.get_half_spect())
    if k == "spectra":
        st["ctx"].radial_batch(st["img"].data_ptr(), case["n"], case["nx"], case["ny"], case["pix"],
                               st["out"].data_ptr(), case["tile"] // 2 + 1,
                               dtype=gctf.DTYPE_F16 if case["half"] else gctf.DTYPE_F32)
        return st["out"]
    if k == "search":
        st["ctx"].do2d_batch_static(st["spect"].data_ptr(), case["n"], st["out"].data_ptr())
        st["ctx"].synchronize()
        return st["out"]
    if k == "grid":
        return _rows(st["ctx"].grid_search_batch(st["img"].data_ptr(), case["n"], case["nx"], case["ny"],
                                                 case["pix"], gctf.GRID_256x32x36))
    net = st["net"]
    if k == "propose":
        return net.forward(st["radial"].data_ptr(), 257, case["n"])
    loss, grad = net.loss_grad(st["radial"].data_ptr(), 257, st["target"].data_ptr(), case["n"], want_grad=True)
    net.adam_step(3.0e-4, weight_decay=1.0e-4)
    return dict(loss=loss, grad=grad, params=net.get_params())


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def _sizes(nx, ny, pix):
    """Rescaled size (CRescaleImage::Setup, in single precision)."""
    b = np.float32(PIX_WORK) / np.float32(pix)
    if b <= 1:
        return nx // 2 * 2, ny // 2 * 2, float(np.float32(pix)), False
    f = lambda n: int(np.float32(n) / b + np.float32(0.5)) // 2 * 2
    return f(nx), f(ny), float(np.float32(pix) * b), True


def _tile_grid(nnx, nny, tile):
    step = tile // 2
    ntx, nty = (nnx - step) // step, (nny - step) // step
    offx, offy = (nnx - (ntx + 1) * step) // 2, (nny - (nty + 1) * step) // 2
    return ntx, nty, offx, offy, step


def _fft(n):
    return 5.0 * n * math.log2(n)


def _spectrum_work(nx, ny, pix, tile, esz):
    """Input read and half spectrum written once; the transforms of the
    rescale (rows, columns, inverse columns, inverse rows) and of the tiles,
    real rows counted as half a complex transform."""
    nnx, nny, _, act = _sizes(nx, ny, pix)
    ntx, nty, _, _, _ = _tile_grid(nnx, nny, tile)
    ncx = nnx // 2 + 1
    fl = 0.0
    if act:
        fl = ny * _fft(nx) / 2 + ncx * (_fft(ny) + _fft(nny)) + nny * _fft(nnx) / 2
    fl += ntx * nty * (tile * _fft(tile) / 2 + (tile // 2 + 1) * _fft(tile))
    return nx * ny * esz + 4.0 * tile * (tile // 2 + 1), fl


# flops of one candidate CTF value and its two correlation sums
_CAND_FLOP = 20.0
# candidates of the plain 2D program: 51 x 51 grid, 19 rounds of 21 + 51 + 31
_CANDS = 51 * 51 + 19 * (21 + 51 + 31)


def _ring_pixels(pix):
    """Half-ring area between 1/(25 p) and 1/max(2 p / 0.8, 3.5) cycles per A."""
    hi = 512.0 * pix / max(2.0 * pix / 0.8, 3.5)
    lo = 512.0 / 25.0
    return 0.5 * math.pi * (hi * hi - lo * lo)


def work(case):
    k = case["kind"]
    if k in ("estimate", "spectra", "grid", "session"):
        n = case.get("n", 1)
        b, f = _spectrum_work(case["nx"], case["ny"], case["pix"], case.get("tile", 512),
                              2 if case.get("half") else 4)
        b, f = b * n, f * n
        pix = max(case["pix"], PIX_WORK)
        if k == "estimate":
            f += n * _CANDS * _ring_pixels(pix) * _CAND_FLOP
        if k == "grid":
            ring = 0.5 * math.pi * (512.0 * pix) ** 2 * (1.0 / 16.0 - 1.0 / 900.0)
            f += 2.0 * 256 * 32 * 36 * ring * n
        return {"bytes": b, "flops": f}
    if k == "list":
        b = f = 0.0
        for ny, nx, half, pix in _list_shapes(case, 0):
            bi, fi = _spectrum_work(nx, ny, pix, 512, 2 if half else 4)
            b, f = b + bi, f + fi + _CANDS * _ring_pixels(max(pix, PIX_WORK)) * _CAND_FLOP
        return {"bytes": b, "flops": f}
    if k == "search":
        c = _CANDS + (19 * 61 if case["phase"] > 0.0 else 0)
        return {"bytes": case["n"] * 4.0 * 512 * 257, "flops": case["n"] * c * _ring_pixels(case["pix"]) * _CAND_FLOP}
    # conv1-4 and fc1-2, multiply-adds per spectrum
    mac = 64 * 7 * 256 + 64 * 448 * (128 + 64 + 32) + 1024 * 128 + 128 * 4
    n = case["n"]
    if k == "propose":
        return {"bytes": 4.0 * proposal.n_params() + 4.0 * n * 257, "flops": 2.0 * mac * n}
    return {"bytes": 4.0 * 8 * proposal.n_params() + 4.0 * n * 261, "flops": 6.0 * mac * n}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _rescale64(img, pix):
    ny, nx = img.shape
    nnx, nny, _, act = _sizes(nx, ny, pix)
    if not act:
        return img[:nny, :nnx].to(torch.float64)
    f = torch.fft.rfft(img.to(torch.float64), dim=1)[:, :nnx // 2 + 1].contiguous()
    f = torch.fft.fft(f, dim=0)
    top = nny // 2 + 1
    f = torch.cat([f[:top], f[ny - (nny - top):]])
    f = torch.fft.ifft(f, dim=0, norm="forward")
    # the inverse row transform reads the real parts of the DC and Nyquist columns
    f[:, 0] = f[:, 0].real.to(f.dtype)
    f[:, -1] = f[:, -1].real.to(f.dtype)
    return torch.fft.irfft(f, n=nnx, dim=1, norm="forward")


def _round_edge64(tile):
    c = torch.arange(tile, dtype=torch.float64, device=DEV)
    f = 2.0 * (c - tile / 2.0).abs() / tile
    r = torch.sqrt(f[:, None] ** 2 + f[None, :] ** 2)
    q = 0.5 * (1.0 - torch.cos(float(np.float32(3.1415926)) * r))
    return torch.where(r >= 1.0, torch.zeros_like(r), 1.0 - q ** 3)


def _tile_spectrum64(img, tile):
    """Tile-averaged amplitude spectrum, DC at row tile / 2."""
    ntx, nty, offx, offy, step = _tile_grid(img.shape[1], img.shape[0], tile)
    mask = _round_edge64(tile)
    acc = torch.zeros((tile, tile // 2 + 1), dtype=torch.float64, device=DEV)
    for j in range(nty):
        rows = img[offy + j * step: offy + j * step + tile]
        t = rows[:, offx: offx + (ntx + 1) * step].unfold(1, tile, step).permute(1, 0, 2)
        t = (t - t.mean(dim=(1, 2), keepdim=True)) * mask
        acc += torch.fft.rfft2(t).abs().sum(0)
    return torch.roll(acc / (ntx * nty), tile // 2, 0)


def _unfold(half):
    """Half spectrum [T][T/2+1] -> periodic full plane [T][T], DC at (T/2, T/2)
    along y and column 0 along x."""
    t = half.shape[0]
    rest = torch.roll(torch.flip(half, (0,)), 1, 0)      # row (T - y) mod T
    return torch.cat([half[:, :t // 2], torch.flip(rest[:, 1:t // 2 + 1], (1,))], 1)


def _background64(raw):
    t = raw.shape[0]
    box = int(np.float32(1.0 / 15.0) * np.float32(t))
    if np.float32(box) > np.float32(0.3) * np.float32(t):
        box = int(np.float32(0.3) * np.float32(t))
    box = max(box // 2 * 2 + 1, 7)
    hb = box // 2
    p = torch.sqrt(_unfold(raw))
    s = torch.zeros_like(p)
    for j in range(-hb, hb + 1):
        s += torch.roll(p, -j, 1)
    q = torch.zeros_like(p)
    for j in range(-hb, hb + 1):
        q += torch.roll(s, -j, 0)
    out = raw - (q[:, :t // 2 + 1] / (box * box)) ** 2
    x = np.arange(t // 2 + 1, dtype=np.float32) * np.float32(0.5) / np.float32(t // 2)
    yc = np.arange(t) - t // 2
    fr = np.sqrt(x[None, :] * x[None, :] + (yc * yc).astype(np.float32)[:, None] / np.float32(t * t))
    return torch.where(torch.from_numpy(fr.astype(np.float64) < 0.04).to(DEV), torch.zeros_like(out), out)


def _lowpass64(half):
    """exp(s (kx^2 + ky^2)) on the periodic full plane when its variance is at least 1."""
    m1, m2 = np.float32(float(half.mean())), np.float32(float((half * half).mean()))
    if m2 - m1 * m1 < 1.0:
        return half
    t = half.shape[0]
    k = torch.arange(t, dtype=torch.float64, device=DEV)
    k = torch.where(k > t // 2, k - t, k)
    h = torch.exp(float(np.float32(-10.0 / (2.0 * t * t))) * (k[:, None] ** 2 + k[None, :] ** 2))
    # plane with DC at column t / 2, row t / 2
    full = torch.roll(_unfold(half), t // 2, 1)
    full = torch.fft.ifft2(torch.fft.fft2(full) * h).real
    return torch.roll(full, -(t // 2), 1)[:, :t // 2 + 1]


def _radial64(half):
    """Radial averages over the sample positions of GRadialAvg, which are
    found in single precision."""
    f = np.float32
    t, cx = half.shape
    s = half.cpu().numpy()
    out = np.zeros(cx)
    for r in range(cx):
        n = min(max(int(f(3.1415926) * f(r) + f(0.5)), 1), 180)
        i = np.arange(n, dtype=f)
        rad = (f(-90.0) + i * (f(180.0) / f(n))) * f(0.017453)
        x = (f(r) * np.cos(rad.astype(np.float64)).astype(f) + f(0.5)).astype(np.int64)
        y = (f(r) * np.sin(rad.astype(np.float64)).astype(f) + f(t // 2) + f(0.5)).astype(np.int64) % t
        out[r] = s[y, x].mean()
    return torch.from_numpy(out)


def _net64(p, radial):
    """The network of gctffind_amd/csrc/gctf_net.hpp on p (float64), raw outputs [n][4]."""
    sl = proposal.layer_slices()
    x = radial[:, :256].to(torch.float64)
    u = x[:, 16:]
    u = (u - u.mean(1, keepdim=True)) / u.std(1, unbiased=False, keepdim=True)
    x = torch.cat([torch.zeros_like(x[:, :16]), u], 1)[:, None, :]
    for name, cin in (("conv1", 1), ("conv2", 64), ("conv3", 64), ("conv4", 64)):
        w, b = (p[s] for s in sl[name])
        # the 7 taps as one product over the shifted copies
        xp = torch.nn.functional.pad(x, (3, 3))
        col = torch.stack([xp[:, :, t:t + x.shape[2]] for t in range(7)], 2).reshape(x.shape[0], cin * 7, -1)
        y = torch.relu(torch.matmul(w.reshape(64, cin * 7), col) + b[:, None])
        x = 0.5 * (y[:, :, 0::2] + y[:, :, 1::2])
    w, b = (p[s] for s in sl["fc1"])
    h = torch.relu(x.reshape(x.shape[0], 1024) @ w.reshape(128, 1024).T + b)
    w, b = (p[s] for s in sl["fc2"])
    return h @ w.reshape(4, 128).T + b


def _loss64(o, t):
    t = t.to(torch.float64)
    e0, e1 = o[:, 0] - torch.log(t[:, 0] * 1e-4), o[:, 1] - t[:, 1] * 1e-3
    d2 = 2.0 * (o[:, 2] - torch.deg2rad(t[:, 2]))
    c, w = (t[:, 3] > 0).to(torch.float64), (t[:, 3] != 0).to(torch.float64)
    bce = torch.nn.functional.softplus(o[:, 3]) - c * o[:, 3]
    return (100.0 * e0 ** 2 + 0.25 * e1 ** 2 + 0.05 * (1.0 - torch.cos(d2)) + 0.5 * w * bce).mean()


def exact(case, seed):
    k = case["kind"]
    if k in ("estimate", "list", "search", "grid"):
        return None     # the end of a search: no closed value
    if k in ("spectra", "session"):
        img = _micrographs(case.get("n", 1), case["ny"], case["nx"], case["pix"], seed, case.get("half", False),
                           df=(5000.0, 40000.0))
        out = []
        for im in img:
            raw = _tile_spectrum64(_rescale64(im, case["pix"]), case["tile"])
            half = _lowpass64(_background64(raw))
            if k == "session":
                return dict(raw=raw, half=half)
            out.append(_radial64(half))
        return torch.stack(out)
    radial, target = _radial_rows(case["n"], seed)
    # on the CPU: its batched products take any strides
    radial, target = radial.cpu(), target.cpu()
    if k == "propose":
        return _net64(torch.from_numpy(proposal.load_params()[0]).to(torch.float64), radial)
    p = torch.from_numpy(_params(seed)).to(torch.float64).requires_grad_(True)
    loss = _loss64(_net64(p, radial), target)
    loss.backward()
    g = p.grad
    # AdamW's first step: the moments' corrections leave g and g^2
    new = p.detach() - 3.0e-4 * (g / (g.abs() + 1.0e-8) + 1.0e-4 * p.detach())
    return dict(loss=float(loss), grad=g, params=new)
