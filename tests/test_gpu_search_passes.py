"""Search passes in which some micrographs of a batch sit out: the learned
path's fallback pass, whose launches follow from the number that takes part."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N, SIDE, PIX = 32, 1024, 1.2
KEYS = ("df_min", "df_max", "azimuth", "ext_phase", "score", "ctf_res")


def _micrographs(proposal, n):
    d1, d2, az, b, s = proposal.draw_params(np.random.default_rng(41), n, df_lo=6000.0, df_hi=36000.0)
    im = torch.empty((n, SIDE, SIDE), dtype=torch.float32, device="cuda")
    for i in range(n):
        proposal.micrograph_batch(torch, 1, SIDE, SIDE, PIX, d1[i:i + 1], d2[i:i + 1], az[i:i + 1], b[i:i + 1],
                                  s[i:i + 1], 410 + i, out=im[i:i + 1], device="cuda")
    return im


def _best(f, reps=6):
    f()
    best = 1e9
    for _ in range(reps):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def test_fallback_pass_on_part_of_a_batch():
    """Every share of a batch: those that fall back equal the plain search,
    the others the narrowed one, bit for bit.  And the pass for k micrographs
    of the batch, the plain search without the spectra, takes at most a
    quarter longer than the plain call on a batch of k."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf, proposal
    ctx = gctf.Context()
    ctx.set_proposal_params(proposal.load_params()[0])
    im = _micrographs(proposal, 2 * N)
    _, props = ctx.estimate_batch_learned(im.data_ptr(), 2 * N, SIDE, SIDE, PIX, conf_threshold=-1.0, proposals=True)
    # micrographs whose narrowed search settles them: only the threshold sends them back
    keep = [i for i, p in enumerate(props) if not p["fallback"]][:N]
    assert len(keep) == N
    im = im[keep].contiguous()
    args = (im.data_ptr(), N, SIDE, SIDE, PIX)
    plain = ctx.estimate_batch(*args)
    free, props = ctx.estimate_batch_learned(*args, conf_threshold=-1.0, proposals=True)
    assert not any(p["fallback"] for p in props)
    base = _best(lambda: ctx.estimate_batch_learned(*args, conf_threshold=-1.0))
    conf = np.sort([p["confidence"] for p in props])
    report, slow = [], []
    for k in (1, 2, 3, 5, 8, 9, 16, 17, 31, 32):
        thr = 2.0 if k == N else float(0.5 * (conf[k - 1] + conf[k]))
        got, p = ctx.estimate_batch_learned(*args, conf_threshold=thr, proposals=True)
        fb = [q["fallback"] for q in p]
        assert sum(fb) == k
        for i in range(N):
            want = plain[i] if fb[i] else free[i]
            assert all(got[i][key] == want[key] for key in KEYS), (k, i, fb[i], got[i], want)
        t = _best(lambda: ctx.estimate_batch_learned(*args, conf_threshold=thr)) - base
        w = _best(lambda: ctx.estimate_batch(im.data_ptr(), k, SIDE, SIDE, PIX))
        report.append((k, round(t * 1e6), round(w * 1e6)))
        if t > 1.25 * w:
            slow.append(report[-1])
    print("fallbacks, us of the pass, us of a plain batch:", report)
    assert not slow, slow


def test_small_blocks_on_a_large_batch():
    """A search blocking of 2 on a batch whose blocks of 2 do not fit the chip:
    the same results, and no slower than 4 by more than a tenth."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gctffind_amd import gctf, proposal
    im = _micrographs(proposal, N)
    ctx = gctf.Context()
    run = lambda: ctx.estimate_batch(im.data_ptr(), N, SIDE, SIDE, PIX)
    res, t = {}, {}
    for block in (4, 2, 8, 16):
        ctx.tune(search_block=block)
        res[block], t[block] = run(), _best(run)
    print("search block: us", {b: round(x * 1e6) for b, x in t.items()})
    assert res[2] == res[4] == res[8] == res[16]
    assert t[2] <= 1.1 * t[4], t
