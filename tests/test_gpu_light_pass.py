"""Passes of at most 2^18 particles take the light stages (one-launch class
partition and list scans, counts kept on the device); larger ones the general
stages.  A particle of zero quantity deposits nothing without calc_mean, so a
set and the same set with one such particle more, on either side of the line,
must give the same image: sums of the same FP64 terms in another order, 1e-12
of the largest pixel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LINE = 1 << 18


def _set(n, npix, seed, hmax):
    r = np.random.default_rng(seed)
    x = r.uniform(-0.5, 0.5, (n, 3))
    h = np.exp(r.uniform(np.log(0.3 / npix), np.log(hmax / npix), n))
    m, rho, w, q = (r.uniform(0.5, 2.0, n) for _ in range(4))
    return x, h, m, rho, q, w


@pytest.mark.parametrize("dims,npix,hmax", [(2, 200, 40.0), (2, 65, 3.0), (3, 30, 7.0),
                                            (3, 100, 1.5)])
def test_light_and_general_passes_agree(s2g, dims, npix, hmax):
    x, h, m, rho, q, w = _set(LINE + 1, npix, 5 + dims + npix, hmax)
    q[-1] = 0.0
    img, st = [], []
    for n in (LINE, LINE + 1):
        s = {}
        img.append(s2g.deposit(x[:n], h[:n], m[:n], rho[:n], q[:n], w[:n], npix=npix,
                               len2pix=float(npix), dimensions=dims, kernel=s2g.WendlandC4(dims),
                               calc_mean=False, stats=s))
        st.append(s)
    for k in ("n_small", "n_large", "n_large_exact", "n_pairs"):
        assert st[0][k] == st[1][k], k
    assert st[1]["n_skipped"] == st[0]["n_skipped"] + 1
    for k in range(2):
        np.testing.assert_allclose(img[0][:, k], img[1][:, k], rtol=0,
                                   atol=1e-12 * np.abs(img[1][:, k]).max())


@pytest.mark.parametrize("nq", [1, 3])
def test_light_batch_with_empty_and_one_sided_maps(s2g, nq):
    """Maps without particles (first, in the middle, last), with only small or
    only large footprints and with all of one's particles skipped share a light
    pass: each map equals its own call."""
    import torch
    r = np.random.default_rng(nq)
    maps, singles = [], []
    for n, npix, lo, hi in [(0, 40, 1, 2), (700, 70, 0.4, 3.0), (0, 33, 1, 2),
                            (300, 130, 20.0, 60.0), (255, 64, 0.4, 40.0), (257, 129, 1.0, 30.0),
                            (40, 20, 1.0, 3.0), (0, 64, 1, 2)]:
        x = r.uniform(-0.5, 0.5, (n, 3))
        h = np.exp(r.uniform(np.log(lo / npix), np.log(hi / npix), n))
        m, rho, w = (r.uniform(0.5, 2.0, n) for _ in range(3))
        q = r.uniform(0.5, 2.0, (n, nq)) * (n != 40)
        t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, h, m, rho, q, w)]
        out = torch.empty((nq + 1) * npix * npix, dtype=torch.float64, device="cuda")
        maps.append(dict(pos=t[0], hsml=t[1], m=t[2], rho=t[3], bin_q=t[4], weights=t[5], out=out,
                         n=n, nq=nq, npix=npix, len2pix=float(npix), kernel=s2g.Cubic(2)))
        singles.append(s2g.deposit(x, h, m, rho, q if nq > 1 else q[:, 0], w, npix=npix,
                                   len2pix=float(npix), kernel=s2g.Cubic(2), calc_mean=False))
    s2g.deposit_batch_device(maps, dtype="f64")
    for d, ref in zip(maps, singles):
        got = d["out"].cpu().numpy().reshape(ref.shape, order="F")
        np.testing.assert_allclose(got, ref, rtol=0, atol=1e-12 * max(np.abs(ref).max(), 1e-300))


@pytest.mark.parametrize("n", [63, 64, 65, 1000, 40000])
def test_small_item_floor(s2g, orc, n):
    """Small footprints piled on one tile, so that its list is cut into items
    of a quarter of the least item (few particles) or half of it (40,000).
    Tolerance: the 2D deposit's (rel-L1 1e-5, conservation 1e-6)."""
    npix = 64
    r = np.random.default_rng(n)
    x = r.uniform(-0.2, 0.0, (n, 3))
    h = r.uniform(0.5, 6.0, n) / npix
    m, rho, w, q = (r.uniform(0.5, 2.0, n) for _ in range(4))
    gpu = s2g.deposit(x, h, m, rho, q, w, npix=npix, len2pix=float(npix), dimensions=2,
                      kernel=s2g.WendlandC4(2), calc_mean=False)
    ref = orc.cic_mapping_2D(x, h, m, rho, q, w, npix, float(npix), "wendlandc4", 2, False)
    for k in range(2):
        assert np.abs(gpu[:, k] - ref[:, k]).sum() <= 1e-5 * np.abs(ref[:, k]).sum(), k
    assert abs(gpu[:, 1].sum() / ref[:, 1].sum() - 1) <= 1e-6


@pytest.mark.parametrize("dims,npix,n,nq,hmax", [(2, 256, 65536, 1, 24.0), (2, 777, 100000, 3, 60.0),
                                                 (3, 100, 100000, 1, 7.0)])
def test_light_pass_memory_follows_its_pairs(s2g, dims, npix, n, nq, hmax):
    """A light pass holds what its (tile, particle) pairs need, not what every
    large footprint on every tile would: the partial sums of one work item per
    tile and one per least item size, a quarter or 16 MB to spare, and per
    particle and pixel less than 400 and 100 bytes."""
    import torch
    from sph2grid import _lib
    x, h, m, rho, q, w = _set(n, npix, 7, hmax)
    q = np.stack([q] * nq, 1) if nq > 1 else q
    ctx = _lib.Context()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    st = {}
    s2g.deposit(x, h, m, rho, q, w, npix=npix, len2pix=float(npix), dimensions=dims,
                kernel=s2g.Cubic(dims), calc_mean=False, context=ctx, stats=st)
    held = free - torch.cuda.mem_get_info()[0]
    ctx.close()
    side, planes, least = (64, nq + 1, 64 if nq < 2 else 128) if dims == 2 else (16, 2, 64)
    tiles = (-(-npix // side)) ** dims
    items = min(tiles, st["n_pairs"]) + min(-(-st["n_pairs"] // least), 16 * 256)
    partial = items * planes * 8 * side ** dims
    assert 0 < st["n_pairs"] < st["n_large"] * tiles / 2
    bound = 1.25 * partial + (16 << 20) + 400 * n + 100 * (nq + 1) * npix ** dims
    print(f"[light memory {dims}d {npix}] held {held >> 20} MB, partials {partial >> 20} MB, "
          f"{st['n_pairs']} pairs", flush=True)
    assert held <= bound, (held, bound)
