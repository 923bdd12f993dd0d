"""The 3D small scatter on special values, with sets dense enough, and boxes
large enough, that the windowed kernel takes them (csrc/k_small3.h)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NPIX = 18


def _set(n, seed, lo=0.0, hi=NPIX):
    """n particles centred in [lo, hi]^3 voxels, boxes of 7 or 8 voxels a side."""
    r = np.random.default_rng(seed)
    x = (r.uniform(lo, hi, (n, 3)) - 0.5 * NPIX) / NPIX
    h = 3.4 / NPIX * r.uniform(0.95, 1.0, n)
    m, rho, w, q = (r.uniform(0.5, 2.0, n) for _ in range(4))
    return [x, h, m, rho, q, w]


def _deposit(s2g, p):
    st = {}
    out = s2g.deposit(*p, npix=NPIX, len2pix=float(NPIX), dimensions=3,
                      kernel=s2g.WendlandC4(3), calc_mean=False, stats=st)
    assert st["n_large"] == 0 and st["n_small"] >= 32 * 8
    return out


def _box(c, h):
    lo = np.clip(np.floor(np.asarray(c) - h).astype(int), 0, NPIX - 1)
    hi = np.clip(np.floor(np.asarray(c) + h).astype(int), 0, NPIX - 1)
    g = np.indices((NPIX,) * 3)
    return np.all([(g[d] >= lo[d]) & (g[d] <= hi[d]) for d in range(3)], axis=0).ravel(), hi - lo + 1


@pytest.mark.parametrize("bad", ["weight inf", "weight nan", "rho 0"])
@pytest.mark.parametrize("centre,h,side", [
    ((8.5, 8.5, 8.5), 3.4, (7, 7, 7)),
    ((8.5, 8.5, 8.5), 2.4, (5, 5, 5)),
    ((8.5, 8.5, 8.5), 1.4, (3, 3, 3)),
    ((-0.9, -2.9, -2.9), 3.4, (3, 1, 1)),   # cut by three faces
    ((9.9, 18.9, 18.9), 3.4, (8, 3, 3)),
    ((-0.9, 19.9, 19.9), 3.4, (3, 2, 2)),
])
def test_scale_that_is_not_finite(s2g, centre, h, side, bad):
    """A particle whose scale is not finite spoils the voxels of its own box
    and no others."""
    p = _set(3000, 11)
    k = 1234
    p[0][k] = (np.array(centre) - 0.5 * NPIX) / NPIX
    p[1][k] = h / NPIX
    if bad == "rho 0":
        p[3][k] = 0.0
    else:
        p[5][k] = np.inf if bad == "weight inf" else np.nan
    inside, got_side = _box(centre, h)
    assert tuple(got_side) == side
    got = _deposit(s2g, p)
    ref = _deposit(s2g, [np.delete(a, k, 0) for a in p])
    assert not np.isfinite(got[inside, 1]).all()
    for c in range(2):
        # two orders of at most 3000 FP64 sums of one sign: 3000 * 1.1e-16
        np.testing.assert_allclose(got[~inside, c], ref[~inside, c], rtol=0,
                                   atol=1e-12 * ref[:, c].max())


@pytest.mark.parametrize("q0", [np.inf, -np.inf, np.nan])
def test_zero_weight_of_a_small_box(s2g, q0):
    """Particles of weight 0 in boxes of one to eight voxels (eight to a wave)
    add nothing, whatever their quantity, among large boxes that share their
    voxels."""
    p = _set(3000, 12)
    p[1][::5] = 0.4 / NPIX
    p[5][::10], p[4][::10] = 0.0, q0
    got = _deposit(s2g, p)
    keep = np.arange(3000) % 10 != 0
    ref = _deposit(s2g, [a[keep] for a in p])
    for c in range(2):
        # two orders of at most 3000 FP64 sums of one sign: 3000 * 1.1e-16
        np.testing.assert_allclose(got[:, c], ref[:, c], rtol=0, atol=1e-12 * ref[:, c].max())


def test_weights_that_cancel(s2g, orc):
    """Two particles of equal geometry and opposite weights: their voxels' sum
    of weights is exactly 0, their sum of quantities is not.  (The rest of the
    set stays clear of them, so that no other sum rounds theirs.)"""
    p = _set(3000, 13, 0.0, 8.0)
    c, h = (14.4, 14.3, 14.6), 2.0
    for k, w, q in ((700, 1.0, 3.0), (2100, -1.0, 1.0)):
        p[0][k] = (np.array(c) - 0.5 * NPIX) / NPIX
        p[1][k], p[2][k], p[3][k], p[4][k], p[5][k] = h / NPIX, 1.0, 1.0, q, w
    inside, _ = _box(c, h)
    got = _deposit(s2g, p)
    ref = orc.cic_mapping_3D(*p, NPIX, float(NPIX), "wendlandc4", 3, False)
    assert (got[inside, 1] == 0.0).all() and ref[inside, 0].max() > 0.0
    # FP64 in both, boxes of 125 voxels: a few hundred roundings of 1.1e-16
    np.testing.assert_allclose(got[inside, 0], ref[inside, 0], rtol=0,
                               atol=1e-12 * ref[inside, 0].max())
