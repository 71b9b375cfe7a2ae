"""Positions so far apart that squared distances overflow float32: a few clumps
whose members lie close, and single points of which some have fewer than k
others within 1.8e19.  Both searches against float64 distances of all pairs,
and against each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 3000])
@pytest.mark.parametrize("k", [20, 32])
@pytest.mark.parametrize("box", [None, 4e22])
@pytest.mark.parametrize("f64", [False, True])
def test_squared_distances_beyond_float32(n, k, box, f64):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import ST_BAND_OVERFLOW, ST_COUNT, ST_HSML_NOCONV

    print("overflow", n, k, box, f64, flush=True)
    rng = np.random.default_rng(n + k)
    pos = rng.random((n, 3)) * 3e22 + 5e21
    m = n // 4
    pos[:m] = pos[0] + rng.standard_normal((m, 3)) * 1e18          # near each other
    pos[m : 2 * m] = pos[m] + rng.standard_normal((m, 3)) * 1e19   # some pairs overflow
    pos = pos[rng.permutation(n)].astype(np.float64 if f64 else np.float32)
    d = pos[:, None].astype(np.float64) - pos[None].astype(np.float64)
    if box:
        d = np.where(np.abs(d) > box / 2, box - np.abs(d), d)
    r = np.sqrt((d**2).sum(-1))
    want = np.argsort(r, 1, kind="stable")[:, :k]
    ix = engine.SpatialIndex().build(torch.from_numpy(pos).cuda(), box)
    res = []
    for lane in (False, True):
        o = engine.knn_hsml(ix, k, lane=lane)
        ngb, dist = o["nlist"].export(f64=True)
        st = o["status"].cpu().numpy()
        assert not (st & ST_COUNT).any()
        assert np.array_equal(ngb.cpu().numpy(), want)
        np.testing.assert_allclose(dist.cpu().numpy(), np.take_along_axis(r, want, 1), rtol=1e-15)
        res.append((st & ~(ST_HSML_NOCONV | ST_BAND_OVERFLOW), o["nlist"].h64().cpu().numpy()))
    assert np.array_equal(res[0][0], res[1][0])
    (_, ha), (_, hb) = res
    assert np.array_equal(np.isfinite(ha), np.isfinite(hb))
    ok = np.isfinite(ha)
    np.testing.assert_allclose(ha[ok], hb[ok], rtol=1e-11)
