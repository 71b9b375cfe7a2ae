"""Smoothing lengths of sets where each particle has a few others next to it, so
that n(h) is flat at the root and the float32 solve is far off: both searches
against bisection on the float64 distances of the positions as the index holds
them (float64 ones as the sum of two floats, 2^-48 of the coordinate: a row's
slope divides that too), and rows without a root against r_1."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NORM = {2: 40 / 7, 3: 32 / 3}


def _kernel(q):
    return np.where(q <= 0.5, 1 - 6 * q * q * (1 - q), 2 * np.clip(1 - q, 0, None) ** 3)


@pytest.mark.parametrize("lane", [False, True])
@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("k,dim,group,box", [(32, 3, 3, None), (32, 3, 3, 1.0), (64, 3, 6, None), (100, 3, 10, None),
                                             (20, 2, 4, None), (8, 3, 1, None), (8, 3, 1, 1.0)])
def test_flat_rows_match_bisection(k, dim, group, box, f64, lane):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import ST_COUNT, ST_HSML_NOCONV

    print("flat rows", k, dim, group, box, f64, lane, flush=True)
    rng = np.random.default_rng(k + group)
    m = 1500
    pos = np.repeat(0.01 + 0.98 * rng.random((m, dim)), group, axis=0)
    pos += 0.002 * m ** (-1 / dim) * rng.random(pos.shape) * (group > 1)  # 0.2% of the spacing
    p = torch.from_numpy(pos if f64 else pos.astype(np.float32)).cuda()
    ix = engine.SpatialIndex().build(p, box)
    nl = engine.knn_hsml(ix, k, lane=lane)
    st = nl["status"].cpu().numpy()
    assert not (st & (ST_COUNT | ST_HSML_NOCONV)).any()
    ngb = nl["nlist"].export(f64=True)[0].cpu().numpy()
    x = p.cpu().numpy().astype(np.float32)
    x = x.astype(np.float64) + (p.cpu().numpy() - x).astype(np.float32)
    d = x[ngb] - x[:, None]
    if box:
        d -= np.round(d / box) * box
    r = np.sort(np.sqrt((d**2).sum(-1)), 1)
    h = nl["nlist"].h64().cpu().numpy()
    if k < NORM[dim]:
        np.testing.assert_allclose(h, r[:, 1], rtol=1e-15)
        return
    lo, hi = r[:, 1], r[:, -1] / (1 - (2 * NORM[dim]) ** (-1 / 3))
    for _ in range(64):
        x = (lo + hi) / 2
        big = NORM[dim] * _kernel(r / x[:, None]).sum(1) > k
        lo, hi = np.where(big, lo, x), np.where(big, x, hi)
    want = (lo + hi) / 2
    q = np.minimum(r / want[:, None], 1.0)
    p_ = NORM[dim] * 6 * (((1 - q) ** 2 - np.clip(1 - 2 * q, 0, None) ** 2) * q).sum(1)
    # n(h) to 16 eps a term in each of the two solves, and the last step's 1e-13
    tol = 1e-13 + 32 * np.finfo(float).eps * k / p_
    bad = np.abs(h - want) > tol * want
    print("  worst", (np.abs(h - want) / want).max(), "beyond", bad.sum(), "smallest slope", p_.min(), flush=True)
    assert not bad.any()
