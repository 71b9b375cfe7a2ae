"""The one-wavefront-per-query search (mhip_knn_wave.hip) against the
one-lane-per-query kernel on the same sets: neighbour rows, distances and
status bits equal, smoothing lengths to the rounding of their float64 sums
(k <= 128 terms of at most 2 each, summed in two orders: below 1e-12)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # n, k, dim, periodic box, float64: one leaf; k = n; the edges of the
    # member registers (32, 64, 65, 128) and of the tree's depth (128, 1024,
    # 8192 particles); one slot per wavefront and four (n > 32768)
    (5, 2, 1, None, False), (16, 16, 2, None, True), (33, 33, 3, None, False), (100, 64, 3, 1.0, True),
    (128, 128, 3, None, True), (129, 65, 2, 1.0, False), (1000, 32, 3, 1.0, False), (1025, 48, 1, 1.0, True),
    (8192, 20, 2, None, False), (8207, 100, 3, 1.0, True), (40001, 32, 3, None, True), (40001, 128, 3, 1.0, False),
    (40013, 65, 3, None, False), (70000, 64, 3, 1.0, True),
]


@pytest.mark.parametrize("n,k,dim,box,f64", CASES)
@pytest.mark.parametrize("masked", [False, True])
def test_wave_search_equals_lane_search(n, k, dim, box, f64, masked):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import ST_COUNT

    print("wave search", n, k, dim, box, f64, masked, flush=True)
    rng = np.random.default_rng(n + k)
    pos = rng.random((n, dim))
    pos[: n // 3] = 0.9 + 0.1 * pos[: n // 3]  # a dense corner, against the faces when periodic
    if n >= 1000:
        pos[n // 2 : n // 2 + 300] = pos[n // 2]  # more coincident points than the buffer keeps
    p = torch.from_numpy(pos if f64 else np.minimum(pos, 0.99999).astype(np.float32)).cuda()
    ix = engine.SpatialIndex().build(p, box)
    q = torch.from_numpy(rng.permutation(n)[: max(1, n // 5)].astype(np.int64)).cuda() if masked else None
    out = [engine.knn_hsml(ix, k, qidx=q, lane=lane) for lane in (False, True)]
    (na, da), (nb, db) = (o["nlist"].export(f64=True) for o in out)
    fa, fb = (o["nlist"].export()[1] for o in out)
    assert torch.equal(out[0]["status"], out[1]["status"])
    # rows with more float64 ties at the k-th than the resolver holds (k > 32)
    # are flagged and padded: their lists are not a result
    full = (out[0]["status"] & ST_COUNT) == 0
    assert torch.equal(na[full], nb[full]) and torch.equal(da[full], db[full]) and torch.equal(fa[full], fb[full])
    ha, hb = (o["nlist"].h64().cpu().numpy() for o in out)
    # rows of coincident points have no root (both solves end at tiny values)
    ok = (da.cpu().numpy()[:, k // 8 + 1] > 0) & full.cpu().numpy()
    np.testing.assert_allclose(ha[ok], hb[ok], rtol=1e-12, atol=0)
