"""Radius seeds that make wavefronts of the one-lane-per-query search leave
their rows to the one-wavefront-per-query search in the second launch only: on a
cubic lattice where every row but those of its edges is ambiguous (k = 12: the
12th and 13th neighbours tie), the rows inside each block of 4^3 have a seed that holds
their neighbours, the others one that misses them.  The first launch finishes
the former; the second, without seeds, meets the periodic faces or more leaves
than the record holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M = 32  # lattice points per axis: Hilbert blocks of 4^3 are the wavefronts


@pytest.mark.parametrize("box,small", [(None, False), (None, True), (1.0, False), (1.0, True)])
@pytest.mark.parametrize("f64", [False, True])
def test_seeded_lattice_equals_unseeded(box, small, f64):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import ST_AMBIGUOUS, ST_RADIUS_MISS

    print("seeded lattice", box, small, f64, flush=True)
    k = 12
    g = np.stack(np.meshgrid(*[np.arange(M)] * 3, indexing="ij"), -1).reshape(-1, 3)
    inside = np.isin(g % 4, (1, 2)).all(1)
    order = np.random.default_rng(0).permutation(len(g))
    g, inside = g[order], inside[order]
    p = torch.from_numpy(((g + 0.5) / M).astype(np.float64 if f64 else np.float32)).cuda()
    sr = torch.from_numpy((np.where(inside, 1.45, 0.3) / M).astype(np.float32)).cuda()
    ix = engine.SpatialIndex().build(p, box)
    plain = engine.knn_hsml(ix, k)
    edge = ((g == 0) | (g == M - 1)).sum(1) == 2
    assert bool(((plain["status"].cpu().numpy() & ST_AMBIGUOUS) != 0)[~edge].all())
    got = engine.knn_hsml(ix, k, seed_r=sr, small_record=small)
    (na, da), (nb, db) = (o["nlist"].export(f64=True) for o in (plain, got))
    assert torch.equal(na, nb) and torch.equal(da, db)
    assert torch.equal(plain["nlist"].export()[1], got["nlist"].export()[1])
    assert torch.equal(plain["status"], got["status"] & ~ST_RADIUS_MISS)
    assert np.array_equal((got["status"] & ST_RADIUS_MISS).cpu().numpy() != 0, ~inside)
    # float64 sums of 12 terms in two orders over a slope h n'(h) > 1
    np.testing.assert_allclose(got["nlist"].h64().cpu().numpy(), plain["nlist"].h64().cpu().numpy(), rtol=1e-12)
