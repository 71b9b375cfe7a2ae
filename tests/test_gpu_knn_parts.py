"""Searches for a part of a large set, whose wavefronts are shared out between
the two kernels by the span of their queries: parts that lie together, at
random, mixed, and with repeated rows, against the one-lane search."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,dim,box,f64", [(5300000, 32, 3, None, False), (5300000, 16, 2, None, True),
                                             (5300000, 20, 3, 1.0, True), (4300000, 40, 3, 1.0, False)])
def test_parts_of_large_sets(n, k, dim, box, f64):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine

    print("part", n, k, dim, box, f64, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    p = torch.rand(n, dim, generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32) * 0.9999
    ix = engine.SpatialIndex().build(p, box)
    order, rnd = ix.order(), torch.randperm(n, generator=g, device="cuda")
    nq = n // (4 if k > 32 else 5) - 7
    for q in (order[1000 : 1000 + nq], rnd[:nq], torch.cat([order[: nq // 2], rnd[: nq // 2]]),
              rnd[: nq // 5].repeat(4)):
        q = q.contiguous()
        a, b = (engine.knn_hsml(ix, k, qidx=q, lane=lane) for lane in (False, True))
        (na, da), (nb, db) = (o["nlist"].export(f64=True) for o in (a, b))
        assert torch.equal(na, nb) and torch.equal(da, db)
        assert torch.equal(a["status"], b["status"])
        ha, hb = (o["nlist"].h64().cpu().numpy() for o in (a, b))
        np.testing.assert_allclose(ha, hb, rtol=1e-12, atol=0)
