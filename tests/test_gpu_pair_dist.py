"""Precision of the pair distances behind the kernel average: a field that is
zero but on a few particles leaves single weights, and near r = h a weight
magnifies an error of the distance by 3 / (1 - q).

Bound: the root 1.7e-16, 1 / h, the product, and the reference's own root and
quotient half an ulp each: below 1e-15 of q and of 1 - q together, so
|dW| <= |W'| 1e-15, and k + 8 roundings of the two sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [None, 1.0])
def test_weights_near_the_edge(box):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine

    print("weights near the edge", box, flush=True)
    n, k = 60000, 32
    rng = np.random.default_rng(5)
    p = torch.from_numpy(np.minimum(rng.random((n, 3)), 0.99999).astype(np.float32)).cuda()
    f = (rng.random(n) < 0.02).astype(np.float64)
    nl = engine.knn_hsml(engine.SpatialIndex().build(p, box), k)["nlist"]
    ngb, dist = (x.cpu().numpy() for x in nl.export(f64=True))
    h = nl.h64().cpu().numpy()
    got = engine.kernel_average(nl, torch.from_numpy(f).cuda()).cpu().numpy()
    q = np.minimum(dist / h[:, None], 1.0)
    a, b = 1 - q, np.clip(1 - 2 * q, 0, None)
    w = np.where(q <= 0.5, 1 + 6 * q * q * (q - 1), 2 * a**3)
    slope = 6 * (a * a - b * b)
    sw, fn = w.sum(1), f[ngb]
    want = (w * fn).sum(1) / sw
    tol = (slope * fn).sum(1) / sw * 1e-15 + want * ((slope / w.clip(1e-300) * w).sum(1) / sw * 1e-15
                                                     + (k + 8) * np.finfo(float).eps)
    some = (fn.sum(1) == 1) & ((fn * a).sum(1) < 0.05) & (want > 0)
    assert some.sum() > 500
    err = np.abs(got - want)
    print("  rows", some.sum(), "largest error over its bound", (err[some] / tol[some]).max(), flush=True)
    assert (err <= tol)[some].all()
