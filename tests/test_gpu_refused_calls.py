"""Calls that the library refuses leave the objects they were given as they
were."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _set(n=400):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine

    ix = engine.SpatialIndex().build(torch.from_numpy(np.random.default_rng(n).random((n, 3)).astype(np.float32)).cuda())
    nl = engine.knn_hsml(ix, 8)["nlist"]
    return engine, ix, nl, nl.export(f64=True), nl.h64()


def _same(nl, rows, h):
    got = nl.export(f64=True)
    assert torch.equal(got[0], rows[0]) and torch.equal(got[1], rows[1]) and torch.equal(nl.h64(), h)


@pytest.mark.parametrize("k,error", [(0, ValueError), (1, ValueError), (129, NotImplementedError),
                                     (10**9, NotImplementedError), (127, ValueError)])
def test_refused_k_keeps_the_list(k, error):
    engine, ix, nl, rows, h = _set(100)
    big = engine.SpatialIndex().build(torch.rand(100000, 3, device="cuda"))
    with pytest.raises(error):
        engine.knn_hsml(ix, k, nlist=nl)
    _same(nl, rows, h)
    if error is NotImplementedError or k < 2:
        with pytest.raises(error):
            engine.knn_hsml(big, k, nlist=nl)
        _same(nl, rows, h)
    with pytest.raises(ValueError):
        engine.knn_hsml(ix, 8, qidx=torch.empty(0, dtype=torch.int64, device="cuda"), nlist=nl)
    _same(nl, rows, h)


def test_refused_subset_keeps_the_lists():
    engine, ix, nl, rows, h = _set()
    q = torch.arange(0, 400, 3, device="cuda")
    many = torch.arange(400, device="cuda").repeat(50)
    for qidx in (q, many):
        with pytest.raises(ValueError):
            engine.nlist_subset(nl, qidx, nlist=nl)
        _same(nl, rows, h)
    sub = engine.nlist_subset(nl, q)["nlist"]
    part, ph = sub.export(f64=True), sub.h64()
    with pytest.raises(ValueError):
        engine.nlist_subset(sub, many, nlist=nl)  # a masked list is no source
    _same(nl, rows, h)
    with pytest.raises(ValueError):
        engine.nlist_subset(sub, q, nlist=sub)
    _same(sub, part, ph)
    other = engine.nlist_subset(nl, many, nlist=sub)["nlist"]  # and a larger one still grows
    assert torch.equal(other.export(f64=True)[0], rows[0][many])


def test_refused_build_keeps_the_index():
    engine, ix, nl, rows, h = _set()
    with pytest.raises(KeyError):
        ix.build(torch.rand(100000, 4, device="cuda"))
    with pytest.raises(ValueError):
        ix.build(torch.rand(0, 3, device="cuda"))
    _same(nl, rows, h)
    again = engine.knn_hsml(ix, 8)["nlist"]
    _same(again, rows, h)
