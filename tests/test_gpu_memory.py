"""Device memory of indices and lists from torch's allocator, host arrays made
on access, and the row outputs and status word that Meshoid reads."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _pos(n=5000, seed=0, dtype=np.float32):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.from_numpy(np.random.default_rng(seed).random((n, 3)).astype(dtype)).cuda()


def test_default_mask_and_masses_are_host_arrays_on_access():
    from meshoid_amd import Meshoid

    M = Meshoid(_pos())
    rho, h = M.density.copy(), M.kernel_radius
    np.testing.assert_allclose(rho, 32 / (4 * np.pi / 3 * h**3), rtol=1e-15)
    assert np.array_equal(M.particle_mask, np.arange(5000)) and np.array_equal(M.m, np.ones(5000))
    M.m[:] = 2.0  # the array handed out is the one used
    M.TreeUpdate()
    np.testing.assert_allclose(M.density, 2 * rho, rtol=1e-15)
    np.testing.assert_allclose(M.vol * M.density, 2.0, rtol=1e-15)
    with pytest.raises(IndexError):
        Meshoid(_pos(), particle_mask=np.array([5, 9, 7]))  # m[mask][mask], as the reference


@pytest.mark.parametrize("k,order", [(32, 1), (48, 2)])
def test_status_word_is_the_or_of_the_rows(k, order):
    from meshoid_amd import engine

    p = _pos(3000, 1)
    p[:200, 1:] = 0.5  # rows on a line: rank-deficient fits
    p[:200, 0] = torch.arange(200, device="cuda") * 1e-5
    ix = engine.SpatialIndex().build(p)
    nl = engine.knn_hsml(ix, k)["nlist"]
    for f in (p[:, :1].contiguous(), p.double()):
        d1, _, st = engine.apply_D(nl, f, order=order)
        word = torch.full((1,), 12345, dtype=torch.int32, device="cuda")
        e1, _, none = engine.apply_D(nl, f, order=order, any_status=word)
        want = 0
        for v in torch.unique(st).tolist():
            want |= v
        assert want != 0 and int(word) == want and none is None
        assert torch.equal(d1.isnan(), e1.isnan()) and torch.equal(d1.nan_to_num(), e1.nan_to_num())


def test_storage_too_small_is_an_error():
    from meshoid_amd import engine
    from meshoid_amd._lib import lib

    p = _pos()
    ix = engine.SpatialIndex()
    small = torch.empty(1024, dtype=torch.uint8, device="cuda")
    assert lib.mhip_index_storage(ix.h, ctypes.c_void_p(small.data_ptr()), 1024) == 0
    ctx = engine.context(p.device)
    assert lib.mhip_index_build(ctx, ix.h, engine.ptr(p), 0, 5000, 3, -1.0) == -1
    assert lib.mhip_index_storage(ix.h, None, 0) == 0  # the library allocates again
    assert lib.mhip_index_build(ctx, ix.h, engine.ptr(p), 0, 5000, 3, -1.0) == 0


def test_dropped_objects_and_streams():
    """Objects made on one stream, used on another and dropped at once: the
    memory is not handed out again before the work that reads it."""
    from meshoid_amd import engine

    p = _pos(200000, 3)
    f = (p[:, :1] * 2).contiguous()

    def once():
        ix = engine.SpatialIndex().build(p)
        nl = engine.knn_hsml(ix, 32, keep_dist=False)["nlist"]
        return engine.apply_D(nl, f)[0]

    want = once()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(5):
        a.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(a):
            ix = engine.SpatialIndex().build(p)
            nl = engine.knn_hsml(ix, 32, keep_dist=False)["nlist"]
        b.wait_stream(a)
        with torch.cuda.stream(b):
            got = engine.apply_D(nl, f)[0]
        size = nl._mem.block.numel()
        del ix, nl
        with torch.cuda.stream(a):  # would take the list's block if it were free
            torch.empty(size, dtype=torch.uint8, device="cuda").fill_(255)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
