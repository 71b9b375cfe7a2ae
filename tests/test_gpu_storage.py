"""Caller storage of an index that a later build outgrows, and storage that is
not aligned: errors, and nothing built before is used afterwards."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_refused_rebuild_leaves_the_index_empty():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import lib

    p = torch.from_numpy(np.random.default_rng(0).random((100000, 3)).astype(np.float32)).cuda()
    n0, k = 1000, 32
    ix, nl = engine.SpatialIndex(), engine.NeighborList()
    ctx = engine.context(p.device)
    mem = torch.empty(lib.mhip_index_bytes(n0, 0), dtype=torch.uint8, device="cuda")
    assert lib.mhip_index_storage(ix.h, ctypes.c_void_p(mem.data_ptr()), mem.numel()) == 0

    def build(n):
        return lib.mhip_index_build(ctx, ix.h, engine.ptr(p), 0, n, 3, -1.0)

    def search():
        return lib.mhip_knn_hsml(ctx, ix.h, None, 0, k, None, None, None, None, None, None, None, 0, nl.h)

    h = torch.empty(n0, dtype=torch.float64, device="cuda")
    order = torch.empty(n0, dtype=torch.int32, device="cuda")
    f, d = torch.rand(n0, 1, device="cuda"), torch.empty(n0, 1, 3, device="cuda")
    assert build(n0) == 0 and search() == 0 and lib.mhip_nlist_hsml(ctx, nl.h, engine.ptr(h)) == 0
    assert build(len(p)) == -1
    n = ctypes.c_int64(-1)
    assert lib.mhip_index_info(ix.h, ctypes.byref(n), None, None, None) == 0
    assert n.value == 0  # (the calls below must not reach the device)
    assert search() == -1
    assert lib.mhip_index_order(ctx, ix.h, engine.ptr(order)) == -1
    assert lib.mhip_nlist_hsml(ctx, nl.h, engine.ptr(h)) == -1
    assert lib.mhip_apply_D(ctx, nl.h, engine.ptr(f), 0, n0, 1, 1, 1, engine.ptr(d), None, None) == -1
    assert build(n0) == 0 and search() == 0 and lib.mhip_nlist_hsml(ctx, nl.h, engine.ptr(h)) == 0


def test_storage_alignment_is_checked():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import lib

    mem = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    ix, nl = engine.SpatialIndex(), engine.NeighborList()
    for fn, o in ((lib.mhip_index_storage, ix), (lib.mhip_nlist_storage, nl)):
        for off in (1, 4, 8):
            assert fn(o.h, ctypes.c_void_p(mem.data_ptr() + off), 1 << 16) == -1
        assert fn(o.h, ctypes.c_void_p(mem.data_ptr() + 16), 1 << 16) == 0
        assert fn(o.h, None, 0) == 0


@pytest.mark.parametrize("bad", ["nan", "outside"])
def test_failed_build_leaves_the_index_empty(bad):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine
    from meshoid_amd._lib import lib

    p = torch.rand(1000, 3, device="cuda")
    ix = engine.SpatialIndex().build(p, 1.0)
    want = engine.knn_hsml(ix, 8)["nlist"].export(f64=True)
    q = torch.rand(50000, 3, device="cuda")
    q[77] = float("nan") if bad == "nan" else 1.5
    with pytest.raises(ValueError):
        ix.build(q, 1.0)
    n = ctypes.c_int64(-1)
    assert lib.mhip_index_info(ix.h, ctypes.byref(n), None, None, None) == 0
    assert n.value == 0  # (outputs of 1000 rows below: the calls must not reach the device)
    with pytest.raises(ValueError):
        engine.knn_hsml(ix, 8)
    with pytest.raises(ValueError):
        engine.nearest(ix, torch.rand(10, 3, device="cuda", dtype=torch.float64))
    got = engine.knn_hsml(ix.build(p, 1.0), 8)["nlist"].export(f64=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
