"""An index or list that grows lets its old memory go before it takes the new."""
import pytest

pytestmark = pytest.mark.gpu


def test_growing_needs_the_larger_block_only():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import engine

    a, b = (torch.rand(n, 3, device="cuda") for n in (600000, 1000000))
    outs = [{"h": torch.empty(len(p), device="cuda")} for p in (a, b)]
    ix, nl = engine.SpatialIndex().build(a), engine.NeighborList()
    engine.knn_hsml(ix, 32, nlist=nl, out=outs[0])
    small = nl._mem.block.numel() + ix._mem.block.numel()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    engine.knn_hsml(ix.build(b), 32, nlist=nl, out=outs[1])
    large = nl._mem.block.numel() + ix._mem.block.numel()
    peak = torch.cuda.max_memory_allocated() - before
    assert large > 1.5 * small
    assert peak <= large - small + (1 << 21)  # (blocks are rounded up)
    got, want = nl.export(f64=True), engine.knn_hsml(engine.SpatialIndex().build(b), 32)["nlist"].export(f64=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
