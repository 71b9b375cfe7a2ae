"""Curl and Div index their argument with the particle mask: what an array of
indices cannot index is refused, with the default mask too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_vector_fields_are_arrays():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from meshoid_amd import Meshoid

    rng = np.random.default_rng(0)
    M, v = Meshoid(rng.random((500, 3))), rng.random((500, 3))
    for f in (M.Curl, M.Div):
        with pytest.raises(TypeError):
            f(v.tolist())
        for bad in (v[:499], np.float64(1.0)):
            with pytest.raises(IndexError):
                f(bad)
        want = f(v)
        assert np.array_equal(f(np.concatenate([v, v])), want)
        t = torch.from_numpy(v).cuda()
        assert torch.equal(f(torch.cat([t, t])), f(t))
        assert np.array_equal(f(np.asfortranarray(v)), want)
