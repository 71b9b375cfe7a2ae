"""radtransfer (src/meshoid/radiation/radtransfer.py:11-177) on the GPU
against the oracle's sequential farthest-first sweep
(tests/test_radtransfer_oracle.py pins it): per-tile segments composed
exactly, one or several bands, scalar / per-band / per-pixel backgrounds,
optically thick and thin particles, particles off the image, clumps whose
tiles span many chunks, no particle on the image."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n,nf,res,i0", [(3000, 1, 32, 0.0), (8000, 3, 48, "band"), (20000, 2, 100, "pixel")])
def test_radtransfer_matches_oracle(oracle, n, nf, res, i0):
    _torch()
    import meshoid_amd

    rng = np.random.default_rng(n)
    x = rng.normal(0.0, 3.0, (n, 3))
    m = rng.random(n) + 0.1
    h = np.exp(rng.normal(-0.3, 0.5, n))
    j = rng.random((n, nf)) * 10
    kap = np.exp(rng.normal(0.0, 1.5, (n, nf)))  # optically thin to thick
    if i0 == "band":
        i0v = rng.random(nf)
    elif i0 == "pixel":
        i0v = rng.random((res, res, nf))
    else:
        i0v = i0
    say("radtransfer n", n, "bands", nf, "res", res, "i0", i0)
    img = meshoid_amd.radtransfer(j, m, kap, x, h, res, 16.0, center=[0.5, -0.3, 0.0], i0=i0v)
    want = oracle.radtransfer(j, m, kap, x, h, res, 16.0, center=[0.5, -0.3, 0.0], i0=i0v)
    assert img.shape == (res, res, nf)
    err = np.abs(img - want).max() / np.abs(want).max()
    say("  max rel to image max", err)
    assert err <= 1e-11


def test_radtransfer_clustered_many_bands(oracle):
    """Clumps put thousands of particles on a few tiles, so one tile's records
    run over many chunks (composed per pixel in order); 20 bands shrink the
    tiles to 8 x 8 sightlines."""
    _torch()
    import meshoid_amd
    from meshoid_amd import synthetic

    n, nf, res = 30000, 20, 64
    x = synthetic.clustered(n, seed=9, nclump=5, box=10.0, background=0.05).astype(np.float64)
    rng = np.random.default_rng(9)
    m = rng.random(n) / n
    h = np.exp(rng.normal(-2.0, 1.0, n))
    j = rng.random((n, nf))
    kap = np.exp(rng.normal(3.0, 2.0, (n, nf)))
    say("radtransfer clustered n", n, "bands", nf, "res", res)
    img = meshoid_amd.radtransfer(j, m, kap, x, h, res, 10.0, center=[5.0, 5.0, 5.0], i0=0.5)
    want = oracle.radtransfer(j, m, kap, x, h, res, 10.0, center=[5.0, 5.0, 5.0], i0=0.5)
    err = np.abs(img - want).max() / np.abs(want).max()
    say("  max rel to image max", err)
    assert err <= 1e-11


def test_radtransfer_no_particles_on_the_image():
    """No particles, or none whose footprint reaches a sightline: the image
    is the background."""
    _torch()
    import meshoid_amd

    i0 = np.random.default_rng(2).random((16, 16, 2))
    e = np.zeros((0, 2))
    img = meshoid_amd.radtransfer(e, np.zeros(0), e, np.zeros((0, 3)), np.zeros(0), 16, 4.0, i0=i0)
    assert np.array_equal(img, i0)
    x = np.full((50, 3), 100.0)
    one = np.ones((50, 2))
    img = meshoid_amd.radtransfer(one, np.ones(50), one, x, np.full(50, 0.1), 16, 4.0, i0=i0)
    assert np.array_equal(img, i0)


def test_radtransfer_thick_particles_before_bright_background(oracle):
    """A bright background seen through particles of per-update optical depth
    up to ~40 with little emission: exp(-tau) must not come from 1 + expm1(-tau)
    there (it cancels to 0 beyond tau ~ 37).  Checked per pixel, relative to
    the pixel itself."""
    _torch()
    import meshoid_amd

    x = np.array([[0.1, -0.2, 1.0], [-0.3, 0.2, 0.0], [0.2, 0.1, -1.0]])
    m = np.ones(3)
    h = np.array([1.5, 1.2, 1.8])
    kap = np.array([[22.0], [30.0], [12.0]])  # kernel2d(0) = 1.819: tau up to ~41 per particle
    j = np.full((3, 1), 1e-3)
    i0 = 1e40
    img = meshoid_amd.radtransfer(j, m, kap, x, h, 32, 4.0, i0=i0)
    want = oracle.radtransfer(j, m, kap, x, h, 32, 4.0, i0=i0)
    pos = want > 0
    err = np.abs(img[pos] - want[pos]) / want[pos]
    say("per-pixel max rel", err.max(), "darkest pixel", want.min())
    assert want.min() < 1e-10 * i0  # the sightlines are optically thick
    assert err.max() <= 1e-11


@pytest.mark.parametrize("width,n", [(1, 1), (1, 64), (2, 65), (3, 500), (5, 500), (9, 500), (16, 500), (40, 130),
                                     (0, 2000)])
def test_radtransfer_footprint_widths(oracle, width, n):
    """Records of at most 4, at most 16, at most and more than 64 cells, alone
    and in the order of a mixed set (width 0), around 64 records and several
    chunks.  2000 ordered steps of three roundings and tau of as many terms:
    2e-12 of the largest value at most."""
    _torch()
    import meshoid_amd

    rng = np.random.default_rng(100 * width + n)
    res, size = 37, 12.0
    dx = size / (res - 1)
    x = rng.random((n, 3)) * 13 - 6.5
    w = np.full(n, width) if width else rng.choice([1, 1, 1, 1, 2, 3, 5, 9, 16], n)
    h = 0.5 * w * dx * (1 + 0.01 * rng.standard_normal(n))
    m = (rng.random(n) + 0.1) * h**2
    for nf in (1, 2):
        j, kap = rng.random((n, nf)) * 10, np.exp(rng.normal(-1.0, 1.5, (n, nf)))
        say("radtransfer width", width, "n", n, "bands", nf)
        img = meshoid_amd.radtransfer(j, m, kap, x, h, res, size, center=[0.0, 0.0, 0.0], i0=1.0)
        want = oracle.radtransfer(j, m, kap, x, h, res, size, center=[0.0, 0.0, 0.0], i0=1.0)
        err = np.abs(img - want).max() / np.abs(want).max()
        say("  max rel to image max", err)
        assert err <= 2e-12
