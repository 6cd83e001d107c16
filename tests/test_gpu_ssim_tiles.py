"""SSIM map and gradient at the edges of the kernels' 32x32 tiles."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 11, 5), (1, 31, 33), (2, 32, 32), (1, 42, 43), (3, 64, 31), (2, 97, 65)]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_ssim_tile_edges(hrf, oracle_mod, shape):
    """Window sums of values up to 1 carry a few 2^-24; the variances they are
    subtracted into are about 0.05 here, so the map is good to about 1e-6 and
    the gradient, with two divisions by them, to about 1e-6."""
    import torch
    from complex_valued_holographic_radiance_fields_amd import ssim

    rng = np.random.default_rng(sum(shape))
    x = rng.uniform(size=shape).astype(np.float32)
    y = np.clip(x + 0.15 * rng.normal(size=shape), 0, 1).astype(np.float32)
    g = rng.normal(size=shape).astype(np.float32)
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    tx, ty, tg = (torch.from_numpy(a).cuda() for a in (x, y, g))
    m = ssim.ssim_map(c1, c2, tx, ty).cpu().numpy()
    gx = ssim.ssim_backward(c1, c2, tx, ty, tg).cpu().numpy()
    assert rel_l2(m, oracle_mod.ssim_map(x, y, c1, c2)) < 4e-6
    assert rel_l2(gx, oracle_mod.ssim_backward(x, y, g, c1, c2)) < 1e-5
