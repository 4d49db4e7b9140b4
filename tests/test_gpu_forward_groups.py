"""The forward's groups of pairs: lists around the ends of a group of four, of eight and of a batch of 64 (each 8 x 8 tile's
list is shared by four waves), every channel count, both weights, every tile size, with and without opacities on the alpha
clamp, and coarse levels (the split launch). Image against the float64 oracle at 1e-5 max-abs, gradients at 1e-4
relative, the bars of the other renders."""

import numpy as np
import pytest
import torch

from _gpu_util import RH, random_scene
from test_gpu_api import compare, device_run, oracle_run
from test_gpu_channels import gout_c, scene_c

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 13, 64, 65, 252, 256, 261, 300])
@pytest.mark.parametrize("C,odds,tile", [(3, False, 8), (4, True, 8), (1, True, 4), (2, False, 16), (4, False, 16)])
def test_list_lengths(dev, n, C, odds, tile):
    """Splats wider than the canvas: all n of them in every tile, one tile row and column past the canvas' edge."""
    H, W = 13, 21
    scene = scene_c(C, n, H, W, seed=n + C, dev=dev, ls_mean_px=8.0, op_max=0.4 if n > 64 else 1.0)
    gout = gout_c(C, H, W, dev, seed=n)
    out, g = device_run(RH.render_alpha_full_triton, scene, gout, H=H, W=W, cull=True, odds=odds, TILE=tile)
    ref, rg = oracle_run("cull", scene, gout, H, W, odds=odds, TILE=tile)
    compare(out, g, ref, rg)


@pytest.mark.parametrize("odds", [False, True])
def test_nan_stays_in_its_own_tiles(dev, odds):
    """A colour that is not a number spoils every pixel of its splat's tiles, and no pixel of another tile."""
    H = W = 64
    scene = random_scene(600, H, W, seed=3, dev=dev, ls_mean_px=1.5, op_max=0.9)
    with torch.no_grad():
        clean = RH.render_alpha_full_triton(*scene[:5], H, W, theta=scene[5], cull=True, odds=odds)
        scene[2][0, 100] = float("nan")
        got = RH.render_alpha_full_triton(*scene[:5], H, W, theta=scene[5], cull=True, odds=odds)
    bad = torch.isnan(got[0]).any(0).cpu().numpy()
    assert bad.any()
    tiles = bad.reshape(8, 8, 8, 8).transpose(0, 2, 1, 3).reshape(64, -1)
    assert np.array_equal(tiles.any(1), tiles.all(1))
    keep = ~torch.from_numpy(bad).to(dev)
    assert torch.equal(got[0][:, keep], clean[0][:, keep])
