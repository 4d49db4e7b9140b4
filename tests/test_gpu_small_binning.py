"""The one-launch binning of small problems at the edges of its range: pair lists and maps bit-exact against the oracle's
binning, for the first call of a configuration (count read first) and later ones (one launch), with capacities exceeded."""

import numpy as np
import pytest
import torch

from _gpu_util import RH, activate_scale, random_scene
from gaussian_splat_encoder import _lib
from oracle import binning

pytestmark = pytest.mark.gpu


def check(bins, b, mu, sc, H, W, TILE, cutoff):
    gid, starts = binning.build_tiles(mu, sc, H, W, TILE, cutoff)
    assert np.array_equal(bins.starts_b[b].cpu().numpy(), starts)
    tot = int(starts[-1])
    assert np.array_equal(bins.gid_b[b].cpu().numpy()[:max(tot, 1)], gid)
    if not tot:
        return
    tx0, tx1, ty0, _, cnt = binning.rects(mu, sc, H, W, TILE, cutoff)
    tile = np.repeat(np.arange(starts.size - 1), np.diff(starts))
    ntx = binning.tile_grid(H, W, TILE)[0]
    off = np.concatenate([[0], np.cumsum(cnt)])
    q = off[gid] + (tile // ntx - ty0[gid]) * (tx1 - tx0 + 1)[gid] + tile % ntx - tx0[gid]
    assert np.array_equal(bins.pq_b[b].cpu().numpy()[:tot], q)
    assert np.array_equal(bins.off_b[b].cpu().numpy(), off)


@pytest.mark.parametrize("H,W,TILE,n,px", [
    (8, 8, 8, 1, 1.0), (8, 8, 8, 33, 3.0), (64, 64, 8, 1023, 1.5), (64, 64, 8, 1024, 1.5), (96, 96, 8, 2047, 2.0),
    (96, 96, 8, 2048, 2.0), (96, 96, 8, 2049, 2.0), (128, 128, 8, 1024, 40.0), (1100, 8, 1, 31, 2.0), (160, 400, 4, 32, 20.0),
    (90, 70, 16, 700, 9.0), (130, 136, 8, 1100, 2.0), (96, 96, 8, 1500, 5.0)])
def test_small_binning_bit_exact(dev, H, W, TILE, n, px):
    """Thrice, then a scene of larger splats (more pairs than the remembered capacity, and in some cases than the one
    launch takes) and the first one again."""
    scenes = [random_scene(n, H, W, seed=n + k, dev=dev, ls_mean_px=px * f, margin=0.2) for k, f in ((0, 1.0), (1, 4.0))]
    for k in (0, 0, 0, 1, 1, 0):
        mu, ls, col, op, _, th = scenes[k]
        sc = activate_scale(ls)
        bins = RH._bin(mu, sc, col, op, th, H, W, TILE, 3.0)
        check(bins, 0, mu[0].cpu().numpy(), sc[0].cpu().numpy(), H, W, TILE, 3.0)


def test_small_binning_of_levels(dev):
    """Octave levels and a merged batch: every level's list equals the oracle's of its own splats and canvas."""
    H, W, n = 72, 56, 500
    mu, ls, col, op, _, th = random_scene(n, H, W, seed=4, dev=dev, ls_mean_px=6.0, ls_std=0.9)
    sc = activate_scale(ls)
    lv = _lib.SplatLevels(1, 6, 8.0, 0, 0, 0)
    batch = _lib.SplatLevels(3, 3, 0.0, n // 3, 0, 0)
    m, s = mu[0].cpu().numpy(), sc[0].cpu().numpy()
    for levels, N in ((lv, n), (batch, n - n % 3)):
        for _ in range(3):
            bins = RH._bin(mu[:, :N].contiguous(), sc[:, :N].contiguous(), col[:, :N].contiguous(),
                           op[:, :N].contiguous(), th[:, :N].contiguous(), H, W, 8, 3.0, lv=levels)
            lev = bins.rect_b[0][:, 3].cpu().numpy()
            starts, gid = bins.starts_b[0].cpu().numpy(), bins.gid_b[0].cpu().numpy()
            for l, (Hl, Wl, ntx, tb, _) in enumerate(bins.geom):
                ids = np.nonzero(lev == l)[0]
                g, st = binning.build_tiles(m[ids], s[ids], Hl, Wl, 8, 3.0)
                assert bins.level_tot_b[0][l] == st[-1]
                assert np.array_equal(starts[tb:tb + st.size] - starts[tb], st)
                if st[-1]:
                    assert np.array_equal(gid[starts[tb]:starts[tb] + st[-1]], ids[g])


def test_small_binning_errors(dev):
    """With the one launch queued, an empty rect still raises and the pair budget too."""
    mu, ls, col, op, _, th = random_scene(200, 64, 64, seed=4, dev=dev)
    sc = activate_scale(ls)
    for _ in range(2):
        RH._bin(mu, sc, col, op, th, 64, 64, 8, 3.0)
    with pytest.raises(ValueError, match="empty tile rect"):
        RH._bin(mu, -sc, col, op, th, 64, 64, 8, 3.0)
    with pytest.raises(RH.PairBudgetExceeded):
        RH._bin(mu, sc, col, op, th, 64, 64, 8, 3.0, max_pairs=10)
