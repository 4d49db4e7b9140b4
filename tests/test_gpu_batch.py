"""The culled render of a batch as one binning and one launch per step: every image's bits are those of its own call."""

import pytest
import torch

from _gpu_util import RH, random_scene
from test_gpu_api import NAMES, device_run

pytestmark = pytest.mark.gpu


def scene_of(B, n, H, W, dev, big):
    """B images' splats; with `big`, image 0's are large enough for the 16-wave kernels and the others' are not."""
    s = list(random_scene(n, H, W, seed=3 * B + n, dev=dev, op_max=0.9, B=B, margin=0.05))
    if big:
        s[1][0] += 2.5
    return s


@pytest.mark.parametrize("B,n,H,W,TILE,big", [(2, 1, 9, 8, 8, False), (3, 300, 40, 56, 8, False), (12, 257, 33, 24, 4, False),
                                              (13, 64, 24, 24, 8, False), (4, 700, 61, 37, 16, False),
                                              (3, 900, 64, 64, 8, True), (2, 200, 5000, 8, 8, False)])
def test_batch_equals_single_calls(dev, B, n, H, W, TILE, big):
    """Image and all gradients, three times over (the first call reads the pair counts first, the others speculate),
    with a batch of other splats in between; a second backward of the same graph included."""
    scene = scene_of(B, n, H, W, dev, big)
    other = scene_of(B, n, H, W, dev, False)
    gout = torch.randn(B, 3, H, W, generator=torch.Generator().manual_seed(B)).to(dev)
    kw = dict(H=H, W=W, cull=True, TILE=TILE)
    single = [device_run(RH.render_alpha_full_triton, [t[b:b + 1] for t in scene], gout[b:b + 1], **kw) for b in range(B)]
    for _ in range(3):
        out, g = device_run(RH.render_alpha_full_triton, scene, gout, **kw)
        for b, (o1, g1) in enumerate(single):
            assert torch.equal(out[b], o1[0]), b
            for k in NAMES:
                assert torch.equal(g[k][b], g1[k][0]), (b, k)
        device_run(RH.render_alpha_full_triton, other, gout, **kw)
    L = [t.detach().clone().requires_grad_(True) for t in scene]
    img = RH.render_alpha_full_triton(*L[:5], theta=L[5], **kw)
    ga = torch.autograd.grad(img, L, gout, retain_graph=True)
    gb = torch.autograd.grad(img, L, gout)
    for x, y in zip(ga, gb):
        assert torch.equal(x, y)


def test_batch_past_the_pair_range(dev, monkeypatch):
    """Images whose pairs together pass the int32 pair index, while each image's own do not (here: the status of such a
    count, given for a merged binning only), are rendered one after another: a speculated call, then a first one."""
    B, n, H, W = 3, 300, 40, 56
    scene = scene_of(B, n, H, W, dev, False)
    gout = torch.randn(B, 3, H, W, generator=torch.Generator().manual_seed(B)).to(dev)
    kw = dict(H=H, W=W, cull=True)
    single = [device_run(RH.render_alpha_full_triton, [t[b:b + 1] for t in scene], gout[b:b + 1], **kw) for b in range(B)]
    device_run(RH.render_alpha_full_triton, scene, gout, **kw)
    settle, calls = RH._settle, []

    def past_the_range(p, rc, pb):
        calls.append(p.geo[3])
        return settle(p, rc if p.geo[3] is None else 4, pb)
    monkeypatch.setattr(RH, "_settle", past_the_range)
    for first in (False, True):
        if first:
            RH._PAIRS_HW.clear()
        out, g = device_run(RH.render_alpha_full_triton, scene, gout, **kw)
        for b, (o1, g1) in enumerate(single):
            assert torch.equal(out[b], o1[0]), b
            for k in NAMES:
                assert torch.equal(g[k][b], g1[k][0]), (b, k)
    assert sum(c is not None for c in calls) == 2 and sum(c is None for c in calls) == 2 * B
