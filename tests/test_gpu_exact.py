"""The exact path's kernels at the edges of their splits: pixel groups of 64 (8 x 8 tiles of a grid, or 64 of a list),
splat batches of 64, the shares of both, and the reach boxes that leave out pairs whose every term is an exact zero."""

import math
import time

import pytest
import torch

from _gpu_util import IMG_TOL, GRAD_REL_TOL, RH, np_, random_scene, rel_err
from gaussian_splat_encoder import render as R_api
from gaussian_splat_encoder import _lib
from test_gpu_api import NAMES, compare, device_run, oracle_run

pytestmark = pytest.mark.gpu


def run_c(scene, H, W, gout, reach=True, grid=True):
    """The C-ABI calls of one image, with or without the reach boxes: out, T, asum, fg and the six gradients."""
    lib, stream, dev = _lib.load(), _lib.stream_ptr(scene[0].device), scene[0].device
    mu, ls, col, op, bg, th = [None if t is None else t[0].contiguous() for t in scene]
    N, C, P = mu.shape[0], col.shape[1], H * W
    ys, xs = R_api._pixel_axes(H, W, dev, torch.float32)
    if not grid:
        ys, xs = ys.repeat_interleave(W).contiguous(), xs.repeat(H).contiguous()
    gw = W if grid else 0
    rec = torch.empty(64 * N + lib.splat_exact_reach_bytes(N), dtype=torch.uint8, device=dev)
    p = _lib.ptr
    r0, rr = rec.data_ptr(), rec.data_ptr() + 64 * N
    _lib.check(lib.splat_decode_exact(p(mu), p(ls), p(th), p(op), p(col), C, N, _lib.FLAG_LOG_SCALE, r0, rr, stream), "d")
    e = lambda *s: torch.empty(s, device=dev)   # noqa: E731
    out, T, asum, fg = e(P, C), e(P), e(P), e(P, C)
    nws = lib.splat_exact_fwd_workspace_bytes(N, C, P, gw)
    ws = torch.empty(max(nws, 1), dtype=torch.uint8, device=dev)
    rp = rr if reach else None
    _lib.check(lib.splat_exact_render(r0, rp, N, C, p(ys), p(xs), P, gw, None, p(bg), p(out), p(T), p(asum), p(fg), p(ws), nws,
                                      stream), "f")
    g = [e(N, 2), e(N, 2), None if th is None else e(N), e(N), e(N, C), e(C)]
    nws = lib.splat_exact_render_bwd_workspace_bytes(N, C, P, gw)
    ws = torch.empty(nws, dtype=torch.uint8, device=dev)
    go = gout[0].permute(1, 2, 0).contiguous()
    _lib.check(lib.splat_exact_render_bwd(r0, rp, N, C, p(ys), p(xs), P, gw, None, p(bg), p(T), p(asum), p(fg), p(go), p(ls),
                                          *[p(t) for t in g], p(ws), nws, stream), "b")
    return [out, T, asum, fg] + [t for t in g if t is not None]


def same(a, b):
    """Values that are not finite in the same places; elsewhere within the rounding of their terms' regrouping."""
    for x, y in zip(a, b):
        fx, fy = torch.isfinite(x), torch.isfinite(y)
        assert torch.equal(fx, fy)
        if fx.any():
            assert rel_err(np_(x[fx]), np_(y[fy])) <= 1e-5


@pytest.mark.parametrize("H,W,N", [(1, 1, 1), (8, 8, 63), (7, 90, 64), (9, 8, 65), (64, 64, 129), (33, 65, 700),
                                   (70, 130, 4200)])
def test_exact_sizes(dev, H, W, N):
    """Image and gradients against the float64 oracle at the edges of the pixel groups and splat batches."""
    scene = random_scene(N, H, W, seed=31 + N, dev=dev, op_max=0.95, theta=N % 2 == 1, margin=0.1)
    gout = torch.randn(1, 3, H, W, generator=torch.Generator().manual_seed(N)).to(dev)
    out, g = device_run(RH.render_alpha_full_triton, scene, gout, H=H, W=W)
    ref, rg = oracle_run("exact", scene, gout, H, W)
    compare(out, g, ref, rg)


@pytest.mark.parametrize("n_px,N", [(1, 300), (63, 64), (65, 5000), (300, 9000), (2000, 40000)])
def test_exact_pixel_list(dev, n_px, N):
    """A pixel list (few groups: the splats split over many workgroups) equals the full render at those pixels, and
    its gradients those of the full render with the upstream gradient at those pixels only."""
    H, W = 40, 56
    scene = random_scene(N, H, W, seed=5, dev=dev, op_max=0.9)
    gen = torch.Generator().manual_seed(n_px)
    idx = torch.randperm(H * W, generator=gen)[:n_px].to(dev)[None]
    go = torch.randn(1, 3, n_px, generator=gen).to(dev)
    full_go = torch.zeros(1, 3, H * W, device=dev)
    full_go[:, :, idx[0]] = go
    full, gf = device_run(RH.render_alpha_full_triton, scene, full_go.view(1, 3, H, W), H=H, W=W)
    L = [t.detach().clone().requires_grad_(True) for t in scene]
    sub, _ = R_api.render_alpha_subsampled(*L[:5], H, W, theta=L[5], pixel_indices=idx)
    (sub * go).sum().backward()
    assert (sub - full.reshape(1, 3, -1)[:, :, idx[0]]).abs().max().item() <= IMG_TOL
    for n, t in zip(NAMES, L):
        assert rel_err(np_(t.grad), np_(gf[n])) <= GRAD_REL_TOL, n


@pytest.mark.parametrize("sigma,std,aspect,op", [(0.05, 1.0, 1.0, 1.0), (2.0, 0.5, 1.0, 0.9), (1.0, 0.3, 300.0, 1.0),
                                                 (60.0, 1.0, 1.0, 0.99)])
@pytest.mark.parametrize("grid", [True, False])
def test_reach_leaves_out_exact_zeros_only(dev, sigma, std, aspect, op, grid):
    """With the reach boxes the outputs differ from those without them by the grouping of the same nonzero terms (at most
    4,697 float32 additions or products each): splats far smaller than a pixel, needles, splats larger than the canvas,
    splats outside it, opacities of 0 and 1."""
    H, W, N = 61, 77, 777
    scene = list(random_scene(N, H, W, seed=8, dev=dev, ls_mean_px=sigma, ls_std=std, op_max=op, margin=0.5))
    scene[1][..., 1] += math.log(aspect)
    scene[3][0, ::50] = 0.0
    scene[3][0, 1::50] = 1.0
    gout = torch.randn(1, 3, H, W, generator=torch.Generator().manual_seed(2)).to(dev)
    same(run_c(scene, H, W, gout, True, grid), run_c(scene, H, W, gout, False, grid))


def test_reach_keeps_values_that_are_not_finite(dev):
    """A colour, opacity or centre that is not finite reaches every pixel, and an upstream gradient that is not finite
    every splat, with the boxes as without."""
    H, W, N = 40, 48, 200
    gout = torch.randn(1, 3, H, W, generator=torch.Generator().manual_seed(2)).to(dev)
    for which, value in ((2, math.inf), (2, math.nan), (3, math.nan), (3, -0.5), (0, math.nan), (1, math.nan), (None, math.inf)):
        scene = list(random_scene(N, H, W, seed=9, dev=dev, ls_mean_px=0.7, op_max=0.9))
        go = gout.clone()
        if which is None:
            go[0, 1, 3, 5] = value
        else:
            scene[which][0, 17] = value
        same(run_c(scene, H, W, go, True), run_c(scene, H, W, go, False))


def axes(H, W, dev):
    return R_api._pixel_axes(H, W, dev, torch.float32)


@pytest.mark.parametrize("H,W,N", [(256, 512, 64), (256, 504, 64), (250, 517, 65), (2048, 64, 0), (1024, 1024, 1),
                                   (1000, 1030, 128), (1024, 1024, 256), (1024, 1008, 256), (1448, 1450, 512)])
def test_few_splats_on_many_pixels(dev, H, W, N):
    """One wave per pixel group, at the sizes where the rule for it begins and just before: every 61st pixel against a list of
    those pixels, whose groups take eight waves. The sums of up to 512 terms are grouped another way: 1e-6 of T, of the
    colours and of S_a relative to its size."""
    mu, ls, col, op, bg, th = random_scene(N, H, W, seed=N + 1, dev=dev, ls_mean_px=0.05 * W, op_max=0.95, margin=0.1)
    ys, xs = axes(H, W, dev)
    full = RH._forward(mu, ls, col, op, bg, ys, xs, th, W, True)[:4]
    idx = torch.arange(0, H * W, 61, device=dev)
    some = RH._forward(mu, ls, col, op, bg, ys[idx // W].contiguous(), xs[idx % W].contiguous(), th, 0, True)[:4]
    for a, b in zip(full, some):
        a = a[:, idx]
        assert ((a - b).abs() <= 1e-6 * b.abs().clamp_min(1.0)).all()


def test_few_splats_on_many_listed_pixels(dev):
    """The same for a list: one of every pixel of a canvas against the canvas."""
    H, W, N = 1024, 1100, 64
    mu, ls, col, op, bg, th = random_scene(N, H, W, seed=3, dev=dev, ls_mean_px=40.0, op_max=0.95)
    ys, xs = axes(H, W, dev)
    full = RH._forward(mu, ls, col, op, bg, ys, xs, th, W, True)[:4]
    some = RH._forward(mu, ls, col, op, bg, ys.repeat_interleave(W).contiguous(), xs.repeat(H).contiguous(), th, 0, True)[:4]
    for a, b in zip(full, some):
        assert ((a - b).abs() <= 1e-6 * b.abs().clamp_min(1.0)).all()


def best_us(f, n=10):
    best = float("inf")
    for _ in range(8):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(n):
            f()
        torch.cuda.synchronize()
        best = min(best, (time.perf_counter() - t0) / n * 1e6)
    return best


def test_few_splats_on_many_pixels_take_no_longer(dev):
    """64 splats on 2048 x 2048, bound by the 134 MB that the forward writes: at most five times a copy of as much, most of
    which the last-level cache holds."""
    H = W = 2048
    mu, ls, col, op, bg, th = random_scene(64, H, W, seed=3, dev=dev, ls_mean_px=100.0, op_max=0.95)
    ys, xs = axes(H, W, dev)
    src = torch.empty(8 * H * W, device=dev)
    dst = torch.empty_like(src)
    copy = best_us(lambda: dst.copy_(src))
    render = best_us(lambda: RH._forward(mu, ls, col, op, bg, ys, xs, th, W, True))
    print(f"render {render:.1f} us, copy {copy:.1f} us", flush=True)
    assert render <= 5 * copy
