"""Performance cases of the renderer: what its users call, from a 64 x 64 preview to a 2048 x 2048 training step.

A case is a dict of plain values:
  path      "cull" (render_alpha_full_triton, cull=True), "octave" (render_alpha_octave), "multires"
            (render_alpha_multires), "exact" (render_alpha_full) or "pixels" (render_alpha_subsampled)
  train     1: the image and the gradients of every parameter from a given upstream gradient; 0: the image, no grad
  B, H, W   batch and canvas
  cell, per, sigma        one group of splats: `per` in every cell x cell pixels (cell-major, as the encoder emits
                          them), of about `sigma` pixels
  cell2, per2, sigma2     a second group of larger splats before it (0: none); "multires" renders it coarsely
  heavy     share of the first group re-drawn at about 40 pixels
  opacity   mean of the opacity logits
  C, theta, odds, tile, cutoff   colour channels, rotated or not, odds weights, TILE and cull radius
  n_px      "pixels": how many pixels are rendered

listed(), draw(rng), prepare(case, seed), run(state), work(case), tolerance(case) and exact(case, seed) are what a
measuring program needs; exact() is plain torch in float64.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gaussian-2d-splat-encoder_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from gaussian_splat_encoder import render as R  # noqa: E402
from gaussian_splat_encoder import render_hip as RH  # noqa: E402

BASE = {"path": "cull", "train": 1, "B": 1, "H": 768, "W": 768, "cell": 8, "per": 10, "sigma": 3.0, "cell2": 0,
        "per2": 0, "sigma2": 0.0, "heavy": 0.0, "opacity": 1.5, "C": 3, "theta": 1, "odds": 0, "tile": 8,
        "cutoff": 3.0, "n_px": 0}

# 98 flops per pixel-pair of a forward and backward (27 + 71; odds 28 + 74), each operation of the compositing
# formulas counted once with the per-splat terms hoisted.
FLOPS_FWD, FLOPS_BWD = (27, 28), (71, 74)


def _case(name, **kw):
    return dict(BASE, name=name, **kw)


def listed():
    # The encoder's splats at an image of S x S pixels: two coarse ones per 8 x 8 cell (sigma 0.045 S) and two fine
    # ones per 4 x 4 cell (sigma 0.0067 S), composited with the odds weights.
    enc768 = dict(cell=4, per=2, sigma=5.1, cell2=8, per2=2, sigma2=34.5, opacity=0.0)
    return [
        # a thumbnail preview: the smallest call, launches and latency
        _case("cull_infer_64", H=64, W=64, per=16, sigma=1.5, train=0, opacity=1.0),
        # a training batch of small images with odd sides, the encoder's weights
        _case("cull_train_batch", B=4, H=250, W=187, per=8, sigma=2.5, odds=1),
        # the headline training step
        _case("cull_train_768"),
        # the largest training step, with a heavy tail of splats of 40 pixels
        _case("cull_train_2048", H=2048, W=2048, heavy=0.02),
        # the encoder's own coarse render, in inference
        _case("octave_infer_384", path="octave", train=0, H=384, W=384, cell=4, per=2, sigma=17.3, odds=1,
              opacity=0.0),
        # the encoder's full render, in inference
        _case("octave_infer_768", path="octave", train=0, odds=1, **enc768),
        # training the encoder through its full render
        _case("octave_train_768", path="octave", odds=1, **enc768),
        # the largest octave training step
        _case("octave_train_2048", path="octave", H=2048, W=2048, heavy=0.02),
        # coarse and fine groups given by the caller, at 1024
        _case("multires_train_1024", path="multires", H=1024, W=1024, cell2=64, per2=4, sigma2=60.0),
        # the exact render as a check of a small scene
        _case("exact_train_64", path="exact", H=64, W=64, per=16, sigma=1.5, opacity=1.0),
        # the exact render at the size where the culled one replaces it
        _case("exact_train_512", path="exact", H=512, W=512, per=4, sigma=4.0),
        # a training step on a subsample of an image's pixels
        _case("pixels_train_768", path="pixels", n_px=10000),
    ]


def _logu(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    path = rng.choice(["cull", "cull", "octave", "octave", "multires", "exact", "pixels"])
    c = dict(BASE, path=path, train=int(rng.random() < 0.6), odds=int(path != "exact" and rng.random() < 0.4),
             theta=int(rng.random() < 0.8), sigma=round(_logu(rng, 1.0, 5.0), 2),
             opacity=rng.choice([0.0, 1.0, 1.5]), C=rng.choice([3, 3, 3, 3, 1, 4]))
    if path in ("exact", "pixels"):
        c["odds"] = 0
        c["H"] = int(_logu(rng, 48, 512))
        c["W"] = max(8, int(c["H"] * rng.uniform(0.6, 1.6)))
        c["cell"], c["per"] = rng.choice([(4, 1), (8, 1), (8, 4), (8, 10), (16, 3)])
        if path == "pixels":
            c["n_px"] = min(c["H"] * c["W"], int(_logu(rng, 256, 16384)))
        while _pairs(c) > 4.0e9:
            c["H"], c["W"] = c["H"] * 3 // 4, c["W"] * 3 // 4
        return c
    c["H"] = int(_logu(rng, 48, 2048))
    c["W"] = max(16, min(2048, int(c["H"] * rng.uniform(0.6, 1.6))))
    c["B"] = rng.choice([1, 1, 2, 4]) if c["H"] <= 300 else 1
    c["tile"] = rng.choice([8, 8, 8, 8, 4, 16])
    c["cutoff"] = rng.choice([3.0, 3.0, 3.0, 2.5, 3.5])
    c["cell"], c["per"] = rng.choice([(4, 1), (4, 2), (8, 4), (8, 10), (16, 7)])
    if path != "cull" and rng.random() < 0.7 or path == "multires":
        c["cell2"], c["per2"] = rng.choice([(16, 1), (32, 3), (64, 4)])
        c["sigma2"] = round(0.045 * min(c["H"], c["W"]), 2)
    else:
        c["heavy"] = rng.choice([0.0, 0.0, 0.02]) if path == "octave" or c["H"] > 700 else 0.0
    while _pairs(c) > 27.0e6 * min(64, c["tile"] ** 2):
        c["sigma"] *= 0.8
        c["heavy"] = 0.0
        c["sigma2"] *= 0.8
    return c


# ------------------------------------------------------------------------------------------------ inputs
def _cells(c, cell):
    return -(-c["H"] // cell), -(-c["W"] // cell)


def _counts(c):
    """Splats of the larger and of the smaller group."""
    n = [0, 0]
    for i, (cell, per) in enumerate(((c["cell2"], c["per2"]), (c["cell"], c["per"]))):
        if cell:
            gy, gx = _cells(c, cell)
            n[i] = gy * gx * per
    return n


def _group(c, B, cell, per, sigma, heavy, g, dev):
    """mu [B,N,2] and raw log-scales [B,N,2] of one group."""
    gy, gx = _cells(c, cell)
    n = gy * gx * per
    hw = torch.tensor([c["H"], c["W"]], dtype=torch.float32, device=dev)
    i = torch.arange(n, device=dev) // per
    yx = torch.stack([i // gx, i % gx], -1).float()
    mu = (yx + torch.rand(B, n, 2, generator=g, device=dev)) * cell / hw
    z = torch.randn(B, n, 2, generator=g, device=dev)
    ls = math.log(sigma) + (0.2 if sigma > 12 else 0.5) * z   # a coarse head's splats sit near its scale floor
    if heavy:
        ls = torch.where(torch.rand(B, n, 1, generator=g, device=dev) < heavy, math.log(40.0) + 0.3 * z, ls)
    return mu.clamp(0, 1), ls - torch.log(hw)


def _inputs(c, seed, dev="cuda", B=None):
    B = c["B"] if B is None else B
    g = torch.Generator(dev).manual_seed(int(seed))
    mus, lss = [], []
    for cell, per, sigma, heavy in ((c["cell2"], c["per2"], c["sigma2"], 0.0),
                                    (c["cell"], c["per"], c["sigma"], c["heavy"])):
        if cell:
            mu, ls = _group(c, B, cell, per, sigma, heavy, g, dev)
            mus.append(mu)
            lss.append(ls)
    mu, ls = torch.cat(mus, 1), torch.cat(lss, 1)
    n = mu.shape[1]
    theta = math.pi * torch.rand(B, n, generator=g, device=dev)
    p = {"mu": mu, "log_scale": ls, "color": torch.rand(B, n, c["C"], generator=g, device=dev),
         "opacity": torch.sigmoid(c["opacity"] + 1.5 * torch.randn(B, n, generator=g, device=dev)),
         "bg": torch.rand(B, c["C"], generator=g, device=dev)}
    if c["theta"]:
        p["theta"] = theta
    s = {"case": c, "p": p}
    if c["path"] == "pixels":
        s["idx"] = torch.randint(0, c["H"] * c["W"], (B, c["n_px"]), generator=g, device=dev)
        s["gout"] = torch.randn(B, c["C"], c["n_px"], generator=g, device=dev)
    else:   # in the image's own layout, as the gradient of a loss of the image arrives
        s["gout"] = torch.randn(B, c["H"], c["W"], c["C"], generator=g, device=dev).permute(0, 3, 1, 2)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["train"]:
        for t in s["p"].values():
            t.requires_grad_(True)
    return s


def _render(s):
    c, p = s["case"], s["p"]
    a = (p["mu"], p["log_scale"], p["color"], p["opacity"], p["bg"], c["H"], c["W"])
    th = p.get("theta")
    if c["path"] == "cull":
        return RH.render_alpha_full_triton(*a, theta=th, cull=True, TILE=c["tile"], cutoff=c["cutoff"],
                                           odds=bool(c["odds"]))
    if c["path"] == "octave":
        return RH.render_alpha_octave(*a, theta=th, cutoff=c["cutoff"], TILE=c["tile"], odds=bool(c["odds"]))
    if c["path"] == "multires":
        return RH.render_alpha_multires(*a, theta=th, n_coarse=_counts(c)[0], cutoff=c["cutoff"], TILE=c["tile"],
                                        odds=bool(c["odds"]))
    if c["path"] == "exact":
        return R.render_alpha_full(*a, theta=th)
    return R.render_alpha_subsampled(*a, theta=th, pixel_indices=s["idx"])[0]


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return {"image": _render(state)}
    p = state["p"]
    img = _render(state)
    grads = torch.autograd.grad(img, list(p.values()), state["gout"])
    return {"image": img.detach(), **{"g_" + k: g for k, g in zip(p, grads)}}


# -------------------------------------------------------------------------------------------- tiles and levels
def _levels(c):
    """[(H_l, W_l)] of the canvases a render uses, the native one first."""
    H, W = c["H"], c["W"]
    if c["path"] == "octave":
        return [(max(8, H >> o), max(8, W >> o)) for o in range(7)]
    if c["path"] == "multires":
        cf = min(8, max(1, min(H, W) // 8))
        return [(H, W), (max(1, H // cf), max(1, W // cf))]
    return [(H, W)]


def _routes(c, scale):
    """Level of every splat [N], from its float32 scales [N, 2]."""
    if c["path"] == "octave":
        px = scale.amax(-1) * min(c["H"], c["W"])
        return torch.ceil(torch.log2((px / 8.0).clamp_min(1e-6))).clamp(0, 6).long()
    lev = torch.zeros(scale.shape[0], dtype=torch.long, device=scale.device)
    if c["path"] == "multires":
        lev[:_counts(c)[0]] = 1
    return lev


def _rects(c, mu, scale, H, W):
    """Tile rects (x0, x1, y0, y1 inclusive) on an (H, W) canvas, in float32 as the binning defines them."""
    T = c["tile"]
    r = c["cutoff"] * scale.amax(-1)
    x, y, rx, ry = mu[:, 1] * W, mu[:, 0] * H, r * W, r * H
    ex = lambda v, n: torch.floor(v / T).clamp(0, -(-n // T) - 1).long()   # noqa: E731
    return ex(x - rx, W), ex(x + rx, W), ex(y - ry, H), ex(y + ry, H)


_PAIRS = {}


def _pairs(c, needed=False):
    """Pixel-pairs of one pass, in expectation from one seeded draw of the splats' own distribution: every pixel of a
    splat's tiles, or every requested pixel for the exact paths. needed: for the exact paths only those where the
    falloff exp(-maha / 2) is not zero in float32 (maha / 2 below 126 ln 2)."""
    if c["path"] in ("exact", "pixels") and not needed:
        return c["B"] * sum(_counts(c)) * (c["n_px"] or c["H"] * c["W"])
    key = (needed,) + tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if key not in _PAIRS:
        p = _inputs(c, 1, "cpu", 1)["p"]
        mu, scale = p["mu"][0], F.softplus(p["log_scale"][0]) + 1e-4
        if c["path"] in ("exact", "pixels"):
            share = (2 * 126 * math.log(2) * math.pi * scale.prod(-1)).clamp(max=1.0)   # of the canvas
            _PAIRS[key] = c["B"] * float(share.double().sum()) * (c["n_px"] or c["H"] * c["W"])
            return _PAIRS[key]
        lev, tot = _routes(c, scale), 0
        for l, (H, W) in enumerate(_levels(c)):
            m = lev == l
            x0, x1, y0, y1 = _rects(c, mu[m], scale[m], H, W)
            tot += int(((x1 - x0 + 1) * (y1 - y0 + 1)).sum())
        _PAIRS[key] = c["B"] * tot * c["tile"] ** 2
    return _PAIRS[key]


def work(case):
    c = case
    n, px = c["B"] * sum(_counts(c)), c["B"] * (c["n_px"] or c["H"] * c["W"])
    per = 5 + c["theta"] + c["C"]           # floats of one splat: mu, log_scale, opacity, theta, colour
    odds = c["odds"]
    pairs = _pairs(c, needed=c["path"] in ("exact", "pixels"))
    b, f = 4 * (n * per + px * c["C"]), FLOPS_FWD[odds] * pairs
    if c["train"]:
        b, f = 2 * b, f + FLOPS_BWD[odds] * pairs
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the largest error against exact() seen over the listed and 40 drawn cases. The binned renders'
    gradients amplify the float32 rounding of 1 - T and of the falloff's exponent at pixels that few splats cover
    (9.4e-5 of a gradient, 3e-2 of a single value); their images are within 3.9e-6 (1.1e-4), the exact ones' images
    and gradients within 3.2e-7 and 1.2e-6."""
    if case["path"] in ("exact", "pixels"):
        return {"rel": 5e-6 if case["train"] else 1.5e-6}
    return {"rel": 4e-4, "max": 0.12} if case["train"] else {"rel": 1.5e-5, "max": 5e-4}


# ------------------------------------------------------------------------------------------------- float64
CLAMP = 0.99989998340606689453125   # 1 - 1e-4 in float32, as the renderer compares alphas
CHUNK = 1 << 22                      # pixel-pairs evaluated at once


def _terms(c, mu, sc, th, op, py, px):
    """log(1 - a) and the colour weight of splats [M] at pixel centres py, px that broadcast against [M, 1, 1]."""
    v = lambda t: t[:, None, None]   # noqa: E731
    dy, dx = py - v(mu[:, 0]), px - v(mu[:, 1])
    if th is None:
        ry, rx = dy / v(sc[:, 0]), dx / v(sc[:, 1])
    else:
        cs, sn = v(torch.cos(th)), v(torch.sin(th))
        ry, rx = (cs * dy + sn * dx) / v(sc[:, 0]), (cs * dx - sn * dy) / v(sc[:, 1])
    a = (v(op) * torch.exp(-0.5 * (ry * ry + rx * rx))).clamp(max=CLAMP)
    return torch.log1p(-a), a / (1 - a) if c["odds"] else a


class _Tiles:
    """The (splat, tile) pairs of one level, evaluated a chunk at a time."""

    def __init__(self, c, mu32, scale32, H, W, ids):
        T, dev = c["tile"], mu32.device
        self.H, self.W, self.T = H, W, T
        self.ty, self.tx = -(-H // T), -(-W // T)
        x0, x1, y0, y1 = _rects(c, mu32[ids], scale32[ids], H, W)
        w, n = x1 - x0 + 1, (x1 - x0 + 1) * (y1 - y0 + 1)
        rep = torch.repeat_interleave(torch.arange(ids.numel(), device=dev), n)
        k = torch.arange(rep.numel(), device=dev) - (n.cumsum(0) - n)[rep]
        self.g, self.row, self.col = ids[rep], y0[rep] + k // w[rep], x0[rep] + k % w[rep]
        self.i = torch.arange(T, device=dev)

    def chunks(self):
        m = max(1, CHUNK // self.T ** 2)
        for o in range(0, self.g.numel(), m):
            r, q = self.row[o:o + m], self.col[o:o + m]
            py = ((r[:, None] * self.T + self.i).float() + 0.5) / self.H     # pixel centres are float32 numbers
            px = ((q[:, None] * self.T + self.i).float() + 0.5) / self.W
            yield self.g[o:o + m], r * self.tx + q, py.double()[:, :, None], px.double()[:, None, :]

    def zeros(self, k, dev):
        return torch.zeros(k, self.ty * self.tx, self.T, self.T, dtype=torch.float64, device=dev)

    def canvas(self, f):
        f = f.view(-1, self.ty, self.tx, self.T, self.T).permute(0, 1, 3, 2, 4)
        return f.reshape(f.shape[0], self.ty * self.T, self.tx * self.T)[:, :self.H, :self.W]

    def tiled(self, f):
        f = F.pad(f, (0, self.tx * self.T - self.W, 0, self.ty * self.T - self.H))
        f = f.view(-1, self.ty, self.T, self.tx, self.T).permute(0, 1, 3, 2, 4)
        return f.reshape(f.shape[0], self.ty * self.tx, self.T, self.T)


class _Every:
    """Every splat at every requested pixel, a block of both at a time."""

    def __init__(self, n, py, px):
        self.n, self.py, self.px = n, py.double(), px.double()

    def chunks(self):
        P = self.py.numel()
        pm = min(P, CHUNK // 64)
        m = max(1, CHUNK // pm)
        for o in range(0, self.n, m):
            g = torch.arange(o, min(o + m, self.n), device=self.py.device)
            for q in range(0, P, pm):
                yield g, slice(q, q + pm), self.py[None, None, q:q + pm], self.px[None, None, q:q + pm]

    def zeros(self, k, dev):
        return torch.zeros(k, 1, self.py.numel(), dtype=torch.float64, device=dev)

    def canvas(self, f):
        return f

    def tiled(self, f):
        return f


def _add(f, at, v):
    """f[k, at[i]] += v[k][i] for tiles, the sum over the splats for a block of pixels."""
    for k, x in enumerate(v):
        if isinstance(at, slice):
            f[k, 0, at] += x.sum((0, 1))
        else:
            f[k].index_add_(0, at, x)


def _gather(acc, g, v):
    """acc[g[i]] += v[i] with equal g in runs (a large splat's pairs: no contended atomics)."""
    ids, n = torch.unique_consecutive(g, return_counts=True)
    acc.index_add_(0, ids, torch.segment_reduce(v, "sum", lengths=n, axis=0))


def _get(f, at):
    return f[:, 0, at][:, None, None, :] if isinstance(at, slice) else f[:, at]


def exact(case, seed):
    c = case
    s = _inputs(c, seed)
    outs = []
    for b in range(c["B"]):
        p32 = {k: v[b] for k, v in s["p"].items()}
        p = {k: v.double() for k, v in p32.items()}
        ls = p["log_scale"].requires_grad_(True)
        sc = F.softplus(ls) + 1e-4
        scd, mu, op, col, th = sc.detach(), p["mu"], p["opacity"], p["color"], p.get("theta")
        dev, C, n = mu.device, c["C"], mu.shape[0]
        if c["path"] in ("exact", "pixels"):
            H, W = c["H"], c["W"]
            if c["path"] == "exact":
                ys = torch.linspace(0.5 / H, 1 - 0.5 / H, H, device=dev)
                xs = torch.linspace(0.5 / W, 1 - 0.5 / W, W, device=dev)
                py, px = ys.repeat_interleave(W), xs.repeat(H)
            else:
                py, px = ((s["idx"][b] // W).float() + 0.5) / H, ((s["idx"][b] % W).float() + 0.5) / W
            parts = [_Every(n, py, px)]
        else:
            scale32 = F.softplus(p32["log_scale"]) + 1e-4
            lev = _routes(c, scale32)
            parts = [_Tiles(c, p32["mu"], scale32, Hl, Wl, (lev == l).nonzero()[:, 0])
                     for l, (Hl, Wl) in enumerate(_levels(c))]
        fields = []
        for t in parts:
            f = t.zeros(2 + C, dev)
            for g, at, py, px in t.chunks():
                lg, w = _terms(c, mu[g], scd[g], None if th is None else th[g], op[g], py, px)
                _add(f, at, [lg, w] + [w * col[g, k][:, None, None] for k in range(C)])
            fields.append(t.canvas(f).contiguous().requires_grad_(True))
        tot = fields[0]
        for f in fields[1:]:
            tot = tot + F.interpolate(f[None], size=tot.shape[1:], mode="bilinear", align_corners=False)[0]
        bg = p["bg"].requires_grad_(True)
        T = torch.exp(tot[0])
        img = (1 - T) * tot[2:] / tot[1].clamp_min(1e-8) + T * bg[:, None, None]
        shape = (C, c["n_px"]) if c["path"] == "pixels" else (C, c["H"], c["W"])
        out = {"image": img.detach().reshape(shape)}
        if c["train"]:
            up = torch.autograd.grad(img, fields + [bg], s["gout"][b].double().reshape(img.shape))
            gm, gs, gc, go = (torch.zeros_like(t) for t in (mu, scd, col, op))
            gt = None if th is None else torch.zeros_like(th)
            for t, d in zip(parts, up[:-1]):
                d = t.tiled(d)
                for g, at, py, px in t.chunks():
                    x = [v[g].detach().requires_grad_(True) for v in (mu, scd, op)]
                    if th is not None:
                        x.append(th[g].detach().requires_grad_(True))
                    dd = _get(d, at)
                    lg, w = _terms(c, x[0], x[1], x[3] if th is not None else None, x[2], py, px)
                    wd = w.detach()
                    da = dd[1]
                    for k in range(C):
                        da = da + dd[2 + k] * col[g, k][:, None, None]
                        _gather(gc[:, k], g, (dd[2 + k] * wd).sum((1, 2)))
                    gr = torch.autograd.grad((dd[0] * lg + da * w).sum(), x)
                    for acc, v in zip((gm, gs, go, gt), gr):
                        _gather(acc, g, v)
            out.update(g_mu=gm, g_log_scale=torch.autograd.grad(sc, ls, gs)[0], g_color=gc, g_opacity=go, g_bg=up[-1])
            if th is not None:
                out["g_theta"] = gt
        outs.append(out)
    return {k: torch.stack([o[k] for o in outs]) for k in outs[0]}
