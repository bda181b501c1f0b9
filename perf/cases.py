"""Performance cases: the calls a user's program makes, over the sizes it makes them at.

Every case goes through a public entry point (``ndimage.draw_lines``,
``ndimage.accumulate_lines``, ``batch.Plan``, ``autograd.render`` /
``render_plan``, ``label.label_threshold`` and what is computed from its
result, ``label.binary_dilation``) on tensors that are
already on the GPU.  ``exact`` restates the drawn images, gradients and region
quantities in 64 bits from their closed forms (a pixel's value is the profile
of its distance to the segment over the width), with none of the package's
code.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cbclib_v2_amd import autograd, batch, label as cl, ndimage

DEV = 'cuda'
KERNELS = ('biweight', 'gaussian', 'parabolic', 'rectangular', 'triangular')


def listed():
    return [
        # one detector frame, a simulated pattern of 1000 lines: the smallest draw, its cost is launches and waits
        dict(name='draw_frame', kind='draw', frames=1, height=512, width=512, lines=1000, length=0.0, wmin=1.0,
             wmax=4.0, kernel='triangular', overlap='sum', dtype='float32'),
        # a stack of large detector frames drawn in one call
        dict(name='draw_stack', kind='draw', frames=64, height=2048, width=2048, lines=128000, length=400.0, wmin=2.0,
             wmax=6.0, kernel='gaussian', overlap='sum', dtype='float32'),
        # double precision images (the type of arrays made by NumPy programs), frames of a ragged size
        dict(name='draw_f64', kind='draw', frames=7, height=1003, width=1205, lines=14000, length=300.0, wmin=1.0,
             wmax=5.0, kernel='gaussian', overlap='sum', dtype='float64'),
        # largest value instead of sum, the default profile: footprints of predicted lines on ragged frames
        dict(name='draw_max', kind='draw', frames=24, height=1021, width=1531, lines=36000, length=250.0, wmin=1.0,
             wmax=4.0, kernel='rectangular', overlap='max', dtype='float32'),
        # a scan of frames with uneven line counts and a profile per line, drawn again and again through a plan
        dict(name='draw_mixed', kind='plan', frames=256, height=1024, width=1024, least=100, most=20000, length=400.0,
             wmin=2.0, wmax=6.0),
        # one step of a fit of all lines of a stack to measured frames: render, squared difference, gradient
        dict(name='fit_stack', kind='fit', frames=32, height=1024, width=1024, lines=160000, length=400.0, wmin=2.0,
             wmax=6.0, kernel='biweight', plan=True),
        # the same step for one small frame without a plan: interactive refinement of a single pattern
        dict(name='fit_frame', kind='fit', frames=1, height=509, width=643, lines=700, length=200.0, wmin=1.0,
             wmax=4.0, kernel='gaussian', plan=False),
        # rotation maps: lines grouped into terms, largest value within a term, terms added into frames
        dict(name='terms', kind='terms', frames=16, height=512, width=512, terms=4000, per_term=16, length=60.0,
             wmin=1.0, wmax=3.0, kernel='gaussian', inner='max', outer='sum'),
        # lines in reciprocal-space volumes
        dict(name='draw_volumes', kind='volume', frames=16, depth=64, height=128, width=128, lines=50000, length=40.0,
             wmin=1.0, wmax=3.0, kernel='gaussian', overlap='sum'),
        # streak detection, labels of a large stack: threshold and 8-connected components per frame
        dict(name='label_stack', kind='label', frames=64, height=2048, width=2048, lines=128000, length=400.0,
             wmin=2.0, wmax=6.0, vmin=0.5, connectivity=2, npts=1),
        # streak detection of a short ragged stack up to the lines: components, their line fits and p-values
        dict(name='regions', kind='regions', frames=6, height=1031, width=1275, length=60.0, wmin=2.0, wmax=5.0,
             vmin=0.15, connectivity=2, npts=5),
        # a bad-pixel or streak mask grown under a second mask, rows of no whole number of words
        dict(name='dilate_mask', kind='dilate', frames=16, height=1062, width=1028, lines=6000, length=300.0,
             wmin=1.0, wmax=4.0, iterations=3, masked=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame(rng, lo, hi):
    """Height and width: often equal and a multiple of 64, otherwise any."""
    if rng.random() < 0.4:
        s = 64 * max(1, _log(rng, lo, hi) // 64)
        return s, s
    return _log(rng, lo, hi), _log(rng, lo, hi)


def draw(rng):
    """One more case: a kind, and sizes spread over its range (frames and lines over their logarithm)."""
    kind = rng.choice(['draw', 'draw', 'draw64', 'plan', 'fit_plan', 'fit', 'terms', 'volume', 'label',
                       'regions', 'dilate'])
    if kind == 'volume':
        frames, d, h, w = _log(rng, 1, 16), _log(rng, 16, 64), _log(rng, 40, 128), _log(rng, 40, 128)
        return dict(kind='volume', frames=frames, depth=d, height=h, width=w, lines=_log(rng, 100, 50000),
                    length=rng.uniform(10.0, 40.0), wmin=1.0, wmax=rng.uniform(1.5, 3.0), kernel=rng.choice(KERNELS),
                    overlap=rng.choice(['sum', 'max']))
    if kind == 'terms':
        frames = _log(rng, 1, 16)
        h, w = _frame(rng, 200, 512)
        return dict(kind='terms', frames=frames, height=h, width=w, terms=_log(rng, 50, 4000),
                    per_term=rng.randint(2, 16), length=rng.uniform(10.0, 60.0), wmin=1.0,
                    wmax=rng.uniform(1.5, 3.0), kernel=rng.choice(KERNELS),
                    **dict(zip(('inner', 'outer'), rng.choice([('max', 'sum'), ('sum', 'max'), ('max', 'sum')]))))
    h, w = _frame(rng, 256, 1500)
    px = h * w
    # lines per frame: from a few to the density of the listed stacks
    wmin = rng.uniform(1.0, 2.0)
    base = dict(height=h, width=w, length=rng.uniform(50.0, 400.0), wmin=wmin, wmax=wmin + rng.uniform(0.5, 4.0))
    if kind in ('draw', 'draw64'):
        frames = _log(rng, 1, max(1, min(64, 60000000 // px)))
        lines = max(1, int(frames * _log(rng, 30, 2000) * (0.5 if kind == 'draw64' else 1.0)))
        return dict(kind='draw', frames=frames, lines=lines, kernel=rng.choice(KERNELS),
                    overlap=rng.choice(['sum', 'sum', 'max']), dtype='float64' if kind == 'draw64' else 'float32',
                    **base)
    if kind == 'plan':
        frames = _log(rng, 4, max(4, min(128, 60000000 // px)))
        least = rng.randint(50, 300)
        return dict(kind='plan', frames=frames, least=least, most=least * rng.randint(4, 30), **base)
    if kind in ('fit', 'fit_plan'):
        plan = kind == 'fit_plan'
        frames = _log(rng, 1, max(1, min(32, (30 if plan else 5) * 1000000 // px)))
        return dict(kind='fit', frames=frames, lines=frames * _log(rng, 100, 5000 if plan else 1500),
                    kernel=rng.choice(('biweight', 'gaussian', 'parabolic', 'triangular')), plan=plan, **base)
    if kind == 'regions':
        base.update(length=rng.uniform(30.0, 150.0), wmin=2.0, wmax=rng.uniform(3.0, 6.0))
        return dict(kind='regions', frames=_log(rng, 1, max(1, min(64, 10000000 // px))), vmin=rng.uniform(0.1, 0.15),
                    connectivity=rng.choice([1, 2, 2]), npts=rng.choice([5, 8]), **base)
    frames = _log(rng, 1, max(1, min(64, 100000000 // px)))
    base['lines'] = frames * _log(rng, 30, 1000)
    if kind == 'dilate':
        return dict(kind='dilate', frames=frames, iterations=rng.randint(1, 4), masked=rng.random() < 0.5, **base)
    return dict(kind='label', frames=frames, vmin=rng.uniform(0.15, 0.35), connectivity=rng.choice([1, 2, 2]),
                npts=rng.choice([1, 3, 5]), **base)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)


def _segments(g, c, n):
    """Rows x0, y0, x1, y1, width: starts uniform in the frame, lengths uniform up to ``length`` in random
    directions (``length`` 0: both ends uniform in the frame)."""
    h, w = c['height'], c['width']
    x0, y0 = _uniform(g, 0.0, w, n), _uniform(g, 0.0, h, n)
    if c['length'] > 0.0:
        a = _uniform(g, 0.0, 2.0 * math.pi, n)
        ln = _uniform(g, min(20.0, 0.1 * c['length']), c['length'], n)
        x1, y1 = x0 + ln * torch.cos(a), y0 + ln * torch.sin(a)
    else:
        x1, y1 = _uniform(g, 0.0, w, n), _uniform(g, 0.0, h, n)
    return torch.stack([x0, y0, x1, y1, _uniform(g, c['wmin'], c['wmax'], n)], 1)


def _even(n, frames):
    """Frame of each of n lines, frame after frame."""
    return torch.div(torch.arange(n, device=DEV) * frames, n, rounding_mode='floor')


def _counts(c):
    """Line counts of the frames of a scan: spread evenly over the logarithm from ``least`` to ``most``."""
    f = np.arange(c['frames']) + 0.5
    return np.round(c['least'] * (c['most'] / c['least']) ** (f / c['frames'])).astype(np.int64)


def _streaks(g, c):
    """Diffraction streaks well apart: one in each cell of a grid over every frame."""
    side = int(c['length'] + 2.0 * c['wmax']) + 6
    ny, nx = max(1, c['height'] // side), max(1, c['width'] // side)
    n = c['frames'] * ny * nx
    k = torch.arange(n, device=DEV)
    cx = (k % nx + 0.5) * (c['width'] / nx)
    cy = (torch.div(k, nx, rounding_mode='floor') % ny + 0.5) * (c['height'] / ny)
    a = _uniform(g, 0.0, 2.0 * math.pi, n)
    half = 0.5 * _uniform(g, 20.0, c['length'], n)
    dx, dy = half * torch.cos(a), half * torch.sin(a)
    lines = torch.stack([cx - dx, cy - dy, cx + dx, cy + dy, _uniform(g, c['wmin'], c['wmax'], n)], 1)
    return lines.float(), torch.div(k, nx * ny, rounding_mode='floor')


def _lines_of(case, seed):
    """(generator, lines in the case's type, frame of every line as int64)."""
    g = _generator(seed)
    if case['kind'] == 'regions':
        return (g,) + _streaks(g, case)
    dt = torch.float64 if case.get('dtype') == 'float64' else torch.float32
    if case['kind'] == 'plan':
        counts = torch.as_tensor(_counts(case), device=DEV)
        counts = counts[torch.randperm(case['frames'], generator=g, device=DEV)]
        n = int(counts.sum())
        idxs = torch.repeat_interleave(torch.arange(case['frames'], device=DEV), counts)
    else:
        n = case['terms'] * case['per_term'] if case['kind'] == 'terms' else case['lines']
        idxs = _even(n, case['frames'])
    return g, _segments(g, case, n).to(dt), idxs


def _measured(case, lines, idxs, g, jitter):
    """Frames as a detector gives them: the lines (moved by up to ``jitter`` px) in fixed point steps, so the same
    for a seed whatever the order of additions."""
    moved = lines.double().clone()
    moved[:, :4] += jitter * torch.randn((moved.shape[0], 4), generator=g, device=DEV, dtype=torch.float64)
    acc = torch.zeros(case['frames'] * case['height'] * case['width'], dtype=torch.int32, device=DEV)
    for ln, fx, pix, u, _ in _pairs(moved.float(), idxs, case['height'], case['width']):
        v = _profile(case.get('kernel', 'gaussian'), u) * 1048576.0
        acc.index_add_(0, pix, torch.round(v).to(torch.int32))
    if case['kind'] == 'regions':   # background noise and a few hot pixels
        acc += torch.round(10000.0 * torch.randn(acc.shape, generator=g, device=DEV)).to(torch.int32)
        acc += 500000 * (torch.rand(acc.shape, generator=g, device=DEV) < 0.0003)
    return (acc.to(torch.float32) / 1048576.0).reshape(case['frames'], case['height'], case['width'])


def _volume_lines(case, seed):
    g = _generator(seed)
    n = case['lines']
    hi = torch.tensor([case['width'], case['height'], case['depth']], device=DEV, dtype=torch.float64)
    p0 = hi * torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float64)
    d = torch.randn((n, 3), generator=g, device=DEV, dtype=torch.float64)
    d = d / d.norm(dim=1, keepdim=True) * _uniform(g, 5.0, case['length'], n, 1)
    lines = torch.cat([p0, p0 + d, _uniform(g, case['wmin'], case['wmax'], n, 1)], 1).float()
    idxs = torch.randint(0, case['frames'], (n,), generator=g, device=DEV)
    return lines, idxs


def _structure(case):
    return cl.Structure([0, 1, 1], case.get('connectivity', 1))


def prepare(case, seed):
    kind = case['kind']
    shape = (case['frames'], case['height'], case['width'])
    if kind == 'volume':
        lines, idxs = _volume_lines(case, seed)
        out = torch.zeros((case['frames'], case['depth']) + shape[1:], dtype=torch.float32, device=DEV)
        return dict(case=case, lines=lines, idxs=idxs.to(torch.int32), out=out)
    g, lines, idxs = _lines_of(case, seed)
    if kind == 'draw':
        return dict(case=case, lines=lines, out=torch.zeros(shape, dtype=lines.dtype, device=DEV),
                    idxs=idxs.to(torch.int64 if lines.dtype == torch.float64 else torch.int32))
    if kind == 'plan':
        kern = torch.where(torch.rand(lines.shape[0], generator=g, device=DEV) < 0.5, 4, 1).to(torch.uint8)
        idxs = idxs.to(torch.int32)
        plan = batch.Plan(shape, lines, idxs, kern, headroom=1.1, tile=64, seg=16)
        return dict(case=case, lines=lines, idxs=idxs, kernels=kern, plan=plan,
                    out=torch.zeros(shape, dtype=torch.float32, device=DEV))
    if kind == 'fit':
        target = _measured(case, lines, idxs, g, 0.5)
        idxs = idxs.to(torch.int32)
        plan = batch.Plan(shape, lines, idxs, kernel=case['kernel'], headroom=1.25) if case['plan'] else None
        return dict(case=case, shape=shape, lines=lines.requires_grad_(True), idxs=idxs, target=target, plan=plan)
    if kind == 'terms':
        terms = torch.arange(case['terms'], device=DEV).repeat_interleave(case['per_term']).to(torch.int32)
        frames = torch.randint(0, case['frames'], (case['terms'],), generator=g, device=DEV).to(torch.int32)
        return dict(case=case, lines=lines, terms=terms, frames=frames,
                    out=torch.zeros(shape, dtype=torch.float32, device=DEV))
    image = _measured(case, lines, idxs, g, 0.0)
    if kind == 'dilate':
        mask = torch.rand(shape, generator=g, device=DEV) < 0.7 if case['masked'] else None
        return dict(case=case, mask=mask, inp=image > 0.3, structure=_structure(case))
    return dict(case=case, image=image, structure=_structure(case))


def run(state):
    case = state['case']
    kind = case['kind']
    if kind in ('draw', 'volume'):
        out = state['out'].zero_()
        return ndimage.draw_lines(out, state['lines'], state['idxs'], 1.0, case['kernel'], case['overlap'])
    if kind == 'plan':
        out = state['out'].zero_()
        return state['plan'].draw(out, state['lines'], state['idxs'], state['kernels'])
    if kind == 'fit':
        lines = state['lines']
        lines.grad = None
        if state['plan'] is not None:
            img = autograd.render_plan(state['plan'], lines, state['idxs'], kernel=case['kernel'])
        else:
            img = autograd.render(lines, state['shape'], state['idxs'], kernel=case['kernel'])
        loss = torch.nn.functional.mse_loss(img, state['target'], reduction='sum')
        loss.backward()
        return {'loss': loss.detach(), 'image': img.detach(), 'grad': lines.grad}
    if kind == 'terms':
        out = state['out'].zero_()
        return ndimage.accumulate_lines(out, state['lines'], state['terms'], state['frames'], 1.0, case['kernel'],
                                        case['inner'], case['outer'])
    if kind == 'dilate':
        return cl.binary_dilation(state['inp'], state['structure'], case['iterations'], state['mask'])
    lab = cl.label_threshold(state['image'], case['vmin'], state['structure'], case['npts'])
    if kind == 'label':
        return {'labels': lab.labels, 'n': int(lab.index.numel())}
    fit = cl.line_fit(lab, state['image'])
    p = cl.p_values(lab, fit, state['image'], 0.3, 1.2 * case['vmin'], 1.5)
    return {'labels': lab.labels, 'index': lab.index, 'lines': fit, 'p': p}


def work(case):
    """Bytes: every input once and every output once (an image that is drawn into: read and written).  Flops: about
    ten for a value, twenty for a gradient, of each pixel that a line covers."""
    kind = case['kind']
    px = case['frames'] * case['height'] * case['width']
    if kind in ('label', 'regions', 'dilate'):
        lab = 8.0 * px
        if kind == 'dilate':
            return {'bytes': (3.0 if case['masked'] else 2.0) * px, 'flops': 8.0 * px * case['iterations']}
        return {'bytes': lab * (2.0 if kind == 'regions' else 1.0), 'flops': 4.0 * px}
    if kind == 'plan':
        n = int(_counts(case).sum())
    elif kind == 'terms':
        n = case['terms'] * case['per_term']
    else:
        n = case['lines']
    w = 0.5 * (case['wmin'] + case['wmax'])
    if kind == 'volume':
        px *= case['depth']
        length = 0.5 * (5.0 + case['length'])
        pairs = n * (math.pi * w * w * length + 4.19 * w ** 3)
        return {'bytes': 8.0 * px + 32.0 * n, 'flops': 10.0 * pairs}
    length = 0.52 * case['length'] if case['length'] else 0.52 * math.sqrt(px / case['frames'])
    pairs = n * (2.0 * w * length + math.pi * w * w)
    size = 8 if case.get('dtype') == 'float64' else 4
    if kind == 'fit':
        return {'bytes': 12.0 * px + 44.0 * n, 'flops': 30.0 * pairs}
    return {'bytes': 2.0 * size * px + 6.0 * size * n, 'flops': 10.0 * pairs}


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------
def _profile(kernel, u):
    """Profile at squared distance over squared width ``u`` in [0, 1]."""
    if kernel == 'biweight':
        return 0.9375 * (1.0 - u) ** 2
    if kernel == 'gaussian':
        return torch.exp(-4.5 * u) / math.sqrt(2.0 * math.pi)
    if kernel == 'parabolic':
        return 0.75 * (1.0 - u)
    if kernel == 'rectangular':
        return torch.ones_like(u)
    return 1.0 - torch.sqrt(u)


def _pairs(lines, idxs, H, W, budget=16000000):
    """Chunks of the pixels within the width of a line: line number, frame, flat pixel, u, and (x, y) of the pixel,
    in the type of ``lines``.  Pixels are taken column by column along the line's longer axis."""
    x0, y0, x1, y1, w = lines.unbind(1)
    tx, ty = x1 - x0, y1 - y0
    steep = ty.abs() > tx.abs()
    a0, a1 = torch.where(steep, y0, x0), torch.where(steep, y1, x1)
    b0, b1 = torch.where(steep, x0, y0), torch.where(steep, x1, y1)
    n_a = torch.where(steep, H, W)
    lo = torch.clamp(torch.ceil(torch.minimum(a0, a1) - w).long(), min=0)
    hi = torch.minimum(torch.floor(torch.maximum(a0, a1) + w).long(), n_a - 1)
    cols = torch.clamp(hi - lo + 1, min=0)
    # pixels across: the band of half-width w * len / |t_a|, at most sqrt(2) w
    rows = int(math.floor(2.0 * math.sqrt(2.0) * float(w.max()))) + 3
    ends = torch.cumsum(cols, 0)
    total = ends.cpu().numpy()
    start, n, step = 0, lines.shape[0], max(1, budget // rows)
    while start < n:
        base = int(total[start - 1]) if start else 0
        stop = max(start + 1, int(np.searchsorted(total, base + step, side='right')))
        k = torch.repeat_interleave(torch.arange(start, stop, device=lines.device), cols[start:stop])
        if k.numel():
            c = lo[k] + torch.arange(k.numel(), device=lines.device) - (ends[k] - cols[k] - base)
            cf = c.to(lines.dtype)
            mid = b0[k] + (b1 - b0)[k] * ((cf - a0[k]) / (a1 - a0)[k])
            b = torch.round(mid).long()[:, None] + (torch.arange(rows, device=lines.device) - rows // 2)[None, :]
            c, k = c[:, None].expand_as(b), k[:, None].expand_as(b)
            sw = steep[k]
            x, y = torch.where(sw, b, c), torch.where(sw, c, b)
            rx, ry = x.to(lines.dtype) - x0[k], y.to(lines.dtype) - y0[k]
            t = torch.clamp((rx * tx[k] + ry * ty[k]) / (tx * tx + ty * ty)[k], 0.0, 1.0)
            u = ((rx - t * tx[k]) ** 2 + (ry - t * ty[k]) ** 2) / (w * w)[k]
            ok = (u <= 1.0) & (x >= 0) & (x < W) & (y >= 0) & (y < H)
            k, x, y, u = k[ok], x[ok], y[ok], u[ok]
            yield k, idxs[k], (idxs[k] * H + y) * W + x, u, (x, y)
        start = stop


def _image(case, lines, idxs, kernel_of=None):
    H, W = case['height'], case['width']
    img = torch.zeros(case['frames'] * H * W, dtype=torch.float64, device=DEV)
    for k, _, pix, u, _ in _pairs(lines, idxs, H, W):
        if kernel_of is None:
            v = _profile(case['kernel'], u)
        else:
            v = torch.where(kernel_of[k] == 4, _profile('triangular', u), _profile('gaussian', u))
        if case.get('overlap', 'sum') == 'sum':
            img.index_add_(0, pix, v)
        else:
            img.scatter_reduce_(0, pix, v, 'amax')
    return img


def _gradient(case, lines, idxs, grad):
    """d sum(grad * image) / d lines."""
    res = torch.zeros((lines.shape[0], 5), dtype=torch.float64, device=DEV)
    kernel = case['kernel']
    for k, _, pix, u, (x, y) in _pairs(lines, idxs, case['height'], case['width']):
        x0, y0, x1, y1, w = lines[k].unbind(1)
        tx, ty = x1 - x0, y1 - y0
        rx, ry = x.double() - x0, y.double() - y0
        t = torch.clamp((rx * tx + ry * ty) / (tx * tx + ty * ty), 0.0, 1.0)
        dx, dy = rx - t * tx, ry - t * ty
        if kernel == 'biweight':
            du = -1.875 * (1.0 - u)
        elif kernel == 'gaussian':
            du = -4.5 * _profile('gaussian', u)
        elif kernel == 'parabolic':
            du = torch.full_like(u, -0.75)
        else:
            du = torch.where(u > 0.0, -0.5 / torch.sqrt(u), torch.zeros_like(u))
        du = du * grad[pix]
        c = -2.0 * du / (w * w)
        s = torch.stack([c * (1.0 - t) * dx, c * (1.0 - t) * dy, c * t * dx, c * t * dy, -2.0 * du * u / w], 1)
        res.index_add_(0, k, s)
    return res


def _volume_image(case, lines, idxs):
    D, H, W = case['depth'], case['height'], case['width']
    img = torch.zeros(case['frames'] * D * H * W, dtype=torch.float64, device=DEV)
    size = torch.tensor([W, H, D], device=DEV)
    for l0 in range(0, lines.shape[0], 2000):
        ln = lines[l0:l0 + 2000]
        p0, p1, w = ln[:, :3], ln[:, 3:6], ln[:, 6]
        t = p1 - p0
        ax = t.abs().argmax(1)
        a0, ta = p0.gather(1, ax[:, None])[:, 0], t.gather(1, ax[:, None])[:, 0]
        lo = torch.clamp(torch.ceil(torch.minimum(a0, a0 + ta) - w).long(), min=0)
        hi = torch.minimum(torch.floor(torch.maximum(a0, a0 + ta) + w).long(), size[ax] - 1)
        cols = torch.clamp(hi - lo + 1, min=0)
        k = torch.repeat_interleave(torch.arange(ln.shape[0], device=DEV), cols)
        c = lo[k] + torch.arange(k.numel(), device=DEV) - (torch.cumsum(cols, 0) - cols)[k]
        # the plane across the long axis: within sqrt(3) w of the line's point in it
        r = int(math.ceil(math.sqrt(3.0) * float(w.max()))) + 1
        off = torch.arange(-r, r + 1, device=DEV)
        centre = torch.round(p0[k] + t[k] * ((c.double() - a0[k]) / ta[k])[:, None]).long()
        b, e = (ax[k] + 1) % 3, (ax[k] + 2) % 3
        pos = torch.empty((k.numel(), off.numel(), off.numel(), 3), dtype=torch.int64, device=DEV)
        pos[:] = centre[:, None, None, :]
        pos.scatter_(3, ax[k][:, None, None, None].expand(-1, off.numel(), off.numel(), 1),
                     c[:, None, None, None].expand(-1, off.numel(), off.numel(), 1))
        pos.scatter_add_(3, b[:, None, None, None].expand(-1, off.numel(), off.numel(), 1),
                         off[None, :, None, None].expand(k.numel(), -1, off.numel(), 1))
        pos.scatter_add_(3, e[:, None, None, None].expand(-1, off.numel(), off.numel(), 1),
                         off[None, None, :, None].expand(k.numel(), off.numel(), -1, 1))
        pos = pos.reshape(-1, 3)
        k = k.repeat_interleave(off.numel() ** 2)
        d = pos.double() - p0[k]
        s = torch.clamp((d * t[k]).sum(1) / (t * t).sum(1)[k], 0.0, 1.0)
        u = ((d - s[:, None] * t[k]) ** 2).sum(1) / (w * w)[k]
        ok = (u <= 1.0) & (pos >= 0).all(1) & (pos < size).all(1)
        k, pos, u = k[ok], pos[ok], u[ok]
        pix = ((idxs[l0:l0 + 2000][k] * D + pos[:, 2]) * H + pos[:, 1]) * W + pos[:, 0]
        if case['overlap'] == 'sum':
            img.index_add_(0, pix, _profile(case['kernel'], u))
        else:
            img.scatter_reduce_(0, pix, _profile(case['kernel'], u), 'amax')
    return img.reshape(case['frames'], D, H, W)


def _terms_image(case, lines, frames):
    H, W = case['height'], case['width']
    out = torch.zeros(case['frames'], H * W, dtype=torch.float64, device=DEV)
    per = case['per_term']
    step = max(1, 40000000 // (H * W))
    for t0 in range(0, case['terms'], step):
        n = min(step, case['terms'] - t0)
        local = torch.arange(n, device=DEV).repeat_interleave(per)
        part = dict(case, frames=n, overlap=case['inner'])
        buf = _image(part, lines[t0 * per:(t0 + n) * per], local).reshape(n, H * W)
        if case['outer'] == 'sum':
            out.index_add_(0, frames[t0:t0 + n], buf)
        else:
            out.scatter_reduce_(0, frames[t0:t0 + n, None].expand(-1, H * W), buf, 'amax')
    return out.reshape(case['frames'], H, W)


def _components(mask, connectivity, npts):
    """Component of every pixel (1.. in raster order of first pixels, 0: none) per frame: smallest neighbouring
    index, then pointer jumping, until nothing changes."""
    F, H, W = mask.shape
    P = mask.numel()
    far = torch.full((F, H + 2, W + 2), P, dtype=torch.int64, device=DEV)
    lab = torch.where(mask, torch.arange(P, device=DEV).reshape(mask.shape), P)
    steps = [(0, 1), (0, -1), (1, 0), (-1, 0)]
    steps += [(1, 1), (1, -1), (-1, 1), (-1, -1)] if connectivity == 2 else []
    while True:
        far[:, 1:-1, 1:-1] = lab
        new = lab
        for dy, dx in steps:
            new = torch.minimum(new, far[:, 1 + dy:H + 1 + dy, 1 + dx:W + 1 + dx])
        new = torch.where(mask, new, P).reshape(-1)
        # a root takes the smallest index that any pixel of its tree saw
        low = torch.cat([torch.arange(P, device=DEV), torch.full((1,), P, device=DEV)])
        low.scatter_reduce_(0, lab.reshape(-1), new, 'amin')
        low[P] = P
        for _ in range(4):
            low = low[low]
        new = torch.where(mask.reshape(-1), torch.minimum(low[lab.reshape(-1)], low[new]), P).reshape(mask.shape)
        if torch.equal(new, lab):
            break
        lab = new
    on = lab[mask]
    ids, inv, cnt = torch.unique(on, return_inverse=True, return_counts=True)
    keep = cnt >= npts
    rank = torch.where(keep, torch.cumsum(keep.long(), 0), 0)
    res = torch.zeros(mask.shape, dtype=torch.int64, device=DEV)
    res[mask] = rank[inv]
    return res, int(keep.sum())


def _region_lines(lab, n, image):
    """Major axis of each component's covariance ellipse, x0, y0, z0, x1, y1, z1."""
    at = (lab > 0).nonzero()
    k = lab[lab > 0] - 1
    v = torch.clamp(image[lab > 0].double(), min=0.0)
    p = at.flip(1).double()
    mu = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, k, v)
    cx = torch.zeros((n, 3), dtype=torch.float64, device=DEV).index_add_(0, k, v[:, None] * p) / mu[:, None]
    d = p - cx[k]
    cov = torch.zeros((n, 3), dtype=torch.float64, device=DEV)
    cov.index_add_(0, k, v[:, None] * torch.stack([d[:, 0] ** 2, d[:, 1] ** 2, d[:, 0] * d[:, 1]], 1))
    xx, yy, xy = (cov / mu[:, None]).unbind(1)
    noise = 1e-12 * (cx[:, 0] ** 2 + cx[:, 1] ** 2)
    dif, xy2 = xx - yy, 2.0 * xy
    dif, xy2 = torch.where(dif.abs() <= noise, 0.0, dif), torch.where(xy2.abs() <= noise, 0.0, xy2)
    a = 0.5 * torch.atan2(xy2, dif)
    hw = torch.sqrt(torch.clamp(2.0 * math.log(2.0) * (xx + yy + torch.sqrt(xy2 ** 2 + dif ** 2)), min=0.0))
    tau = torch.stack([torch.cos(a), torch.sin(a), torch.zeros_like(a)], 1) * hw[:, None]
    return torch.cat([cx + tau, cx - tau], 1)


def _region_p(lab, n, image, lines, p0, vmin, xtol):
    at = (lab > 0).nonzero()
    k = lab[lab > 0] - 1
    p = at.flip(1).double()
    a, b = lines[:, :3], lines[:, 3:]
    t, mid = b - a, 0.5 * (a + b)
    mag = (t * t).sum(1)
    s = torch.clamp(((p - mid[k]) * t[k]).sum(1) / torch.where(mag > 0, mag, 1.0)[k], -0.5, 0.5)
    near = ((p - mid[k] - s[:, None] * t[k]) ** 2).sum(1).sqrt() < xtol
    hit = near & (image[lab > 0] >= vmin)
    tot = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, k, near.double())
    sig = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, k, hit.double())
    res = torch.full((n,), -math.inf, dtype=torch.float64, device=DEV)
    for j in range(int(tot.max()) + 1 if n else 0):
        i = sig + j
        term = (torch.lgamma(tot + 1) - torch.lgamma(i + 1) - torch.lgamma(torch.clamp(tot - i, min=0.0) + 1) +
                i * math.log(p0) + (tot - i) * math.log1p(-p0))
        res = torch.where(i <= tot, torch.logaddexp(res, term), res)
    return torch.where(sig == 0, 0.0, res)


def exact(case, seed):
    kind = case['kind']
    shape = (case['frames'], case['height'], case['width'])
    if kind in ('label', 'dilate'):
        return None     # whole numbers and truth values only
    if kind == 'volume':
        lines, idxs = _volume_lines(case, seed)
        return _volume_image(case, lines.double(), idxs)
    g, lines, idxs = _lines_of(case, seed)
    if kind == 'regions':
        image = _measured(case, lines, idxs, g, 0.0)
        lab, n = _components(image > case['vmin'], case['connectivity'], case['npts'])
        fit = _region_lines(lab, n, image)
        # (the p-values of the fitted lines as they are handed over, in the image's type)
        p = _region_p(lab, n, image, fit.float().double(), 0.3, 1.2 * case['vmin'], 1.5)
        return {'labels': None, 'index': None, 'lines': fit, 'p': p}
    if kind == 'plan':
        kern = torch.where(torch.rand(lines.shape[0], generator=g, device=DEV) < 0.5, 4, 1).to(torch.uint8)
        return _image(case, lines.double(), idxs, kern).reshape(shape)
    if kind == 'terms':
        frames = torch.randint(0, case['frames'], (case['terms'],), generator=g, device=DEV)
        return _terms_image(case, lines.double(), frames)
    if kind == 'fit':
        target = _measured(case, lines, idxs, g, 0.5).double().reshape(-1)
        img = _image(case, lines.double(), idxs)
        diff = img - target
        return {'loss': (diff * diff).sum(), 'image': img.reshape(shape),
                'grad': _gradient(case, lines.double(), idxs, 2.0 * diff)}
    return _image(case, lines.double(), idxs).reshape(shape)
