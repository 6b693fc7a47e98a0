"""Timed cases of the render path, through the package's public entry points.

A case names an entry (`RenderFunction`, a resident `DeviceScene`, a `Batch`, the
generative front end), a kind of scene and its sizes:

  render      serialize_scene + RenderFunction.apply (+ L2 loss + backward): how an
              optimisation script or a viewer renders one scene
  resident    one device scene kept over the steps of a loop: update with new values,
              forward, loss gradient, backward, gradients (the C ABI's training loop)
  batch       many uneven scenes, resident, one launch per stage and direction
  generative  bezier_render on a batch of stroke sequences, and its backward

Scenes are drawn from the seed: closed Bezier paths with fills and strokes, open
strokes, drawings of mixed shapes, one circle, and long paths.
"""
import math
import random

import numpy as np
import torch

import diffvg_amd as dvg
from diffvg_amd import _lib, diffvg, generative
from diffvg_amd.render_pytorch import flatten_args

FILTERS = ('box', 'tent', 'parabolic', 'hann', 'gaussian')


# ------------------------------------------------------------------------- the cases
def listed():
    return [
        # fitting one primitive to a target (the single_circle app): launches and latency
        dict(name='circle_256', entry='render', scene='circle', w=256, h=256, n=1, nsx=2, nsy=2, filter='box',
             radius=0.5, output='color', prefilter=False, train=True, direct=False),
        # a drawing as an SVG file holds it: opaque and translucent shapes of every kind,
        # gradients, transforms, over a background; odd sizes, 3x2 samples, tent filter
        dict(name='drawing_333x217', entry='render', scene='mixed', w=333, h=217, n=40, nsx=3, nsy=2, filter='tent',
             radius=1.0, output='color', prefilter=False, train=True, direct=False),
        # image fitting with closed paths, wide filter
        dict(name='paths_300_512', entry='render', scene='closed', w=512, h=512, n=300, lo=4, hi=20, spread=15.0,
             stroked=0.3, nsx=2, nsy=2, filter='gaussian', radius=1.5, output='color', prefilter=False, train=True,
             direct=False),
        # the same optimisation with analytic prefiltering instead of edge sampling
        dict(name='paths_300_512_prefiltered', entry='render', scene='closed', w=512, h=512, n=300, lo=4, hi=20,
             spread=15.0, stroked=0.3, nsx=2, nsy=2, filter='gaussian', radius=1.5, output='color', prefilter=True,
             train=True, direct=False),
        # painterly rendering at full size: a loop over a resident scene
        dict(name='strokes_2048_512', entry='resident', scene='strokes', w=512, h=512, n=2048, step=20.0, nsx=2,
             nsy=2, filter='box', radius=0.5, output='color', prefilter=False, train=True),
        # a small painterly run with gradients written straight into the leaves
        dict(name='strokes_200_224', entry='render', scene='strokes', w=224, h=224, n=200, step=12.0, nsx=2, nsy=2,
             filter='box', radius=0.5, output='color', prefilter=False, train=True, direct=True),
        # the generator's rasteriser in a GAN: a batch of stroke sequences at 32x32
        dict(name='generative_32', entry='generative', scene='strokes', w=32, h=32, n=16, items=32, nsx=2, nsy=2,
             filter='box', radius=0.5, output='color', prefilter=False, train=True),
        # many scenes of uneven size at once, gradient fills among them
        dict(name='uneven_batch_256', entry='batch', scene='closed', w=256, h=256, n=512, items=256, lo=2, hi=8,
             stroked=0.0, nsx=2, nsy=2, filter='box', radius=0.5, output='color', prefilter=False, train=True),
        # fitting a signed distance field (the single_curve_sdf app, with many curves)
        dict(name='sdf_300_256', entry='render', scene='closed', w=256, h=256, n=300, lo=2, hi=8, spread=9.0,
             stroked=0.3, nsx=1, nsy=1, filter='box', radius=0.5, output='sdf', prefilter=False, train=True,
             direct=False),
        # looking at a finished drawing: forward only, a large odd canvas
        dict(name='view_1021x767', entry='render', scene='closed', w=1021, h=767, n=1000, lo=2, hi=8, spread=18.0,
             stroked=0.3, nsx=2, nsy=2, filter='box', radius=0.5, output='color', prefilter=False, train=False,
             direct=False),
        # traced outlines: a path of 1,500 segments and a stroke of 600 on a small canvas
        dict(name='long_paths_128', entry='render', scene='long', w=128, h=128, n=1500, nsx=2, nsy=2, filter='box',
             radius=0.5, output='color', prefilter=False, train=True, direct=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['closed', 'closed', 'closed', 'strokes', 'strokes', 'mixed', 'circle', 'long', 'batch',
                       'generative', 'resident', 'sdf'])
    w, h = _log_int(rng, 24, 640), _log_int(rng, 24, 640)
    nsx, nsy = rng.choice([(2, 2), (2, 2), (1, 1), (3, 2), (3, 3), (4, 4)])
    if w * h * nsx * nsy > 1100000:  # no larger than the listed ones
        nsx = nsy = 1
    filt = rng.choice(FILTERS)
    radius = 0.5 if filt == 'box' else rng.choice([1.0, 1.5])
    c = dict(entry='render', scene=kind, w=w, h=h, n=1, nsx=nsx, nsy=nsy, filter=filt, radius=radius, output='color',
             prefilter=False, train=rng.random() < 0.8, direct=rng.random() < 0.3)
    if kind == 'closed' or kind == 'sdf':
        n = _log_int(rng, 1, 400)
        lo = rng.randint(2, 5)
        c.update(scene='closed', n=n, lo=lo, hi=lo + rng.randint(0, 14), stroked=rng.choice([0.0, 0.3, 1.0]),
                 spread=round(max(1.0, 0.5 * math.sqrt(w * h / n) * rng.uniform(0.3, 1.0)), 3))
        if kind == 'sdf':
            c.update(output='sdf', nsx=1, nsy=1, filter='box', radius=0.5, n=min(n, 200))
        elif rng.random() < 0.35:
            c.update(prefilter=True)
    elif kind == 'strokes' or kind == 'resident':
        n = _log_int(rng, 1, 1500 if kind == 'resident' else 300)
        c.update(scene='strokes', n=n, step=round(rng.uniform(0.01, 0.04) * max(w, h), 3))
        if kind == 'resident':
            c.pop('direct')
            c.update(entry='resident', train=True)
    elif kind == 'mixed':
        c.update(n=_log_int(rng, 6, 200))
    elif kind == 'long':
        c.update(n=_log_int(rng, 40, 1500), w=min(w, 200), h=min(h, 200))
    elif kind == 'batch':
        c.pop('direct')
        side = _log_int(rng, 28, 200)
        c.update(entry='batch', scene='closed', w=side, h=side, n=_log_int(rng, 4, 300), items=_log_int(rng, 2, 64),
                 lo=2, hi=rng.randint(2, 8), stroked=0.0, nsx=2, nsy=2, train=True)
    elif kind == 'generative':
        c.pop('direct')
        side = rng.choice([24, 32, 47, 64])
        c.update(entry='generative', scene='strokes', w=side, h=side, n=rng.randint(1, 24), items=rng.randint(1, 48),
                 nsx=2, nsy=2, filter='box', radius=0.5, train=True)
    return c


# ------------------------------------------------------------------------- scenes
# A scene is a dict of plain numpy values, from which both the package's objects and the
# 64-bit evaluation are made.  Its topology (segment counts, which shapes are stroked, which
# paints are gradients and their stops) follows from the case, its values from the seed.
def _const(rng, lo=0.3):
    return ('const', np.r_[rng.uniform(0, 1, 3), rng.uniform(lo, 1.0)].astype(np.float32))


def _gradient(rng, top, centre, spread):
    ns = int(top.integers(2, 5))
    offs = np.sort(rng.uniform(0, 1, ns)).astype(np.float32)
    offs[0] = 0.0
    cols = rng.uniform(0, 1, (ns, 4)).astype(np.float32)
    if top.uniform() < 0.5:
        return ('linear', (centre - spread).astype(np.float32), (centre + spread).astype(np.float32), offs, cols)
    return ('radial', centre.astype(np.float32), np.full(2, 2 * spread, np.float32), offs, cols)


def _path(pts, ncp, closed, width):
    return dict(kind='path', pts=np.asarray(pts, np.float32), ncp=np.asarray(ncp, np.int32), closed=closed,
                width=np.float32(width))


def _group(shape, fill=None, stroke=None, even_odd=False, xform=None):
    return dict(shape=shape, fill=fill, stroke=stroke, even_odd=even_odd, xform=xform)


def _closed_scene(rng, w, h, n, lo, hi, spread, stroked, grad_frac=0.0):
    shapes, groups = [], []
    top = np.random.default_rng([n, lo, hi])
    for i in range(n):
        nseg = int(top.integers(lo, hi + 1))
        centre = rng.uniform((0, 0), (w, h))
        pts = centre + rng.normal(0, spread, (3 * nseg, 2))
        has_stroke = top.uniform() < stroked
        shapes.append(_path(pts, np.full(nseg, 2), True, rng.uniform(0.5, 3.0) if has_stroke else 1.0))
        fill = _gradient(rng, top, centre, spread) if top.uniform() < grad_frac else _const(rng)
        groups.append(_group(i, fill, _const(rng, 0.0) if has_stroke else None, True))
    return shapes, groups


def _stroke_scene(rng, w, h, n, step):
    shapes, groups = [], []
    for i in range(n):
        p0 = rng.uniform((0, 0), (w, h))
        pts = np.vstack([p0, p0 + np.cumsum(rng.normal(0, step, (9, 2)), axis=0)])
        shapes.append(_path(pts, np.full(3, 2), False, rng.uniform(1.0, 4.0)))
        groups.append(_group(i, None, _const(rng, 0.0)))
    return shapes, groups


def _mixed_scene(rng, w, h, n):
    """Circles, ellipses, rects, polygons, quadratic and cubic outlines, open strokes, some
    under a rotation, two thirds of the fills opaque (as in drawings)."""
    shapes, groups = [], []
    size = 0.5 * math.sqrt(w * h / max(n, 4))
    top = np.random.default_rng([n, 1])
    for i in range(n):
        c = rng.uniform((0, 0), (w, h))
        r = size * rng.uniform(0.4, 1.6)
        kind = i % 7
        xform = None
        if i % 4 == 3:
            a, s = rng.uniform(-0.6, 0.6), rng.uniform(0.8, 1.25)
            rot = s * np.array([[math.cos(a), -math.sin(a)], [math.sin(a), math.cos(a)]])
            xform = np.eye(3)
            xform[:2, :2] = rot
            xform[:2, 2] = c - rot @ c
            xform = xform.astype(np.float32)
        fill = _const(rng, 0.4) if i % 3 == 0 else ('const', np.r_[rng.uniform(0, 1, 3), 1.0].astype(np.float32))
        if i % 5 == 4:
            fill = _gradient(rng, top, c, r)
        stroke = _const(rng, 0.5) if i % 2 else None
        if kind == 0:
            shapes.append(dict(kind='circle', radius=np.float32(r), centre=c.astype(np.float32),
                               width=np.float32(rng.uniform(0.5, 2.0))))
        elif kind == 1:
            shapes.append(dict(kind='ellipse', radius=np.array([r, 0.6 * r], np.float32), centre=c.astype(np.float32),
                               width=np.float32(1.0)))
            stroke = None
        elif kind == 2:
            shapes.append(dict(kind='rect', lo=(c - [r, 0.7 * r]).astype(np.float32),
                               hi=(c + [r, 0.7 * r]).astype(np.float32), width=np.float32(rng.uniform(0.5, 2.0))))
        else:
            ang = np.sort(rng.uniform(0, 2 * math.pi, 5))
            ring = c + r * np.stack([np.cos(ang), np.sin(ang)], 1)
            if kind == 3:  # polygon
                shapes.append(_path(ring, np.zeros(5), True, rng.uniform(0.5, 2.0)))
            elif kind == 4:  # quadratic outline
                mid = 0.5 * (ring + np.roll(ring, -1, 0)) + rng.normal(0, 0.2 * r, (5, 2))
                shapes.append(_path(np.stack([ring, mid], 1).reshape(-1, 2), np.ones(5), True, rng.uniform(0.5, 2.0)))
            elif kind == 5:  # cubic outline
                nxt = np.roll(ring, -1, 0)
                m1 = ring + (nxt - ring) / 3 + rng.normal(0, 0.2 * r, (5, 2))
                m2 = ring + 2 * (nxt - ring) / 3 + rng.normal(0, 0.2 * r, (5, 2))
                shapes.append(_path(np.stack([ring, m1, m2], 1).reshape(-1, 2), np.full(5, 2), True,
                                    rng.uniform(0.5, 2.0)))
            else:  # open pen line: a line, a quadratic and a cubic piece
                pts = c + np.cumsum(rng.normal(0, 0.5 * r, (7, 2)), axis=0)
                shapes.append(_path(pts, [0, 1, 2], False, rng.uniform(0.5, 2.0)))
                fill, stroke = None, _const(rng, 0.5)
        groups.append(_group(i, fill, stroke, False, xform))
    return shapes, groups


def _long_scene(rng, w, h, n):
    c = np.array([w / 2, h / 2])
    t = np.linspace(0, 2 * math.pi, 3 * n, endpoint=False)
    rad = 0.36 + 0.05 * np.sin(37 * t) + rng.normal(0, 0.003, t.shape)
    ring = c + np.stack([w * rad * np.cos(t), h * rad * np.sin(t)], 1)
    m = max(1, 2 * n // 5)
    u = np.linspace(0, 6 * math.pi, 3 * m + 1)
    sr = 0.04 + 0.018 * u + rng.normal(0, 0.0005, u.shape)
    spiral = c + np.stack([w * sr * np.cos(u), h * sr * np.sin(u)], 1)
    shapes = [dict(kind='rect', lo=np.array([0.1 * w, 0.2 * h], np.float32), hi=np.array([0.8 * w, 0.7 * h], np.float32),
                   width=np.float32(1.0)),
              _path(ring, np.full(n, 2), True, 1.2), _path(spiral, np.full(m, 2), False, 1.5)]
    return shapes, [_group(0, _const(rng)), _group(1, _const(rng), _const(rng, 0.5)),
                    _group(2, None, _const(rng, 0.5))]


def _scene(case, rng):
    w, h, n = case['w'], case['h'], case['n']
    if case['scene'] == 'circle':
        c = rng.uniform((0.4 * w, 0.4 * h), (0.6 * w, 0.6 * h)).astype(np.float32)
        shapes = [dict(kind='circle', radius=np.float32(0.16 * min(w, h) * rng.uniform(0.8, 1.2)), centre=c,
                       width=np.float32(1.0))]
        groups = [_group(0, ('const', np.r_[rng.uniform(0, 1, 3), 1.0].astype(np.float32)))]
    elif case['scene'] == 'closed':
        shapes, groups = _closed_scene(rng, w, h, n, case['lo'], case['hi'], case['spread'], case['stroked'])
    elif case['scene'] == 'strokes':
        shapes, groups = _stroke_scene(rng, w, h, n, case['step'])
    elif case['scene'] == 'mixed':
        shapes, groups = _mixed_scene(rng, w, h, n)
    else:
        shapes, groups = _long_scene(rng, w, h, n)
    return dict(w=w, h=h, shapes=shapes, groups=groups)


def _batch_scenes(case, seed):
    """Sizes are a quarter, a half or the whole of the case's; path counts log-uniform up to
    its n; a tenth of the fills are gradients.  The sizes and path counts follow from the
    case, the shapes from the seed."""
    sizes = np.random.default_rng([case['w'], case['n'], case['items']])
    rng = np.random.default_rng([seed, 11])
    out = []
    for k in range(case['items']):
        s = max(8, int(case['w'] * sizes.choice([0.11, 0.25, 0.5, 1.0])))
        n = max(1, int(math.exp(sizes.uniform(0, math.log(case['n'])))))
        if k == 0:
            s, n = case['w'], case['n']
        shapes, groups = _closed_scene(rng, s, s, n, case['lo'], case['hi'], s * 60.0 / 512.0, case['stroked'], 0.1)
        out.append(dict(w=s, h=s, shapes=shapes, groups=groups))
    return out


# ------------------------------------------------------------------------- package objects
def _filter(case):
    return dvg.PixelFilter(type=getattr(diffvg.FilterType, case['filter']), radius=torch.tensor(case['radius']))


def _objects(scene, device, train):
    """The scene as the package's shapes and groups; its parameter tensors by kind."""
    vals, slots = [], []

    def leaf(kind, a):
        a = np.asarray(a, np.float32)
        slots.append((kind, a.shape, a.size))
        vals.append(a.reshape(-1))
        return len(slots) - 1

    plan = []
    for s in scene['shapes']:
        names = {'path': ('pts',), 'circle': ('radius', 'centre'), 'ellipse': ('radius', 'centre'),
                 'rect': ('lo', 'hi')}[s['kind']]
        plan.append(([leaf('geometry', s[k]) for k in names], leaf('width', s['width'])))
    paints = []
    for g in scene['groups']:
        paints.append([None if p is None else [leaf('color', a) for a in p[1:]] for p in (g['fill'], g['stroke'])])
    flat = torch.from_numpy(np.concatenate(vals)).to(device)
    tensors = [t.view(shape).clone().requires_grad_(train)
               for t, (_, shape, _) in zip(flat.split([n for _, _, n in slots]), slots)]
    shapes, groups = [], []
    for s, (geo, wid) in zip(scene['shapes'], plan):
        t, width = [tensors[i] for i in geo], tensors[wid]
        if s['kind'] == 'path':
            shapes.append(dvg.Path(num_control_points=torch.from_numpy(s['ncp']), points=t[0], is_closed=s['closed'],
                                   stroke_width=width))
        elif s['kind'] == 'circle':
            shapes.append(dvg.Circle(radius=t[0], center=t[1], stroke_width=width))
        elif s['kind'] == 'ellipse':
            shapes.append(dvg.Ellipse(radius=t[0], center=t[1], stroke_width=width))
        else:
            shapes.append(dvg.Rect(p_min=t[0], p_max=t[1], stroke_width=width))

    def paint(spec, ids):
        if spec is None:
            return None
        t = [tensors[i] for i in ids]
        if spec[0] == 'const':
            return t[0]
        if spec[0] == 'linear':
            return dvg.LinearGradient(begin=t[0], end=t[1], offsets=t[2], stop_colors=t[3])
        return dvg.RadialGradient(center=t[0], radius=t[1], offsets=t[2], stop_colors=t[3])

    for g, (f, s) in zip(scene['groups'], paints):
        kw = {}
        if g['xform'] is not None:
            kw['shape_to_canvas'] = torch.from_numpy(g['xform']).to(device)
        groups.append(dvg.ShapeGroup(shape_ids=torch.tensor([g['shape']], dtype=torch.int32),
                                     fill_color=paint(g['fill'], f), stroke_color=paint(g['stroke'], s),
                                     use_even_odd_rule=g['even_odd'], **kw))
    params = {}
    for t, (kind, _, _) in zip(tensors, slots):
        params.setdefault(kind, []).append(t)
    return shapes, groups, params


def _device_scene(scene, case, device):
    shapes, groups, _ = _objects(scene, 'cpu', False)
    args = dvg.RenderFunction.serialize_scene(scene['w'], scene['h'], shapes, groups, _filter(case))
    return _lib.DeviceScene(flatten_args(args).desc, device.index or 0)


def _uniform(rng, *shape):
    return rng.uniform(0, 1, shape).astype(np.float32)


def _inputs(case, seed):
    """What the seed gives, on the host: (scene or scenes, target, background, render seed)."""
    rng = np.random.default_rng([seed, 5])
    render_seed = int(rng.integers(0, 1 << 20))
    if case['entry'] == 'batch':
        scenes = _batch_scenes(case, seed)
        return scenes, _uniform(rng, sum(s['w'] * s['h'] for s in scenes), 4), None, render_seed
    ch = 1 if case['output'] == 'sdf' else 4
    scene = _scene(case, np.random.default_rng([seed, 7]))
    target = _uniform(rng, case['h'], case['w'], ch)
    if case['output'] == 'sdf':
        target = 0.1 * max(case['w'], case['h']) * (target - 0.5)
    bg = None
    if case['scene'] == 'mixed':
        bg = _uniform(rng, case['h'], case['w'], 4)
        bg[..., 3] = 1.0
    return scene, target, bg, render_seed


# ------------------------------------------------------------------------- one pass
def prepare(case, seed):
    dev = torch.device('cuda:0')
    dvg.set_use_gpu(True)
    dvg.set_device(dev)
    st = dict(case=case, dev=dev)
    if case['entry'] == 'generative':
        rng = np.random.default_rng([seed, 3])
        b, n, s = case['items'], case['n'], case['w']
        for name, v in (('pts', _uniform(rng, b, n, 7, 2) * 1.6 - 0.8), ('widths', _uniform(rng, b, n) * 1.5 + 0.5),
                        ('alphas', _uniform(rng, b, n) * 0.8 + 0.2), ('colors', _uniform(rng, b, n, 3))):
            st[name] = torch.from_numpy(v).to(dev).requires_grad_(True)
        st['target'] = torch.from_numpy(_uniform(rng, b, 3, s, s)).to(dev)
        st['seed'] = int(rng.integers(0, 1 << 20))
        return st
    scene, target, bg, st['seed'] = _inputs(case, seed)
    st['target'] = torch.from_numpy(target).to(dev)
    if case['entry'] == 'render':
        st['shapes'], st['groups'], st['params'] = _objects(scene, dev, case['train'])
        st['background'] = None if bg is None else torch.from_numpy(bg).to(dev)
        st['filter'] = _filter(case)
    elif case['entry'] == 'resident':
        sc = st['scene'] = _device_scene(scene, case, dev)
        d = sc.flat
        st['values'] = {k: torch.from_numpy(d[k].copy()).to(dev) for k in ('points', 'stroke_width', 'color_params')}
    else:
        scenes = [_device_scene(s, case, dev) for s in scene]
        sizes = [(s['w'], s['h']) for s in scene]
        st['image'] = torch.zeros_like(st['target'])
        st['d_image'] = torch.zeros_like(st['target'])
        cut = [w * h for w, h in sizes]

        def views(t):
            return [v.view(h, w, 4) for v, (w, h) in zip(t.split(cut), sizes)]

        common = dict(nsx=case['nsx'], nsy=case['nsy'], seed=st['seed'], use_prefiltering=case['prefilter'])
        st['forward'] = dvg.Batch([(sc, dict(width=w, height=h, render_image=v, **common))
                                   for sc, (w, h), v in zip(scenes, sizes, views(st['image']))], zero_grads=False)
        st['backward'] = dvg.Batch([(sc, dict(width=w, height=h, d_render_image=v, **common))
                                    for sc, (w, h), v in zip(scenes, sizes, views(st['d_image']))], zero_grads=True)
        st['scenes'] = scenes
    return st


def run(st):
    return {'render': _run_render, 'resident': _run_resident, 'batch': _run_batch,
            'generative': _run_generative}[st['case']['entry']](st)


def _run_render(st):
    c = st['case']
    dvg.set_direct_leaf_gradients(c['direct'])
    F = dvg.RenderFunction
    out = dvg.OutputType.sdf if c['output'] == 'sdf' else dvg.OutputType.color
    with torch.set_grad_enabled(c['train']):
        args = F.serialize_scene(c['w'], c['h'], st['shapes'], st['groups'], filter=st['filter'], output_type=out,
                                 use_prefiltering=c['prefilter'])
        img = F.apply(c['w'], c['h'], c['nsx'], c['nsy'], st['seed'], st['background'], *args)
        if not c['train']:
            return {'image': img}
        for ps in st['params'].values():  # zero_grad(set_to_none=True)
            for p in ps:
                p.grad = None
        ((img - st['target']) ** 2).sum().backward()
    res = {'image': img.detach()}
    for kind, ps in st['params'].items():
        res['d_' + kind] = torch.cat([(torch.zeros_like(p) if p.grad is None else p.grad).reshape(-1) for p in ps])
    return res


def _run_resident(st):
    c, sc, dev = st['case'], st['scene'], st['dev']
    stream = torch.cuda.current_stream().cuda_stream
    kw = dict(stream=stream, use_prefiltering=c['prefilter'])
    sc.update(c['radius'], stream, **st['values'])
    img = torch.zeros(c['h'], c['w'], 4, device=dev)
    sc.render(c['w'], c['h'], c['nsx'], c['nsy'], st['seed'], render_image=img, **kw)
    d_img = 2.0 * (img - st['target'])
    sc.zero_grads(stream)
    sc.render(c['w'], c['h'], c['nsx'], c['nsy'], st['seed'], d_render_image=d_img, **kw)
    block, at = sc.grads_device(dev, stream)
    res = {'image': img}
    for kind, v in st['values'].items():
        res['d_' + kind] = block[at[kind]:at[kind] + v.numel()]
    return res


def _run_batch(st):
    stream = torch.cuda.current_stream().cuda_stream
    st['image'].zero_()
    st['forward'].render(stream)
    torch.mul(st['image'] - st['target'], 2.0, out=st['d_image'])
    st['backward'].render(stream)
    d_color, d_rest = [], []
    for sc in st['scenes']:
        block, at = sc.grads_device(st['dev'], stream)
        f = sc.flat
        d_color.append(block[at['color_params']:at['color_params'] + f['num_color_params']])
        d_rest.append(block[at['points']:at['points'] + 2 * f['num_points_total']])
    return {'image': st['image'], 'd_color_params': torch.cat(d_color), 'd_points': torch.cat(d_rest)}


def _run_generative(st):
    leaves = [st['pts'], st['widths'], st['alphas'], st['colors']]
    for p in leaves:
        p.grad = None
    # the front end jitters the points and draws its render seeds
    torch.manual_seed(st['seed'])
    random.seed(st['seed'])
    out, _ = generative.bezier_render(*leaves[:3], canvas_size=st['case']['w'], colors=st['colors'])
    ((out - st['target']) ** 2).sum().backward()
    return {'image': out.detach(), 'd_points': st['pts'].grad, 'd_widths': st['widths'].grad,
            'd_alphas': st['alphas'].grad, 'd_colors': st['colors'].grad}


# ------------------------------------------------------------------------- cost, tolerance
def work(case):
    """Bytes: parameters in, image out; for a training step also the target in and the
    gradients out.  Operations: every sample of the image (and, with edge sampling, both
    sides of as many boundary samples) takes a position, tests the shapes whose boxes hold
    it and composites those that cover it.  A box holds a sample of a canvas `area` large
    with probability box / area; a test costs a crossing test of the few segments level
    with the sample (fills) or a distance to one curve (strokes, prefiltering, distance
    fields)."""
    if case['entry'] == 'batch':
        scenes = [(s['w'], s['h'], len(s['shapes'])) for s in _batch_scenes(case, 0)]
    else:
        scenes = [(case['w'], case['h'], case['n'])] * case.get('items', 1)
    spp = case['nsx'] * case['nsy']
    values = {'circle': 7, 'closed': 3 * (case.get('lo', 2) + case.get('hi', 2)) + 5, 'strokes': 25, 'mixed': 16,
              'long': 6}[case['scene']]
    nbytes = flops = 0.0
    for w, h, n in scenes:
        params = 4.0 * values * (n + (2 * n // 5 if case['scene'] == 'long' else 0))
        ch = 4.0 if case['output'] == 'sdf' else 16.0
        nbytes += params * (2 if case['train'] else 1) + w * h * ch * (2 if case['train'] else 1)
        area = float(w * h)
        if case['scene'] == 'closed':
            spread = case.get('spread', w * 60.0 / 512.0)
            hold, test = n * min(1.0, (4.0 * spread) ** 2 / area), 150.0
        elif case['scene'] == 'strokes':
            step = case.get('step', 0.2 * w)
            hold, test = n * min(1.0, (3.0 * step) ** 2 / area), 200.0
        else:
            hold, test = min(float(n), 3.0), 120.0
        if case['prefilter'] or case['output'] == 'sdf':
            test = 600.0
        sides = 1
        if case['train'] and case['output'] == 'color' and not case['prefilter']:
            sides = 3
        flops += area * spp * (60.0 + sides * hold * test)
    return {'bytes': nbytes, 'flops': flops}


def tolerance(case):
    """Images are sums of a few float32 products per pixel; gradients are float32 sums of
    up to a million terms of both signs, added in an order that is not defined: the same
    inputs twice differ by up to 1.1e-5 (one circle, every term on three addresses), by
    about 1e-6 elsewhere."""
    return {'rel': 4e-5, 'max': 4e-4}


# ------------------------------------------------------------------------- 64-bit evaluation
# The forward image (or distance field) and the gradients of constant paints, evaluated
# with dense float64 tensor operations at the sample positions the render seed defines.
_M64 = (1 << 64) - 1


def _wrap(x):
    x &= _M64
    return x - (1 << 64) if x >> 63 else x


def _pcg_pair(idx, seed):
    """The two uniform floats of the PCG32 stream of each sample index."""
    mul = _wrap(6364136223846793005)
    inc = ((idx + 1) << 1) | 1
    inc1 = inc | 1
    state = inc1 + _wrap(0x853c49e6748fea9b + seed)
    state = state * mul + inc1
    out = []
    for _ in range(2):
        old = state
        state = old * mul + inc1
        xs = ((((old >> 18) & ((1 << 46) - 1)) ^ old) >> 27) & 0xffffffff
        rot = (old >> 59) & 31
        v = ((xs >> rot) | (xs << ((32 - rot) & 31))) & 0xffffffff
        out.append((v >> 9).to(torch.float32) * (2.0 ** -23))
    return out


def _positions(case, scene, seed, centre, device):
    """Sample positions (render pixels, float32 as the path defines them) and their pixels."""
    W, H, nx, ny = scene['w'], scene['h'], case['nsx'], case['nsy']
    idx = torch.arange(W * H * nx * ny, device=device, dtype=torch.int64)
    sx, sy, x, y = idx % nx, idx // nx % ny, idx // (nx * ny) % W, idx // (nx * ny * W)
    rx, ry = _pcg_pair(idx, seed)
    if centre:
        rx, ry = torch.full_like(rx, 0.5), torch.full_like(ry, 0.5)
    px = x.to(torch.float32) + (sx.to(torch.float32) + rx) / nx
    py = y.to(torch.float32) + (sy.to(torch.float32) + ry) / ny
    return px.double(), py.double(), x, y


def _filter_weight(kind, r, dx, dy):
    inside = (dx.abs() <= r) & (dy.abs() <= r)
    if kind == 'box':
        v = torch.full_like(dx, 1.0 / (4 * r * r))
    elif kind == 'tent':
        v = (r - dx.abs()) * (r - dy.abs()) / r ** 4
    elif kind == 'parabolic':
        v = (16.0 / 9.0) * (1 - (dx / r) ** 2) * (1 - (dy / r) ** 2)
    elif kind == 'hann':
        v = 0.25 * (1 - torch.cos(2 * math.pi * (dx / (2 * r) + 0.5))) * \
            (1 - torch.cos(2 * math.pi * (dy / (2 * r) + 0.5))) / (r * r)
    else:
        s = r / 3
        v = torch.exp(-(dx * dx + dy * dy) / (2 * s * s)) / (2 * math.pi * s * s)
    return torch.where(inside, v, torch.zeros_like(v))


def _segments(s, device):
    """The path's segments as power-basis cubics [nseg, 4, 2] (constant term first)."""
    pts = torch.from_numpy(s['pts']).to(device).double()
    out, k, n = [], 0, len(s['pts'])
    for c in s['ncp']:
        ids = [(k + j) % n for j in range(int(c) + 2)]
        p = [pts[i] for i in ids]
        zero = torch.zeros_like(p[0])
        if c == 0:
            out.append(torch.stack([p[0], p[1] - p[0], zero, zero]))
        elif c == 1:
            out.append(torch.stack([p[0], 2 * (p[1] - p[0]), p[0] - 2 * p[1] + p[2], zero]))
        else:
            out.append(torch.stack([p[0], 3 * (p[1] - p[0]), 3 * (p[0] - 2 * p[1] + p[2]),
                                    p[3] - p[0] + 3 * (p[1] - p[2])]))
        k += int(c) + 1
    return torch.stack(out)


def _poly(c, t):
    return ((c[..., 3] * t + c[..., 2]) * t + c[..., 1]) * t + c[..., 0]


def _winding(segs, x, y):
    """Crossings of the ray to +x, over the pieces of each segment on which y is monotone."""
    cy, cx = segs[:, :, 1], segs[:, :, 0]
    a, b, c = 3 * cy[:, 3], 2 * cy[:, 2], cy[:, 1]
    disc = (b * b - 4 * a * c).clamp_min(0).sqrt()
    q = -0.5 * (b + torch.where(b >= 0, disc, -disc))
    roots = torch.stack([q / a, c / q], 1)
    roots = torch.where(torch.isfinite(roots), roots, torch.zeros_like(roots)).clamp(0, 1).sort(1).values
    cuts = torch.cat([torch.zeros_like(roots[:, :1]), roots, torch.ones_like(roots[:, :1])], 1)
    w = torch.zeros(x.shape, dtype=torch.int64, device=x.device)
    for k in range(3):
        lo, hi = cuts[:, k], cuts[:, k + 1]
        up_lo = _poly(cy, lo)[:, None] > y[None]
        up_hi = _poly(cy, hi)[:, None] > y[None]
        i, j = (up_lo != up_hi).nonzero(as_tuple=True)
        if i.numel() == 0:
            continue
        rising = up_hi[i, j]
        l, h, cyi, yj = lo[i], hi[i], cy[i], y[j]
        for _ in range(52):
            m = 0.5 * (l + h)
            above = (_poly(cyi, m) > yj) == rising
            l, h = torch.where(above, l, m), torch.where(above, m, h)
        hit = _poly(cx[i], 0.5 * (l + h)) > x[j]
        w.index_add_(0, j[hit], torch.where(rising[hit], 1, -1))
    return w


def _nearest(segs, x, y, cells=24):
    """Distance to the nearest point of the segments: coarse samples, then a bracketed
    search around each segment's two best cells."""
    t = torch.linspace(0, 1, cells + 1, device=x.device, dtype=torch.float64)
    gx, gy = _poly(segs[:, None, :, 0], t), _poly(segs[:, None, :, 1], t)
    best = torch.full(x.shape, math.inf, device=x.device, dtype=torch.float64)
    for s in range(segs.shape[0]):
        d = (gx[s, :, None] - x) ** 2 + (gy[s, :, None] - y) ** 2
        hop = math.sqrt(float(((gx[s, 1:] - gx[s, :-1]) ** 2 + (gy[s, 1:] - gy[s, :-1]) ** 2).max()))
        low = d.min(0).values
        near = (low.sqrt() - hop < best).nonzero().squeeze(1)
        best = torch.minimum(best, low.sqrt())
        if near.numel() == 0:
            continue
        two = d[:, near].topk(min(2, cells + 1), 0, largest=False).indices
        cx, cy, xn, yn = segs[s, :, 0], segs[s, :, 1], x[near], y[near]
        for k in range(two.shape[0]):
            l = ((two[k].double() - 1) / cells).clamp(0, 1)
            h = ((two[k].double() + 1) / cells).clamp(0, 1)
            for _ in range(40):
                m1, m2 = l + (h - l) / 3, h - (h - l) / 3
                d1 = (_poly(cx, m1) - xn) ** 2 + (_poly(cy, m1) - yn) ** 2
                d2 = (_poly(cx, m2) - xn) ** 2 + (_poly(cy, m2) - yn) ** 2
                left = d1 < d2
                l, h = torch.where(left, l, m1), torch.where(left, m2, h)
            m = 0.5 * (l + h)
            dm = ((_poly(cx, m) - xn) ** 2 + (_poly(cy, m) - yn) ** 2).sqrt()
            best[near] = torch.minimum(best[near], dm)
    return best


class _Shape64:
    """Coverage queries of one shape at points given in its own space."""

    def __init__(self, s, device):
        self.s = s
        if s['kind'] == 'path':
            self.segs = _segments(s, device)
            lo, hi = s['pts'].min(0), s['pts'].max(0)
        elif s['kind'] == 'rect':
            lo, hi = s['lo'], s['hi']
        else:
            r = s['radius'] * np.ones(2)
            lo, hi = s['centre'] - r, s['centre'] + r
        self.box = [float(v) for v in (*lo, *hi)]

    def inside(self, x, y, even_odd):
        s = self.s
        if s['kind'] == 'path':
            w = _winding(self.segs, x, y)
            return (w % 2 != 0) if even_odd else (w != 0)
        if s['kind'] == 'rect':
            return (x > float(s['lo'][0])) & (x < float(s['hi'][0])) & (y > float(s['lo'][1])) & (y < float(s['hi'][1]))
        r = s['radius'] * np.ones(2)
        return ((x - float(s['centre'][0])) / float(r[0])) ** 2 + ((y - float(s['centre'][1])) / float(r[1])) ** 2 < 1

    def distance(self, x, y):
        s = self.s
        if s['kind'] == 'path':
            return _nearest(self.segs, x, y)
        if s['kind'] == 'circle':
            return (((x - float(s['centre'][0])) ** 2 + (y - float(s['centre'][1])) ** 2).sqrt()
                    - float(s['radius'])).abs()
        (x0, y0), (x1, y1) = s['lo'].astype(float), s['hi'].astype(float)
        dx, dy = torch.maximum(x0 - x, x - x1), torch.maximum(y0 - y, y - y1)
        out = (dx.clamp_min(0) ** 2 + dy.clamp_min(0) ** 2).sqrt()
        return torch.where((dx < 0) & (dy < 0), -torch.maximum(dx, dy), out)


def _paint64(p, x, y):
    """[N, 4] colours of a paint at canvas points."""
    if p[0] == 'const':
        return torch.from_numpy(p[1]).to(x.device).double().expand(x.shape[0], 4)
    a, b, offs, cols = (torch.from_numpy(v).to(x.device).double() for v in p[1:])
    if p[0] == 'linear':
        d = b - a
        t = ((x - a[0]) * d[0] + (y - a[1]) * d[1]) / max(float((d * d).sum()), 1e-3)
    else:
        t = (((x - a[0]) / b[0]) ** 2 + ((y - a[1]) / b[1]) ** 2).sqrt()
    k = (torch.searchsorted(offs, t, right=True) - 1).clamp(0, len(offs) - 2)
    f = (t - offs[k]) / (offs[k + 1] - offs[k])
    mixed = cols[k] * (1 - f)[:, None] + cols[k + 1] * f[:, None]
    return torch.where((t < offs[0])[:, None], cols[0], torch.where((t >= offs[-1])[:, None], cols[-1], mixed))


def _smooth(d):
    t = ((d + 1) / 2).clamp(0, 1)
    return t * t * (3 - 2 * t)


def _local(g, x, y, device):
    if g['xform'] is None:
        return x, y
    m = torch.linalg.inv(torch.from_numpy(g['xform']).double()).to(device)
    return m[0, 0] * x + m[0, 1] * y + m[0, 2], m[1, 0] * x + m[1, 1] * y + m[1, 2]


def _fragments(case, scene, x, y, device):
    """In compositing order: (paint, samples it covers, coverage weights or None)."""
    for g in scene['groups']:
        sh = _Shape64(scene['shapes'][g['shape']], device)
        lx, ly = _local(g, x, y, device)
        x0, y0, x1, y1 = sh.box
        width = float(sh.s['width'])
        grow = (width + 1.001) if case['prefilter'] else (width if g['stroke'] else 0.0)
        near = ((lx >= x0 - grow) & (lx <= x1 + grow) & (ly >= y0 - grow) & (ly <= y1 + grow)).nonzero().squeeze(1)
        if near.numel() == 0:
            continue
        lx, ly = lx[near], ly[near]
        dist = sh.distance(lx, ly) if (case['prefilter'] or g['stroke']) else None
        if g['stroke']:
            if case['prefilter']:
                w = _smooth(dist + width) - _smooth(dist - width)
                on = w > 0
                yield g['stroke'], near[on], w[on]
            else:
                yield g['stroke'], near[dist < width], None
        if g['fill']:
            inn = sh.inside(lx, ly, g['even_odd'])
            if case['prefilter']:
                w = _smooth(torch.where(inn, dist, -dist))
                on = (w > 0) & (inn | (dist < 1))
                yield g['fill'], near[on], w[on]
            else:
                yield g['fill'], near[inn], None


def _exact_color(case, scene, target, bg, seed, device):
    """(image, gradients of the constant paints in parameter order or None)"""
    W, H = scene['w'], scene['h']
    px, py, ix, iy = _positions(case, scene, seed, case['prefilter'], device)
    jx, jy = (px, py) if not case['prefilter'] else _positions(case, scene, seed, False, device)[:2]
    n = px.numel()
    color, alpha = torch.zeros(n, 3, device=device, dtype=torch.float64), torch.zeros(n, device=device,
                                                                                      dtype=torch.float64)
    if bg is not None:
        b = torch.from_numpy(bg).to(device).double()[iy, ix]
        color, alpha = b[:, :3].clone(), b[:, 3].clone()
    tape = []
    for paint, at, weight in _fragments(case, scene, px, py, device):
        c = _paint64(paint, px[at], py[at])
        a = c[:, 3] if weight is None else c[:, 3] * weight
        tape.append((paint, at, weight, c[:, :3], a, color[at], alpha[at]))
        color[at] = color[at] * (1 - a)[:, None] + a[:, None] * c[:, :3]
        alpha[at] = alpha[at] * (1 - a) + a
    some = alpha > 1e-6
    rgb = torch.where(some[:, None], color / alpha.clamp_min(1e-6)[:, None], color)
    out = torch.cat([rgb, alpha[:, None]], 1)
    r = float(np.float32(case['radius']))
    ri = int(math.ceil(r))
    taps = []
    for dy in range(-ri, ri + 1):
        for dx in range(-ri, ri + 1):
            xx, yy = ix + dx, iy + dy
            ok = (xx >= 0) & (xx < W) & (yy >= 0) & (yy < H)
            taps.append((dx, dy, ok, torch.where(ok, yy * W + xx, torch.zeros_like(xx))))
    zero = torch.zeros((), device=device, dtype=torch.float64)

    def tap_weight(dx, dy, ok, sx, sy):
        return torch.where(ok, _filter_weight(case['filter'], r, ix + dx + 0.5 - sx, iy + dy + 0.5 - sy), zero)

    wsum = torch.zeros(W * H, device=device, dtype=torch.float64)
    img = torch.zeros(W * H, 4, device=device, dtype=torch.float64)
    for dx, dy, ok, at in taps:
        wsum.index_add_(0, at, tap_weight(dx, dy, ok, jx, jy))
        img.index_add_(0, at, tap_weight(dx, dy, ok, px, py)[:, None] * out)
    inv = torch.where(wsum > 0, 1 / wsum, zero)
    img = img * inv[:, None]
    if not case['train']:
        return img.view(H, W, 4), None
    d_img = 2 * (img - torch.from_numpy(target).to(device).double().view(W * H, 4)) * inv[:, None]
    d = torch.zeros(n, 4, device=device, dtype=torch.float64)
    for dx, dy, ok, at in taps:
        d += tap_weight(dx, dy, ok, px, py)[:, None] * d_img[at]
    d_rgb = torch.where(some[:, None], d[:, :3] / alpha.clamp_min(1e-6)[:, None], d[:, :3])
    d_alpha = d[:, 3] - torch.where(some, (d_rgb * rgb).sum(1), zero)
    grads = {}
    for paint, at, weight, c, a, prev, prev_a in reversed(tape):
        dc, da = d_rgb[at], d_alpha[at]
        d_a = da * (1 - prev_a) + (dc * (c - prev)).sum(1)
        if weight is not None:
            d_a = d_a * weight
        g = torch.cat([(dc * a[:, None]).sum(0), d_a.sum()[None]])
        grads[id(paint)] = grads.get(id(paint), 0) + g
        d_rgb[at], d_alpha[at] = dc * (1 - a)[:, None], da * (1 - a)
    flat = []
    for g in scene['groups']:
        for p in (g['fill'], g['stroke']):
            if p is not None:
                if p[0] != 'const':
                    return img.view(H, W, 4), None
                flat.append(grads.get(id(p), torch.zeros(4, device=device, dtype=torch.float64)))
    return img.view(H, W, 4), torch.cat(flat)


def _exact_sdf(case, scene, seed, device):
    W, H = scene['w'], scene['h']
    px, py, ix, iy = _positions(case, scene, seed, False, device)
    best = torch.full(px.shape, math.inf, device=device, dtype=torch.float64)
    sign = torch.ones_like(best)
    for g in reversed(scene['groups']):
        sh = _Shape64(scene['shapes'][g['shape']], device)
        x0, y0, x1, y1 = sh.box
        gap = (torch.maximum(x0 - px, px - x1).clamp_min(0) ** 2 + torch.maximum(y0 - py, py - y1).clamp_min(0) ** 2)
        near = (gap.sqrt() < best).nonzero().squeeze(1)
        if near.numel() == 0:
            continue
        d = sh.distance(px[near], py[near])
        on = d < best[near]
        near, d = near[on], d[on]
        best[near] = d
        sign[near] = torch.where(sh.inside(px[near], py[near], g['even_odd']), -1.0, 1.0).double() if g['fill'] else 1.0
    spp = case['nsx'] * case['nsy']
    out = torch.zeros(W * H, device=device, dtype=torch.float64)
    out.index_add_(0, iy * W + ix, best * sign / spp)
    return out.view(H, W, 1)


def exact(case, seed):
    if case['entry'] == 'generative' or case['scene'] == 'long':
        return None
    scene, target, bg, render_seed = _inputs(case, seed)
    device = torch.device('cuda:0' if torch.cuda.is_available() else 'cpu')
    if case['entry'] == 'batch':
        if sum(len(s['shapes']) for s in scene) > 1500:
            return None  # minutes of dense tensor work
        imgs, grads, at = [], [], 0
        for s in scene:
            n = s['w'] * s['h']
            img, g = _exact_color(case, s, target[at:at + n], None, render_seed, device)
            imgs.append(img.reshape(-1, 4))
            grads.append(g)
            at += n
        g = None if any(x is None for x in grads) else torch.cat(grads)
        return {'image': torch.cat(imgs), 'd_color_params': g, 'd_points': None}
    if case['output'] == 'sdf':
        res = {'image': _exact_sdf(case, scene, render_seed, device)}
        if case['train']:
            res.update(d_geometry=None, d_width=None, d_color=None)
        return res
    img, g = _exact_color(case, scene, target, bg, render_seed, device)
    if not case['train']:
        return {'image': img}
    if case['entry'] == 'resident':
        return {'image': img, 'd_points': None, 'd_stroke_width': None, 'd_color_params': g}
    return {'image': img, 'd_geometry': None, 'd_width': None, 'd_color': g}
