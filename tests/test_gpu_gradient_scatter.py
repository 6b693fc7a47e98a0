"""Gradient scatter of the tiled kernels against the CPU oracle, where lanes of a wave share
destinations: gradient paints whose samples fall before, between and past the stops, stops
in any order (a value may then lie in several intervals), one to five stops, fills and
strokes of one shape over many samples.  Bars as in test_gpu_parity."""
import numpy as np
import pytest
import torch

import diffvg_amd as pd
from gpudrive import GpuRunner
from refdrive import OracleRunner, flatten
from test_oracle_pins import GRAD_KEYS, _rel

pytestmark = pytest.mark.gpu


def _gradient(kind, offsets, size):
    offs = torch.tensor(offsets)
    cols = torch.from_numpy(np.random.default_rng(len(offsets)).uniform(0.1, 0.9, (len(offsets), 4)).astype(np.float32))
    if kind == 'linear':
        return pd.LinearGradient(begin=torch.tensor([0.2 * size, 0.3 * size]),
                                 end=torch.tensor([0.8 * size, 0.6 * size]), offsets=offs, stop_colors=cols)
    return pd.RadialGradient(center=torch.tensor([0.5 * size, 0.45 * size]),
                             radius=torch.tensor([0.4 * size, 0.3 * size]), offsets=offs, stop_colors=cols)


def _check(shapes, groups, w, h, nsx, nsy, pre):
    f = flatten(w, h, shapes, groups, 0, 0.5)
    d = np.random.default_rng(2).uniform(-1, 1, (h, w, 4)).astype(np.float32)
    o, g = OracleRunner(f), GpuRunner(f)
    g.render(w, h, nsx, nsy, 3, prefilter=pre)
    a = g.render(w, h, nsx, nsy, 3, prefilter=pre, d_image=d, translation=True)
    b = o.render(w, h, nsx, nsy, 3, prefilter=pre, d_image=d, translation=True)
    for k in GRAD_KEYS:
        assert _rel(a['grads'][k], b['grads'][k]) <= 1e-3, k
    assert _rel(a['d_translation'], b['d_translation']) <= 1e-3


@pytest.mark.parametrize('pre', [False, True])
@pytest.mark.parametrize('kind', ['linear', 'radial'])
@pytest.mark.parametrize('offsets', [[0.5], [0.0, 1.0], [0.3, 0.6, 0.7], [0.1, 0.8, 0.4, 0.9, 0.2]])
def test_gradient_paints(kind, offsets, pre):
    print('gradient paint', kind, offsets, pre, flush=True)
    size = 40
    sq = torch.tensor([[2.0, 3.0], [37.0, 2.0], [38.0, 36.0], [3.0, 38.0]])
    tri = torch.tensor([[20.0, 1.0], [39.0, 30.0], [1.0, 25.0]])
    shapes = [pd.Path(num_control_points=torch.zeros(4, dtype=torch.int32), points=sq, is_closed=True,
                      stroke_width=torch.tensor(2.5)),
              pd.Path(num_control_points=torch.zeros(3, dtype=torch.int32), points=tri, is_closed=True,
                      stroke_width=torch.tensor(1.5))]
    p = _gradient(kind, offsets, size)
    groups = [pd.ShapeGroup(shape_ids=torch.tensor([0]), fill_color=p, stroke_color=torch.tensor([0.1, 0.9, 0.3, 0.7])),
              pd.ShapeGroup(shape_ids=torch.tensor([1]), fill_color=torch.tensor([0.8, 0.3, 0.2, 0.5]),
                            stroke_color=_gradient('radial' if kind == 'linear' else 'linear', offsets, size))]
    _check(shapes, groups, size, size, 2, 2, pre)


@pytest.mark.parametrize('w,h,nsx,nsy', [(16, 16, 2, 2), (33, 17, 3, 1), (96, 65, 2, 2), (7, 5, 4, 4)])
def test_one_shape_many_samples(w, h, nsx, nsy):
    print('one shape', w, h, nsx, nsy, flush=True)
    r = np.random.default_rng(w)
    pts = torch.from_numpy((r.uniform(0.1, 0.9, (6, 2)) * [w, h]).astype(np.float32))
    path = pd.Path(num_control_points=torch.tensor([2, 2]), points=pts, is_closed=True, stroke_width=torch.tensor(0.8))
    group = pd.ShapeGroup(shape_ids=torch.tensor([0]), fill_color=torch.tensor([0.3, 0.6, 0.3, 0.7]),
                          stroke_color=torch.tensor([0.9, 0.2, 0.1, 0.8]))
    for pre in (False, True):
        _check([path], [group], w, h, nsx, nsy, pre)


@pytest.mark.parametrize('h', [196592, 196608, 196624])
def test_boundary_samples_of_canvases_around_the_count_table(h):
    """Boundary samples are counted per tile in LDS up to 12288 tiles, one by one above."""
    print('tall canvas', h, flush=True)
    pts = torch.tensor([[0.2, 0.01 * h], [1.8, 0.45 * h], [0.5, 0.97 * h]])
    path = pd.Path(num_control_points=torch.tensor([0, 0, 0]), points=pts, is_closed=True, stroke_width=torch.tensor(0.1))
    group = pd.ShapeGroup(shape_ids=torch.tensor([0]), fill_color=torch.tensor([0.3, 0.6, 0.3, 0.7]),
                          stroke_color=torch.tensor([0.9, 0.2, 0.1, 0.8]))
    _check([path], [group], 2, h, 1, 1, False)


@pytest.mark.parametrize('h, direct', [(96, False), (97, True)])
def test_primitives_on_both_sides_of_the_direct_line(h, direct):
    """Boundary adjoints of primitives are combined up to 12,288 samples per shape, added one by
    one past it: 3 shapes, 4 samples a pixel, 96 x 96 (the line) and 96 x 97."""
    print('primitives at the line', h, flush=True)
    shapes = [pd.Circle(radius=torch.tensor(20.0), center=torch.tensor([30.0, 34.0]), stroke_width=torch.tensor(2.0)),
              pd.Ellipse(radius=torch.tensor([24.0, 12.0]), center=torch.tensor([60.0, 60.0])),
              pd.Rect(p_min=torch.tensor([40.0, 10.0]), p_max=torch.tensor([80.0, 44.0]),
                      stroke_width=torch.tensor(1.5))]
    groups = [pd.ShapeGroup(shape_ids=torch.tensor([i]), fill_color=torch.tensor([0.2 + 0.3 * i, 0.7, 0.4, 0.6]),
                            stroke_color=None if i == 1 else torch.tensor([0.1, 0.2, 0.9, 0.8])) for i in range(3)]
    f = flatten(96, h, shapes, groups, 0, 0.5)
    assert GpuRunner(f).scene.samples_per_wave_matters(96, h, 2, 2) == direct
    _check(shapes, groups, 96, h, 2, 2, False)
