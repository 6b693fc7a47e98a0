"""Strokes and distance fields of cubics whose closest points hang on the last bits of the
reference's arithmetic (dvg_quintic.h) -- quadratics written as cubics, handles on the segment's
ends -- against the CPU oracle: shared tests of a wave, per-lane tests (two shapes in a group) and
the closest point."""
import numpy as np
import pytest
import torch

import diffvg_amd as pd
from gpudrive import GpuRunner
from refdrive import OracleRunner, flatten
from test_oracle_pins import _rel

pytestmark = pytest.mark.gpu


def _scene(kind, per_group, size=160, n=120):
    r = np.random.default_rng(8)
    shapes = []
    for _ in range(n):
        q = np.float32(r.uniform(0, size, 2) + np.cumsum(r.normal(0, 12, (3, 2)), 0))
        if kind == 'quadratics':
            third = np.float32(3)
            pts = np.stack([q[0], (q[0] + 2 * q[1]) / third, (q[2] + 2 * q[1]) / third, q[2]])
        else:  # handles on the ends
            pts = q[np.array([[0, 1, 1, 1], [0, 1, 0, 1], [0, 1, 1, 0], [0, 0, 0, 1]][r.integers(0, 4)])]
        shapes.append(pd.Path(num_control_points=torch.tensor([2], dtype=torch.int32), points=torch.from_numpy(pts),
                              is_closed=False, stroke_width=torch.tensor(np.float32(r.uniform(1, 4)))))
    groups = [pd.ShapeGroup(shape_ids=torch.arange(i, i + per_group), fill_color=None,
                            stroke_color=torch.from_numpy(np.float32(np.r_[r.uniform(0, 1, 3), r.uniform(0.3, 0.9)])))
              for i in range(0, n, per_group)]
    return flatten(size, size, shapes, groups, 0, 0.5)


@pytest.mark.parametrize('kind', ['quadratics', 'ends'])
@pytest.mark.parametrize('per_group', [1, 2])
def test_strokes(per_group, kind):
    print('cubics whose roots hang on rounding, strokes', per_group, kind, flush=True)
    f = _scene(kind, per_group)
    a = GpuRunner(f).render(160, 160, 4, 4, 5)['image']
    b = OracleRunner(f).render(160, 160, 4, 4, 5)['image']
    assert np.abs(a - b).max() <= 1e-5


@pytest.mark.parametrize('kind', ['quadratics', 'ends'])
def test_distance_field(kind):
    print('cubics whose roots hang on rounding, distance', kind, flush=True)
    f = _scene(kind, 1)
    o, g = OracleRunner(f), GpuRunner(f)
    a, b = g.render(160, 160, 2, 2, 5, output='sdf')['sdf'], o.render(160, 160, 2, 2, 5, output='sdf')['sdf']
    assert np.abs(a - b).max() <= 1e-5
    d = np.random.default_rng(5).uniform(-1, 1, (160, 160, 1)).astype(np.float32)
    a, b = g.render(160, 160, 2, 2, 5, output='sdf', d_sdf=d), o.render(160, 160, 2, 2, 5, output='sdf', d_sdf=d)
    assert _rel(a['grads']['points'], b['grads']['points']) <= 1e-3
