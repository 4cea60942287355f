"""Host side of the kernel staging: descriptors packed at once hold what their fields say, and a batch's
mappings are those of leniax's loop (leniax/kernels.py:91-111)."""
import math

import numpy as np
import pytest

from leniax_amd import _lib, kernels


@pytest.mark.parametrize('slug', sorted(_lib.KERNEL_SHAPES))
@pytest.mark.parametrize('rings', [[1.0], [0.5, 1, 0.25], (1, 2), np.array([0.5, 0.75], np.float32), 0.5,
                                   [0.125] * _lib.LX_MAX_RINGS])
@pytest.mark.parametrize('kf_params', [[], [4], [0.5, 0.25], np.array([1., 2., 3.]), 2.])
def test_packed_descriptor_fields(slug, rings, kf_params):
    p = {'k_slug': slug, 'k_params': [0.75, rings, 0.5, 0.25, 1.5], 'kf_slug': 'gauss', 'kf_params': kf_params}
    d = kernels.kernel_desc(p, 13.)
    bs = np.asarray(rings, np.float64).reshape(-1)
    kf = np.asarray(kf_params, np.float64).reshape(-1)[:2]
    assert (d.shape, d.kf, d.nb, d.kr) == (_lib.KERNEL_SHAPES[slug], _lib.KERNEL_FNS['gauss'], len(bs),
                                           math.ceil(0.75 * 13.))
    assert (d.a, d.b, d.theta) == ((0., 0., 0.) if slug == 'circle_2d' else (0.5, 0.25, 1.5)) and d.r == 0.75
    assert list(d.bs) == list(bs) + [0.] * (_lib.LX_MAX_RINGS - len(bs))
    assert list(d.kf_params) == list(kf) + [0.] * (2 - len(kf))


def test_mappings_of_a_batch():
    cfgs = [[{'k_params': [1., [c]], 'kf_slug': f'f{c}{k}', 'gf_slug': 'gaussian', 'gf_params': [c, k], 'h': c + k / 8,
              'c_in': (0, 0, 0, 2)[k], 'c_out': (c + k) % 3} for k in range(4)] for c in range(3)]
    for kps, m in zip(cfgs, kernels._mappings_of(cfgs, 3)):
        want = kernels.KernelMapping(3, 4)
        for i, p in enumerate(kps):
            for field, key in (('cin_k_params', 'k_params'), ('cin_kfs', 'kf_slug'), ('cin_gfs', 'gf_slug'),
                               ('cin_gf_params', 'gf_params')):
                getattr(want, field)[p['c_in']].append(p[key])
            want.cin_kernels[p['c_in']].append(i)
            want.kernels_weight_per_channel[p['c_out']][i] = p['h']
        want.true_channels = [True] * 3 + [False] * 3 + [True, False, False]
        assert m == want


@pytest.mark.parametrize('r', [2.0 ** 29, 2.0 ** 40, 1e300])
def test_a_radius_past_32_bits_is_a_value_error(r):
    """As every other radius that does not fit its world (the C field has 32 bits)."""
    p = {'k_slug': 'circle_2d', 'k_params': [r, [1.0]], 'kf_slug': 'gauss', 'kf_params': [4.]}
    with pytest.raises(ValueError, match='radius'):
        kernels.kernel_desc(p, 13.)
