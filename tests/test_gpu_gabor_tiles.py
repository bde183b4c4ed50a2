"""GPU: Gabor energies as sums of two row x column filters, where blocks meet.

A block forms 27 x 64 energies; below 512 blocks it takes one filter, beyond
all eight; and where its pixels are outside [1e-24, 1e290] (or infinite) it
adds the 1,444 taps.  The counts are taken over blocks of 8,192 pixels and
certified against the reference's sums, so every ratio equals the direct
path's (WNDGPU_GABOR_DIRECT=1) exactly."""
import numpy as np
import pytest

import wndcharm
from helpers import features_in_context

pytestmark = pytest.mark.gpu


def check(imgs):
    plan = wndcharm.FeatureComputationPlan('gabor tiles')
    plan.add('Gabor Textures ()')
    plan.finalize()
    want = features_in_context({'WNDGPU_GABOR_DIRECT': '1'}, imgs, plan)
    got = features_in_context({}, imgs, plan)
    assert np.array_equal(got, want, equal_nan=True), (got, want)


def image(shape, seed):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:shape[0], 0:shape[1]]
    return 40 + 20 * np.sin(y / 3.0 + x / 17.0) + rng.normal(0, 6, shape)


@pytest.mark.parametrize('shape', [(16, 16), (26, 63), (27, 64), (28, 65), (54, 128), (55, 129), (64, 128), (127, 129), (300, 70)])
def test_block_edges(shape):
    print('gabor tiles', shape, flush=True)
    check([image(shape, 1), image(shape[::-1], 2)])


def test_all_filters_in_a_block():
    print('gabor tiles: 520 blocks', flush=True)
    check([image((27, 64), k) for k in range(500)] + [image((28, 65), k) for k in range(5)])


@pytest.mark.parametrize('scale', [1e-30, 1e-26, 1e-24, 1e-20, 1e20, 1e289])
def test_magnitudes(scale):
    print('gabor tiles: scale', scale, flush=True)
    a = image((60, 140), 3) * scale
    a[:, :70] *= 0.9  # blocks of one plane on both sides of a limit
    check([a])


@pytest.mark.parametrize('value', [np.inf, -np.inf, 0.0])
def test_blocks_with_an_odd_value(value):
    """in one block's window only; a plane of zeros"""
    print('gabor tiles:', value, flush=True)
    a = image((90, 200), 4)
    a[40, 100] = value
    check([a, np.zeros((32, 32))])
