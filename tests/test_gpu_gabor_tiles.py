"""GPU: Gabor energies as sums of two row x column filters, where blocks meet.

A block forms 27 x 64 energies; below 512 blocks it takes one filter, beyond
all eight; and where its largest pixel is outside [1e-24, 1e290] (or infinite) it
adds the 1,444 taps in the direct path's order.  The counts are taken over blocks of 8,192 pixels and
certified against the reference's sums, so every ratio equals the direct
path's (WNDGPU_GABOR_DIRECT=1) exactly."""
import numpy as np
import pytest

import wndcharm
from helpers import features_in_context

pytestmark = pytest.mark.gpu


def check(imgs, finite=False):
    plan = wndcharm.FeatureComputationPlan('gabor tiles')
    plan.add('Gabor Textures ()')
    plan.finalize()
    want = features_in_context({'WNDGPU_GABOR_DIRECT': '1'}, imgs, plan)
    got = features_in_context({}, imgs, plan)
    assert np.array_equal(got, want, equal_nan=True), (got, want)
    assert not finite or np.isfinite(got).all(), got


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


def near_ties(seed, scale):
    """planes of two equal patches, the second times 0.4 (1 + k / 2^52): its
    low-pass energies lie a few units in the last place from the level 0.4 of the
    first's, so that the base count hangs on how the sums round"""
    patch = np.random.default_rng(seed).uniform(50, 100, (38, 38))
    out = []
    for k in range(-12, 13):
        a = np.zeros((60, 160))
        a[11:49, 20:58] = patch
        a[11:49, 100:138] = patch * (0.4 * (1 + k * 2.0 ** -52))
        out.append(a * scale)
    return out


@pytest.mark.parametrize('scale', [2.0 ** -200, 2.0 ** -130, 2.0 ** -120, 2.0 ** -100, 2.0 ** -78, 1.0, 2.0 ** 130])
def test_energies_next_to_a_level(scale):
    """2^-120: pixels around 1e-34, where a bound is less than any float"""
    print('gabor tiles: near ties, scale', scale, flush=True)
    check([im for seed in range(6) for im in near_ties(seed, scale)], finite=True)


@pytest.mark.parametrize('small', [1e-26, 1e-30, 1e-38, 1e-60])
def test_blocks_of_small_pixels_beside_others(small):
    """whole windows below the limit in planes whose other blocks lie above it"""
    print('gabor tiles: blocks scaled by', small, flush=True)
    a, b = image((190, 340), 4), image((190, 340), 6)
    a[:, :150] *= small
    b[:100] *= small
    check([a, b, a * 1e-20, b * 1e-20], finite=True)


@pytest.mark.parametrize('value', [np.inf, -np.inf, 0.0])
def test_blocks_with_an_odd_value(value):
    """in one block's window only; a plane of zeros.  An infinite maximum leaves no
    base count, so the ratios are NaN on both paths: the energies of such blocks are
    compared by test_energies_next_to_a_level, which takes the same branch."""
    print('gabor tiles:', value, flush=True)
    a = image((90, 200), 4)
    a[40, 100] = value
    check([a, np.zeros((32, 32))])
