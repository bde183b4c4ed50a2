"""GPU: Tamura textures where the summed-area table's strips and the pixel runs meet.

The table is formed in strips of 64 rows, eight at once, in groups of 16
columns; pixels are taken in runs of 64 columns x 8 rows (2 rows in planes of up
to 4,096 pixels) and their histograms in blocks of 16,384, planes of one block by
one launch.  Planes just below, at and above these sizes against the
oracle.  Best scales and phi go through histograms, whose counts are whole
numbers: a wrong table entry moves a count, i.e. a result by more than 1 / P.
The rest are sums of P terms in another order, P * 2^-53 < 1e-9 apart."""
import numpy as np
import pytest

import wndcharm
from helpers import ALG_NAMES, orc_algorithm

pytestmark = pytest.mark.gpu
ALG = 'Tamura Textures'
COARSENESS = [0, 1, 2, 5]


def check(img):
    got = np.asarray(wndcharm.FeatureAlgorithm(ALG).execute(img))
    want = orc_algorithm(ALG_NAMES.index(ALG), np.asarray(img, np.float64))
    assert np.allclose(got, want, rtol=1e-9, atol=1e-12, equal_nan=True), (img.shape, got, want)


# one strip and less, runs and groups cut short, eight strips, a wave's second
# strip where it follows after 41 groups (narrow) and after all groups (wide)
@pytest.mark.parametrize('shape', [(16, 16), (16, 64), (16, 256), (16, 257), (256, 16), (17, 65), (63, 17), (31, 129), (64, 64), (65, 63), (64, 256), (129, 128), (128, 129),
                                   (511, 40), (512, 17), (513, 33), (577, 593), (576, 594), (1100, 61), (1030, 700)])
def test_strips_and_runs(shape):
    print('tamura', shape, flush=True)
    rng = np.random.default_rng(sum(shape))
    y, x = np.mgrid[0:shape[0], 0:shape[1]]
    check(np.round(900 + 300 * np.sin(x / 5.0 + y / 11.0)) + rng.integers(0, 400, shape))


@pytest.mark.parametrize('kind', ['flat', 'step', 'negative', 'tiny', 'float32'])
def test_values(kind):
    """all equal; two values; a negative maximum; differences near the smallest double; 24-bit values"""
    print('tamura', kind, flush=True)
    rng = np.random.default_rng(5)
    noise = rng.normal(0, 1, (70, 150))
    img = {'flat': np.full((70, 150), 7.0), 'step': np.where(np.arange(150) < 70, 10.0, 200.0) * np.ones((70, 1)),
           'negative': noise - 50, 'tiny': 1.0 + np.round(noise) * 2.0 ** -52,
           'float32': noise.astype(np.float32).astype(np.float64) + 9}[kind]
    check(img)


@pytest.mark.parametrize('exponent', [-1074, -1073, -1070, -1060, -1022, -1015])
def test_window_means_of_subnormal_sums(exponent):
    """pixels of a few units near the smallest double: subnormal means, where a
    quotient can lie halfway between two doubles.  The largest pixel is 1, so
    that normalisation keeps the values, and the last, so that the sums before
    it stay small."""
    print('tamura subnormal 2 **', exponent, flush=True)
    rng = np.random.default_rng(-exponent)
    img = np.ldexp(rng.integers(0, 40, (70, 150)).astype(np.float64), exponent)
    img[-1, -1] = 1.0
    check(img)


def test_planes_of_all_kinds_in_one_call():
    """each plane's features are those that it has on its own, bit for bit"""
    rng = np.random.default_rng(11)
    shapes = [(16, 16), (64, 64), (64, 65), (17, 65), (256, 16), (128, 128), (129, 128), (31, 130), (600, 40), (300, 301)]
    imgs = [rng.integers(0, 4000, s).astype(np.uint16) for s in shapes]
    plan = wndcharm.FeatureComputationPlan('tamura')
    plan.add('Tamura Textures ()')
    plan.finalize()
    print('tamura', shapes, flush=True)
    one = np.concatenate([wndcharm.compute_features([im], plan) for im in imgs])
    assert np.array_equal(wndcharm.compute_features(imgs, plan), one, equal_nan=True)
    assert np.array_equal(wndcharm.compute_features(imgs[:5], plan), one[:5], equal_nan=True)


@pytest.mark.parametrize('value', [np.nan, np.inf, -np.inf, 1e39])
def test_odd_pixels(value):
    """One odd pixel poisons the table's entries right of and below it, and every
    window mean from them; 1e39 is finite but beyond what the statistics count.
    Compared are the coarseness and its histogram: contrast and direction add up
    the odd pixels themselves, which the oracle leaves out."""
    print('tamura', value, flush=True)
    rng = np.random.default_rng(8)
    for at in ((0, 0), (40, 80), (129, 149), (100, 3), (64, 0)):
        img = np.round(rng.normal(100, 30, (130, 150)))
        img[at] = value
        got = np.asarray(wndcharm.FeatureAlgorithm(ALG).execute(img))
        want = orc_algorithm(ALG_NAMES.index(ALG), img)
        assert np.allclose(got[COARSENESS], want[COARSENESS], rtol=1e-9, atol=1e-12, equal_nan=True), (at, got, want)
