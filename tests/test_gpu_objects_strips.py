"""GPU: object features and edge medians where their blocks of pixels meet.

Connected components are labelled in strips of up to 16,384 pixels and joined
across the strips' first rows; roots are ranked and areas added in blocks of
4,096 pixels; medians are selected from the bins that hold the middle ranks.
Planes just below, at and above these sizes, with components that wind through
many strips, against the oracle: counts exactly, the rest to 1e-9."""
import numpy as np
import pytest

import wndcharm
from helpers import ALG_NAMES, orc_algorithm

pytestmark = pytest.mark.gpu

OBJ_EXACT = list(range(0, 14)) + [15, 16, 17] + list(range(18, 29)) + [30, 31, 33]
EDGE_EXACT = list(range(14)) + list(range(17, 25)) + [26]  # not the direction's mean, median and variance (atan2)


def check(alg, img, exact):
    got = np.asarray(wndcharm.FeatureAlgorithm(alg).execute(img))
    want = orc_algorithm(ALG_NAMES.index(alg), np.asarray(img, np.float64))
    assert np.array_equal(got[exact], want[exact]), (alg, img.shape, got, want)
    assert np.allclose(got, want, rtol=1e-9, atol=1e-9), (alg, img.shape, got, want)


def winding(h, w, seed):
    """bands that meander down the plane, combs that join them, and specks"""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    a = (np.sin(x / 3.0 + 2 * np.sin(y / 9.0)) > 0.3) | ((x + y) % 23 == 0) | ((x - y) % 31 == 0)
    a = a ^ (rng.random((h, w)) < 0.02)
    return np.where(a, 200.0, 40.0) + rng.integers(0, 9, (h, w))


@pytest.mark.parametrize('shape', [(16, 16), (64, 64), (64, 63), (65, 64), (16, 1024), (17, 1024), (128, 128), (127, 129),
                                   (129, 128), (33, 4096), (4096, 17), (300, 301)])
def test_objects_across_strips(shape):
    print('objects', shape, flush=True)
    for alg in ('Otsu Object Features', 'Inverse-Otsu Object Features'):
        check(alg, winding(*shape, seed=sum(shape)), OBJ_EXACT)


def test_objects_one_component_through_every_strip():
    """a serpentine one pixel wide, its two halves joined only in the last row"""
    img = np.zeros((260, 200))
    img[:, 3] = img[:, 190] = 100.0
    img[259, 3:191] = 100.0
    img[::4, 10:180] = 100.0
    img[2::8, 100] = 100.0
    print('objects serpentine', flush=True)
    check('Otsu Object Features', img, OBJ_EXACT)
    check('Inverse-Otsu Object Features', img, OBJ_EXACT)


@pytest.mark.parametrize('shape', [(16, 17), (64, 128), (91, 90), (91, 91), (64, 129), (256, 257)])
@pytest.mark.parametrize('kind', ['noise', 'flat', 'two', 'ramp', 'skewed'])
def test_edge_medians(shape, kind):
    """even and odd pixel counts; all values equal; two values whose middle
    ranks straddle a gap; a plane whose values crowd one bin"""
    h, w = shape
    rng = np.random.default_rng(h * w)
    img = {'noise': rng.integers(0, 4096, shape).astype(float), 'flat': np.full(shape, 5.0),
           'two': np.where(np.mgrid[0:h, 0:w][0] < h // 2, 1.0, 7.0),
           'ramp': np.mgrid[0:h, 0:w][1] * 3.0, 'skewed': np.exp(rng.normal(0, 6, shape))}[kind]
    print('edge', shape, kind, flush=True)
    check('Edge Features', img, EDGE_EXACT)


def test_more_planes_than_a_grid_dimension_holds():
    """33,000 images: 66,000 edge planes, and 66,000 object planes over two
    nodes, in one call (a grid has up to 65,536 blocks in y); every row equal to
    its image's in a call of 40"""
    plan = wndcharm.FeatureComputationPlan('many planes')
    for group in ('Edge Features ()', 'Otsu Object Features ()', 'Otsu Object Features (Edge ())',
                  'Inverse-Otsu Object Features ()'):
        plan.add(group)
    plan.finalize()
    imgs = [winding(16, 16 + k % 3, seed=k).astype(np.uint8) for k in range(40)]
    some = wndcharm.compute_features(imgs, plan)
    print('objects and edges: 33,000 images', flush=True)
    many = wndcharm.compute_features(imgs * 825, plan)
    assert np.array_equal(many, np.tile(some, (825, 1)), equal_nan=True)


ODD = {'nan': [np.nan], '+inf': [np.inf], '-inf': [-np.inf], 'all': [np.nan, np.inf, -np.inf]}


def odd_pixels(img, kind, seed):
    """the plane with seven pixels of each odd value"""
    rng = np.random.default_rng(seed)
    img = np.array(img, np.float64)
    for value in ODD[kind]:
        img.reshape(-1)[rng.permutation(img.size)[:7]] = value
    return img


@pytest.mark.parametrize('kind', list(ODD))
@pytest.mark.parametrize('shape', [(64, 70), (131, 130)])
def test_objects_with_odd_pixels(shape, kind):
    """The range is that of the finite pixels, infinities count in the outermost
    bins and lie on their side of the threshold, as the finite extremes do that
    the oracle gets in their place (its histogram converts them to integers, which
    C leaves undefined); NaN is in no mask."""
    print('objects', shape, kind, flush=True)
    img = odd_pixels(winding(*shape, seed=1), kind, 2)
    finite = img[np.isfinite(img)]
    oracle_img = np.where(img == np.inf, finite.max(), np.where(img == -np.inf, finite.min(), img))
    for alg in ('Otsu Object Features', 'Inverse-Otsu Object Features'):
        got = np.asarray(wndcharm.FeatureAlgorithm(alg).execute(img))
        want = orc_algorithm(ALG_NAMES.index(alg), oracle_img)
        assert np.array_equal(got[OBJ_EXACT], want[OBJ_EXACT]), (alg, got, want)
        assert np.allclose(got, want, rtol=1e-9, atol=1e-9), (alg, got, want)


def prewitt(a):
    """the gradient's magnitude; sums of whole numbers, so in any order"""
    p = np.pad(a, 1)
    with np.errstate(invalid='ignore'):
        sx = sum(p[j:j + a.shape[0], :-2] - p[j:j + a.shape[0], 2:] for j in range(3))
        sy = sum(p[:-2, k:k + a.shape[1]] - p[2:, k:k + a.shape[1]] for k in range(3))
        return np.sqrt(sx * sx + sy * sy)


@pytest.mark.parametrize('kind', list(ODD))
@pytest.mark.parametrize('shape', [(64, 70), (63, 71), (131, 130), (131, 131)])
@pytest.mark.parametrize('crowded', [False, True])
def test_edge_medians_with_odd_pixels(shape, kind, crowded):
    """the magnitude's median with infinite and NaN magnitudes among the sorted
    values: each NaN at the one end or the other by its sign, which depends on
    whether its pixel was added or subtracted and on the machine, so any number of
    them below the rest; crowded: most magnitudes are 0 and so in one bin"""
    print('edge', shape, kind, crowded, flush=True)
    rng = np.random.default_rng(sum(shape))
    img = np.full(shape, 50.0) if crowded else np.round(rng.normal(100, 30, shape))
    img = odd_pixels(img, kind, 3)
    m = np.sort(prewitt(img).reshape(-1))  # NaN last
    nans = int(np.isnan(m).sum())
    got = np.asarray(wndcharm.FeatureAlgorithm('Edge Features').execute(img))[26]
    want = [(v[(m.size - 1) // 2] + v[m.size // 2]) / 2 for v in (np.roll(m, k) for k in range(nans + 1))]
    assert got in want, (got, want)
