"""GPU: the Schur kernels behind Haralick f14 at the sizes where their windows,
bands and launch rules have edges, bit for bit against the oracle.

The small-launch kernel chases a bulge in windows of 16 steps, keeps a band of
64 columns in a wave and updates rows above a window 64 at a time, so matrix
orders around multiples of 16 and 64 (order = number of gray tones) exercise
its remainders; the Hessenberg reduction keeps more columns in LDS from 171 and
129 tones down and updates the rows above 32 at a time; order 256 is the largest, and orders below 3 have no f14.
Launches of up to 256 matrices, up to 6144 and beyond take different kernels,
and from 1025 to 6144 the tones decide between two of them."""
import numpy as np
import pytest

import wndcharm
from helpers import ALG_NAMES, features_in_context, orc_algorithm

pytestmark = pytest.mark.gpu

F14 = [16, 17]  # mean and range over the four angles


def toned(ng, seed, shape=(40, 56)):
    """an image whose quantised plane has exactly ng tones (0 and 255 among them)"""
    rng = np.random.default_rng(1000 * ng + seed)
    if ng == 1:
        return np.full(shape, 7.0)
    tones = np.concatenate([[0, 255], rng.permutation(np.arange(1, 255))[:ng - 2]]).astype(np.float64)
    y, x = np.mgrid[0:shape[0], 0:shape[1]]
    # smooth structure plus noise over the sorted tones, every tone at least once
    u = (0.5 + 0.3 * np.sin(x / 5.0 + seed) * np.cos(y / 7.0) + 0.2 * rng.uniform(-1, 1, shape)).clip(0, 0.999)
    idx = (u * ng).astype(int)
    idx.reshape(-1)[rng.permutation(idx.size)[:ng]] = np.arange(ng)
    return np.sort(tones)[idx]


@pytest.mark.parametrize('ng', [1, 2, 3, 4, 5, 17, 18, 19, 20, 31, 32, 33, 34, 35, 63, 64, 65, 66, 80, 81, 82, 83, 98, 99, 127, 128, 129,
                                130, 162, 163, 171, 172, 194, 195, 255, 256])
def test_schur_orders_equal_oracle(ng):
    img = toned(ng, 3, (64, 72) if ng > 128 else (40, 56))
    print('schur order', ng, flush=True)
    got = np.asarray(wndcharm.FeatureAlgorithm('Haralick Textures').execute(img))
    assert wndcharm.last_haralick_work()[0][0] == ng
    want = orc_algorithm(ALG_NAMES.index('Haralick Textures'), img)
    assert np.array_equal(got[F14], want[F14], equal_nan=True), (got[F14], want[F14])


def test_schur_low_rank_and_binary_planes_equal_oracle():
    """matrices with zero rows, exact zeros below the diagonal and repeated
    eigenvalues: deflations of one and two roots, reflectors of zero vectors"""
    y, x = np.mgrid[0:48, 0:48]
    planes = [((x // 8) % 2) * 255.0, (x % 5) * 51.0, ((x * y) % 17).astype(float), np.where(x == y, 255.0, x % 3),
              (x // 3).astype(float)]
    for k, img in enumerate(planes):
        print('schur structured', k, flush=True)
        got = np.asarray(wndcharm.FeatureAlgorithm('Haralick Textures').execute(img))
        want = orc_algorithm(ALG_NAMES.index('Haralick Textures'), img)
        assert np.array_equal(got[F14], want[F14], equal_nan=True), (k, got[F14], want[F14])


def test_schur_launch_rules_agree():
    """the same images in launches of 4 x 1, 4 x 100 and 4 x 1600 matrices (eight
    waves, four waves and one wave per matrix) give the same bits"""
    kinds = [toned(int(ng), s, (24, 32)) for s, ng in enumerate(np.linspace(3, 200, 100))]
    plan = wndcharm.FeatureComputationPlan('haralick')
    plan.add('Haralick Textures ()')
    plan.finalize()
    print('schur 1600 / 100 / 1', flush=True)
    many = wndcharm.compute_features(kinds * 16, plan)
    some = wndcharm.compute_features(kinds, plan)
    one = np.concatenate([wndcharm.compute_features([im], plan) for im in kinds[::9]])
    assert np.array_equal(many, np.concatenate([some] * 16), equal_nan=True)
    assert np.array_equal(one, some[::9], equal_nan=True)


@pytest.mark.parametrize('n', [256, 257, 700])
@pytest.mark.parametrize('kind', ['few', 'spread', 'one'])
def test_kernel_picked_by_tones(kind, n):
    """256 entries take four waves per matrix; beyond, entries of few tones take
    one wave per matrix, and many tones among few ones four; whichever it is,
    every entry has the bits that it has on its own"""
    tones = {'few': [12] * 9, 'spread': range(5, 200, 22), 'one': [250] + [9] * 8}[kind]
    kinds = [toned(ng, k, (24, 32)) for k, ng in enumerate(tones)]
    plan = wndcharm.FeatureComputationPlan('haralick')
    plan.add('Haralick Textures ()')
    plan.finalize()
    print('schur picked', kind, n, flush=True)
    got = wndcharm.compute_features([kinds[k % 9] for k in range(n)], plan)
    work = wndcharm.last_haralick_work()[1]
    one = np.concatenate([wndcharm.compute_features([im], plan) for im in kinds])
    assert np.array_equal(got, one[np.arange(n) % 9], equal_nan=True)
    assert np.array_equal(work, work[np.arange(n) % 9]) and (work > 0).all()


@pytest.mark.parametrize('n', [1, 100, 300])
def test_a_wait_in_vain_fails_the_call(n):
    """no polls: a wave that does not find the reflectors at once gives up, the
    kernel ends, and the call fails instead of returning what a stale reflector
    gave; another context is not affected"""
    imgs = [toned(150, k, (40, 56)) for k in range(3)]
    plan = wndcharm.FeatureComputationPlan('haralick')
    plan.add('Haralick Textures ()')
    plan.finalize()
    print('schur without polls', n, flush=True)
    want = wndcharm.compute_features(imgs, plan)
    with pytest.raises(wndcharm.WndGpuError):
        features_in_context({'WNDGPU_SCHUR_NO_POLLS': '1'}, [imgs[k % 3] for k in range(n)], plan)
    assert np.array_equal(wndcharm.compute_features(imgs, plan), want, equal_nan=True)
