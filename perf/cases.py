"""The calls a user of this framework makes, for timing: feature vectors of one
image and of batches over the standard sets and sample types, sampling, the
reduced-precision contractions, a transform on its own, gradients, and the
classifier.  Sizes follow the configurations of wndcharm/synthetic.py, the
reference's own test images (301x300, 1388x1040 and its 6x5 tiling) and the
limits of the API; pixels follow the synthetic generator (gratings, blobs,
Poisson noise)."""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath('wnd-charm_amd'))  # imported with the repository's root as working folder
import wndcharm  # noqa: E402

SETS = {'short': 0, 'long': 1, 'short_color': 2, 'long_color': 3}
# the four contraction families that a plan's precision applies to
CONTRACTIONS = ('Chebyshev Coefficients ()', 'Zernike Coefficients ()', 'Chebyshev-Fourier Coefficients ()',
                'Gabor Textures ()')
# groups of the untransformed image that exact() computes: compared on their own
ROOT = ('Pixel Intensity Statistics ()', 'Gini Coefficient ()', 'Multiscale Histograms ()', 'Fractal Features ()',
        'Zernike Coefficients ()')
# the differentiable groups of the gradient configuration
GRADIENT = ('Zernike Coefficients ()', 'Zernike Coefficients (Fourier ())', 'Zernike Coefficients (Chebyshev ())',
            'Chebyshev Coefficients (raw) ()', 'Chebyshev-Fourier Coefficients (raw) ()', 'Comb Moments (raw) ()',
            'Gabor Textures (raw) ()')


def listed():
    return [
        # one transform of one plane: the smallest call, all launches and copies
        dict(name='fourier_301x300', kind='transform', h=300, w=301),
        # the reference's granularity, FeatureComputationPlanExecutor::run on one image
        dict(name='one_short_128', kind='features', set='short', n=1, h=128, w=128, dtype='u16'),
        dict(name='one_long_256', kind='features', set='long', n=1, h=256, w=256, dtype='u16'),
        # the headline configuration: the long set over 400 images of one size
        dict(name='batch_long_256', kind='features', set='long', n=400, h=256, w=256, dtype='u16'),
        # a small study of 8-bit images through the short set
        dict(name='batch_short_128', kind='features', set='short', n=100, h=128, w=128, dtype='u8'),
        # tiles of uneven sizes, every side in [64, 1024]
        dict(name='tiles_long_ragged', kind='features', set='long', n=64, h=0, w=0, dtype='u16'),
        # whole microscope frames as 32-bit floats
        dict(name='frames_short_1388x1040', kind='features', set='short', n=3, h=1040, w=1388, dtype='f32'),
        # colour images through the largest set
        dict(name='color_long_231x208', kind='features', set='long_color', n=16, h=208, w=231, dtype='rgb8'),
        # one frame cut into 6 x 5 tiles, the long set of each
        dict(name='sampled_6x5', kind='sampled', n=1, h=1040, w=1388, tiles_x=6, tiles_y=5, rotations=1),
        # the reduced-precision form of the contractions
        dict(name='contractions_bf16', kind='contractions', n=200, h=128, w=128, precision=2),
        # forward and backward through the differentiable features
        dict(name='gradient_512', kind='gradient', n=16, h=512, w=512),
        # training statistics and the classification of a test set
        dict(name='classify_400', kind='classify', n=400, features=2919, classes=4, tests=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['features'] * 7 + ['sampled', 'contractions', 'gradient', 'classify', 'transform'])
    if kind == 'transform':
        return dict(kind=kind, h=_log_int(rng, 64, 1100), w=_log_int(rng, 64, 1400))
    if kind == 'features':
        s = rng.choice(['short', 'long', 'long', 'long', 'short_color', 'long_color'])
        color = s.endswith('color')
        dtype = rng.choice(['rgb8', 'rgb16'] if color else ['u8', 'u16', 'u16', 'f32', 'f64'])
        if not color and rng.random() < 0.25:  # uneven tiles
            return dict(kind=kind, set=s, n=rng.randint(8, 64), h=0, w=0, dtype=dtype)
        h, w = _log_int(rng, 64, 1024), _log_int(rng, 64, 1024)
        top = max(1, min(300, int(8e6 / (h * w) / (2 if s.startswith('long') else 1))))
        return dict(kind=kind, set=s, n=_log_int(rng, 1, top), h=h, w=w, dtype=dtype)
    if kind == 'sampled':
        return dict(kind=kind, n=1, h=rng.randint(400, 1040), w=rng.randint(400, 1388), tiles_x=rng.randint(1, 6),
                    tiles_y=rng.randint(1, 5), rotations=1)
    if kind == 'contractions':
        return dict(kind=kind, n=_log_int(rng, 8, 300), h=rng.randint(64, 256), w=rng.randint(64, 256),
                    precision=rng.choice([0, 1, 2]))
    if kind == 'gradient':
        return dict(kind=kind, n=_log_int(rng, 1, 16), h=rng.randint(96, 512), w=rng.randint(96, 512))
    return dict(kind=kind, n=_log_int(rng, 40, 1000), features=rng.choice([1059, 2919]), classes=rng.randint(2, 8),
                tests=_log_int(rng, 1, 200))


# ------------------------------------------------------------------ inputs
def _sizes(case):
    """(h, w) of every image: one size, or uneven tiles from the case alone"""
    if case['h']:
        return [(case['h'], case['w'])] * case['n']
    r = random.Random(case['n'])
    return [(r.randint(64, 1024), r.randint(64, 1024)) for _ in range(case['n'])]


def _planes(gen, n, h, w):
    """[n, h, w] int32 planes on the GPU: gratings of four periods, five blobs, Poisson noise, 12 bits"""
    dev = gen.device
    y = torch.arange(h, device=dev, dtype=torch.float32)[None, :, None]
    x = torch.arange(w, device=dev, dtype=torch.float32)[None, None, :]

    def u(lo, hi):
        return torch.empty(n, 1, 1, device=dev).uniform_(lo, hi, generator=gen)
    period = torch.tensor([6.0, 12.0, 24.0, 48.0], device=dev).repeat((n + 3) // 4)[:n, None, None]
    lam = torch.full((n, h, w), 500.0, device=dev)
    for _ in range(3):
        t, phi = u(0, math.pi), u(0, 2 * math.pi)
        lam += 200 * torch.sin(2 * math.pi * (x * torch.cos(t) + y * torch.sin(t)) / period + phi)
    for _ in range(5):
        a, s, cy, cx = u(300, 1500), u(4, 10), u(0, h), u(0, w)
        lam += a * torch.exp(-((y - cy) ** 2 + (x - cx) ** 2) / (2 * s * s))
    return torch.poisson(lam.clamp_(min=0), generator=gen).clamp_(0, 4095).to(torch.int32)


def _images(gen, sizes, dtype):
    """host arrays of the sample type"""
    out = []
    k = 0
    while k < len(sizes):
        j = k
        while j < len(sizes) and sizes[j] == sizes[k]:
            j += 1
        h, w = sizes[k]
        rgb = dtype.startswith('rgb')
        p = _planes(gen, (j - k) * (3 if rgb else 1), h, w).cpu().numpy()
        if rgb:
            p = np.ascontiguousarray(p.reshape(j - k, 3, h, w).transpose(0, 2, 3, 1))
        if dtype in ('u8', 'rgb8'):
            p = np.minimum(p >> 3, 255).astype(np.uint8)
        elif dtype in ('u16', 'rgb16'):
            p = p.astype(np.uint16)
        else:
            p = p.astype(np.float32 if dtype == 'f32' else np.float64)
        out += [np.ascontiguousarray(p[i]) for i in range(j - k)]
        k = j
    return out


def _standard(name):
    s = wndcharm.StdFeatureComputationPlans
    return [s.getFeatureSet, s.getFeatureSetLong, s.getFeatureSetColor, s.getFeatureSetLongColor][SETS[name]]()


def _families(plan):
    """column indices of each feature algorithm of a plan, so that every family is compared at its own scale"""
    fam = {}
    for c, name in enumerate(plan.feature_names()):
        group = name[:name.rindex(' [')]
        fam.setdefault(group if group in ROOT else group[:group.index(' (')], []).append(c)
    return {k: np.array(v) for k, v in fam.items()}


def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(seed * 7919 + 11)


def _classify_data(case, seed):
    """training features of separable classes with constant and heavy-tailed columns, and test vectors"""
    r = np.random.default_rng(seed)
    n, f, c = case['n'], case['features'], case['classes']
    cls = (np.arange(n) % c + 1).astype(np.int32)
    centre = r.normal(0, 1, (c, f)) * r.gamma(1.0, 1.0, f)
    scale = np.exp(r.normal(0, 2, f))
    train = (centre[cls - 1] + r.normal(0, 1, (n, f))) * scale
    train[:, ::97] = 3.0
    tcls = r.integers(0, c, case['tests'])
    test = (centre[tcls] + r.normal(0, 1, (case['tests'], f))) * scale
    test[:, ::97] = 3.0
    return train, cls, test


def prepare(case, seed):
    kind = case['kind']
    st = dict(case)
    if kind == 'transform':
        st['plane'] = _images(_gen(seed), [(case['h'], case['w'])], 'f64')[0]
        st['op'] = wndcharm.ImageTransform('Fourier')
    elif kind == 'features':
        st['images'] = _images(_gen(seed), _sizes(case), case['dtype'])
        st['plan'] = _standard(case['set'])
        st['families'] = _families(st['plan'])
    elif kind == 'sampled':
        st['images'] = _images(_gen(seed), _sizes(case), 'u16')
        st['plan'] = _standard('long')
        st['families'] = _families(st['plan'])
        st['sampling'] = wndcharm.Sampling(rotations=case['rotations'], tiles=(case['tiles_x'], case['tiles_y']))
    elif kind == 'contractions':
        st['images'] = _images(_gen(seed), _sizes(case), 'u16')
        plan = wndcharm.FeatureComputationPlan('contractions')
        for g in CONTRACTIONS:
            plan.add(g)
        plan.finalize()
        plan.set_precision(case['precision'])
        st['plan'] = plan
        st['families'] = _families(plan)
    elif kind == 'gradient':
        from wndcharm import autograd
        gen = _gen(seed)
        st['plan'] = autograd.DifferentiablePlan(list(GRADIENT))
        st['x'] = (_planes(gen, case['n'], case['h'], case['w']).to(torch.float64) / 4095).requires_grad_(True)
        st['g'] = torch.empty(case['n'], st['plan'].n_features, dtype=torch.float64,
                              device='cuda').normal_(generator=gen)
    else:
        st['train'], st['cls'], st['test'] = _classify_data(case, seed)
    return st


# ------------------------------------------------------------------ one pass
def _by_family(st, rows):
    return {k: rows[:, c] for k, c in st['families'].items()}


def run(st):
    kind = st['kind']
    if kind == 'transform':
        return st['op'].execute(st['plane'])
    if kind == 'features' and st['n'] == 1 and not st['dtype'].startswith('rgb'):
        vec = wndcharm.DoubleVector(st['plan'].n_features)
        wndcharm.FeatureComputationPlanExecutor(st['plan']).run(st['images'][0], vec, 0)
        return _by_family(st, vec.as_ndarray()[None])
    if kind in ('features', 'contractions'):
        return _by_family(st, wndcharm.compute_features(st['images'], st['plan']))
    if kind == 'sampled':
        return _by_family(st, wndcharm.compute_features(st['images'], st['plan'], sampling=st['sampling']))
    if kind == 'gradient':
        f = st['plan'](st['x'])
        grad, = torch.autograd.grad(f, st['x'], st['g'])
        out = {g: f.detach()[:, a:a + k] for a, k, g in st['plan'].columns}
        out['gradient'] = grad
        return out
    train, mins, maxs = wndcharm.normalize_train(st['train'])
    weights = wndcharm.fisher_weights(train, st['cls'], st['classes'])
    test = np.stack([wndcharm.normalize_test(v, mins, maxs) for v in st['test']])
    prob, norm, pred = wndcharm.wnd5(train, st['cls'], st['classes'], weights, test)
    return {'train': train, 'mins': mins, 'maxs': maxs, 'weights': weights, 'test': test, 'prob': prob,
            'norm': norm, 'predicted': pred}


# ------------------------------------------------------------------ what a pass cannot do without
_BYTES = {'u8': 1, 'u16': 2, 'f32': 4, 'f64': 8, 'rgb8': 3, 'rgb16': 6}


def work(case):
    """Each pixel read once and each feature written once; the arithmetic of the
    contractions, per pixel and plane: Gabor 8 filters of 38 x 38 complex taps
    with 4 operations, Chebyshev-Fourier 2 x 23 x 23 products over the disk,
    Zernike 72 complex moments, the Chebyshev transform 2 N products per pixel
    and pass; and per co-occurrence matrix of 128 tones (the order of the
    usual images) the 10/3 N^3 of a Hessenberg reduction and the 10 N^3 of the
    QR iteration."""
    kind = case['kind']
    if kind == 'classify':
        n, f, t = case['n'], case['features'], case['tests']
        return {'bytes': 16.0 * f * (n + t), 'flops': 3.0 * n * f * t + 10.0 * n * f}
    if kind == 'transform':
        p = case['h'] * case['w']
        return {'bytes': 16.0 * p, 'flops': 5.0 * p * math.log2(p)}
    sizes = _sizes(case)
    p = float(sum(h * w for h, w in sizes))
    gabor, cf, zern = 46208.0 * p, 1661.0 * p, 288.0 * p
    if kind == 'gradient':
        c = sum(8.0 * min(h, w) * h * w for h, w in sizes)
        return {'bytes': 16.0 * p, 'flops': 3 * gabor + 3 * (3 * zern + cf) + 2 * c}
    if kind == 'contractions':
        return {'bytes': 2.0 * p + 8.0 * 143 * case['n'], 'flops': gabor + cf + zern}
    nf, nodes, cheb, colour = {'short': (1059, 6, 2, 0), 'long': (2919, 12, 4, 0), 'short_color': (2199, 10, 3, 1),
                               'long_color': (4059, 16, 5, 1)}['long' if kind == 'sampled' else case['set']]
    m = case['n'] * (case['tiles_x'] * case['tiles_y'] if kind == 'sampled' else 1)
    c = sum(4.0 * min(h, w) * h * w for h, w in sizes) / (1 if m == case['n'] else case['tiles_x'])
    b = _BYTES['u16' if kind == 'sampled' else case['dtype']]
    return {'bytes': b * p + 8.0 * nf * m,
            'flops': gabor + nodes / 2 * (cf + zern) + cheb * c + m * nodes * 4 * (10 / 3 + 10) * 128.0 ** 3}


def tolerance(case):
    kind = case['kind']
    if kind == 'classify':
        return {'rel': 1e-12, 'max': 1e-10}
    if kind == 'gradient':
        return {'rel': 1e-10, 'max': 1e-8}
    if kind == 'transform':
        return {'rel': 1e-14, 'max': 1e-12}
    # histograms and counts are whole numbers (or ratios of them); sums over
    # pixels differ by rounding, most where they cancel
    return {'rel': 1e-9, 'max': 1e-7}


# ------------------------------------------------------------------ in 64 bits, without the framework
def _fourier(x):
    return torch.fft.fft2(x).abs()


def _chebyshev(x, order=None):
    h, w = x.shape[-2:]
    n = order or min(h, w)

    def basis(length):
        a = torch.arange(length, dtype=torch.float64, device=x.device)
        j = torch.arange(n, dtype=torch.float64, device=x.device)
        t = torch.cos(j[None, :] * torch.acos((2 * (a + 1) / length - 1).clamp(-1, 1))[:, None]) * (2.0 / length)
        t[:, 0] = 1.0 / length
        return t
    return 0.25 * (basis(w).t().contiguous() @ x.t().contiguous() @ basis(h))


def _zernike(img):
    """order 15, the angle of repetition m taken as (m + 1) theta"""
    h, w = img.shape
    total = img.sum()
    i = torch.arange(1, w + 1, dtype=torch.float64, device=img.device)
    j = torch.arange(1, h + 1, dtype=torch.float64, device=img.device)
    x = ((i[None, :] - (img * i[None, :]).sum() / total) / min(w, h)).expand(h, w)
    y = ((j[:, None] - (img * j[:, None]).sum() / total) / min(w, h)).expand(h, w)
    r = torch.sqrt(x * x + y * y)
    inside = (r >= 2.0 ** -52) & (r <= 1)
    r, theta, f = r[inside], torch.atan2(y[inside], x[inside]), img[inside] / total
    out = []
    for n in range(16):
        for m in range(n % 2, n + 1, 2):
            radial = sum((-1) ** s * math.factorial(n - s) /
                         (math.factorial(s) * math.factorial((n + m) // 2 - s) * math.factorial((n - m) // 2 - s)) *
                         r ** (n - 2 * s) for s in range((n - m) // 2 + 1))
            k = (n + 1) / math.pi * f * radial
            out.append(torch.hypot((k * torch.cos((m + 1) * theta)).sum(), (k * torch.sin((m + 1) * theta)).sum()))
    return torch.stack(out)


def _statistics(img):
    v = img.reshape(-1).sort().values
    n = v.numel()
    return torch.stack([v.mean(), (v[n // 2] + v[(n - 1) // 2]) / 2, v.std(), v[0], v[-1]])


def _gini(img):
    v = img.reshape(-1)
    v = v[v > 0].sort().values
    n = v.numel()
    i = torch.arange(1, n + 1, dtype=torch.float64, device=v.device)
    return (((2 * i - n - 1) * v).sum() / (v.mean() * n * (n - 1))).reshape(1)


def _multiscale(img):
    lo, hi = float(img.min()), float(img.max())
    counts = torch.cat([torch.bincount(((img - lo) * (b / (hi - lo))).long().clamp(max=b - 1).reshape(-1), minlength=b)
                        for b in (3, 5, 7, 9)]).double()
    return counts / counts.max()


def _fractal(img):
    h, w = img.shape
    top = min(h, w) // 5
    out = torch.zeros(20, dtype=torch.float64, device=img.device)
    for i, k in enumerate(list(range(1, top, max(1, top // 20)))[:20]):
        d = (img[:-k] - img[k:]).abs().sum() + (img[:, :-k] - img[:, k:]).abs().sum()
        out[i] = d / (w * (w - k) + h * (h - k))
    return out


def _exact_classify(case, seed):
    raw, cls, test = _classify_data(case, seed)
    mins, maxs = raw.min(0), raw.max(0)
    span, eps = maxs - mins, np.finfo(np.float64).eps

    def norm(v):
        q = np.where(v > maxs, 100.0, 100 * (v - mins) / np.where(span < eps, 1.0, span))
        return np.where((v < mins) | (span < eps), 0.0, q)
    return {'train': norm(raw), 'mins': mins, 'maxs': maxs, 'weights': None, 'test': norm(test), 'prob': None,
            'norm': None, 'predicted': None}


def exact(case, seed):
    """The transform; the normalisation; of the gradient case the Zernike and
    Chebyshev groups; of gray images the groups of ROOT.  The other features
    are histograms of values at the edges of their bins, or follow the order
    of the reference's own operations, and have no other value."""
    kind = case['kind']
    if kind == 'classify':
        return _exact_classify(case, seed)
    if kind == 'transform':
        plane = torch.from_numpy(_images(_gen(seed), [(case['h'], case['w'])], 'f64')[0])
        return _fourier(plane.cuda()).cpu().numpy()
    if kind == 'gradient':
        x = _planes(_gen(seed), case['n'], case['h'], case['w']).to(torch.float64) / 4095
        out = dict.fromkeys(GRADIENT + ('gradient',))
        out['Zernike Coefficients ()'] = torch.stack([_zernike(p) for p in x])
        out['Zernike Coefficients (Fourier ())'] = torch.stack([_zernike(_fourier(p)) for p in x])
        out['Zernike Coefficients (Chebyshev ())'] = torch.stack([_zernike(_chebyshev(p)) for p in x])
        out['Chebyshev Coefficients (raw) ()'] = torch.stack([_chebyshev(p, 20).reshape(-1) for p in x])
        return out
    if kind == 'sampled' or case.get('set', '').endswith('color') or sum(h * w for h, w in _sizes(case)) > 3e7:
        return None
    plan = prepare(case, seed)
    out = dict.fromkeys(plan['families'])
    alg = {'Pixel Intensity Statistics ()': _statistics, 'Gini Coefficient ()': _gini,
           'Multiscale Histograms ()': _multiscale, 'Fractal Features ()': _fractal, 'Zernike Coefficients ()': _zernike}
    planes = [torch.from_numpy(im.astype(np.float64)).cuda() for im in plan['images']]
    for g in ROOT:
        if g in out:
            out[g] = torch.stack([alg[g](p) for p in planes]).cpu().numpy()
    return out
