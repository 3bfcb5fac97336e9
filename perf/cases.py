"""Timed workloads of the framework's image formation, each through its public entry points.

listed()    the workloads by name: from a chip of 128 x 128 pixels to the 12,288 x 8,192 image of the benchmark,
            factorized backprojection (ImageFormer), exact backprojection (ExactFormer) and a batch of uneven images
draw(rng)   one more workload of the same ranges
prepare     the geometry's former and a phase history, resident on the GPU unless the workload is a host one
run         one image (or one batch of images)
work        the bytes and operations the method itself needs
exact       the image in float64 by direct backprojection in torch, where that takes seconds

A workload is a dict: kind ('ffbp', 'exact' or 'batch'), the grid nx x ny at spacing sp, pulses x samples, the squint,
the former's options, how the history is stored ('complex64', 'cphd16', 'float16', 'bfloat16') and where it lies.

Scenes: an X-band spotlight collection at 10 km slant range and 30 degrees grazing, sampled for its image as a
processor's input is (range and azimuth extents unambiguous over the image's diagonal, range resolution no finer
than the pixel, apertures up to 6 degrees); point targets with Rayleigh amplitudes over white clutter 25 dB down.
"""
import math

import numpy as np
import torch

from fastsar_amd import ExactFormer, ImageFormer, _hip, metrics
from fastsar_amd import plan as planner
from fastsar_amd.batch import Batch
from fastsar_amd.precision import CphdSignal, pack

C = 299792458.0
R0, GRAZE, FC = 10e3, math.radians(30.0), 9.6e9
E1, E2 = (0.0, 1.0, 0.0), (1.0, 0.0, 0.0)
TARGETS = 24
DEV = 'cuda'

FFBP = dict(kind='ffbp', sp=0.5, squint=0.0, T=0, levels=0, atten=70.0, precision='float32', history='complex64',
            host=False, weighted=False, gate=False, bandwidth=0.0, aperture=0.0)
EXACT = dict(kind='exact', sp=0.5, squint=0.0, interp='cubic', profiles='auto', history='complex64', host=False,
             bandwidth=0.0, aperture=0.0)


def _ffbp(name, nx, ny, P, K, **kw):
    return dict(FFBP, name=name, nx=nx, ny=ny, P=P, K=K, **kw)


def _exact(name, nx, ny, P, K, **kw):
    return dict(EXACT, name=name, nx=nx, ny=ny, P=P, K=K, **kw)


def listed():
    return [
        # a target chip with the former's default options: the smallest call, all launches and host work (the
        # autofocus loop forms such an image on every iteration)
        _ffbp('chip_128', 128, 128, 190, 190),
        # the small spotlight image of the benchmark (512 x 512 from 512 pulses x 1,024 samples)
        _ffbp('spot_512', 512, 512, 512, 1024, T=8, levels=4, atten=80.0, bandwidth=300e6, aperture=3.0),
        # a squinted patch of odd sizes straight from a CPHD file's int16 signal array, default options
        _ffbp('patch_1001x747_cphd', 1001, 747, 1403, 2045, squint=2.0, history='cphd16'),
        # a small image from a wide-band history (a large first range decimation), finest final tiles
        _ffbp('wideband_534', 534, 534, 1400, 4088, squint=2.0, T=4, levels=4, atten=80.0),
        # a mosaic's patch: per-pixel aperture weights, each pulse cut in range to the patch on the device
        _ffbp('mosaic_patch_384', 384, 384, 1535, 2048, weighted=True, gate=True),
        # an image of a few megapixels at the benchmark's accuracy settings
        _ffbp('spot_2048', 2048, 2048, 4096, 2048, T=8, levels=4, atten=80.0),
        # the same kind of image as most programs call it: host history in, host image out, default options
        _ffbp('host_1536', 1536, 1536, 3000, 1536, host=True),
        # a wide image with float16 level rows, the lower-precision option
        _ffbp('strip_4095x3001_float16', 4095, 3001, 8190, 3073, T=8, levels=4, atten=80.0, precision='float16'),
        # the benchmark's image
        _ffbp('image_12288x8192', 12288, 8192, 16384, 8192, sp=6000.0 / 12288, T=8, levels=4, atten=80.0,
              bandwidth=300e6, aperture=6.0),
        # exact backprojection, default options
        _exact('exact_1024', 1024, 1024, 2048, 2048),
        # exact backprojection of a larger odd grid, linear reads of float16 profile pairs
        _exact('exact_2001x1603_linear16', 2001, 1603, 4001, 2048, interp='linear', profiles='float16-pair'),
        # uneven images formed together in one graph launch
        dict(kind='batch', name='batch_12', images=12, seed=5),
    ]


def _log(rng, lo, hi):
    return int(round(2.0 ** rng.uniform(math.log2(lo), math.log2(hi))))


def draw(rng):
    if rng.random() < 0.25:
        P = _log(rng, 200, 4096)
        interp = rng.choice(['cubic', 'linear'])
        prof = rng.choice(['auto', 'float16'] if interp == 'cubic' else ['auto', 'float16', 'float16-pair'])
        c = dict(EXACT, nx=_log(rng, 100, 2600), ny=_log(rng, 100, 2600), P=P, K=_log(rng, 200, 4096), interp=interp,
                 profiles=prof, squint=rng.choice([0.0, 2.0]))
        return c
    nx, ny = _log(rng, 128, 4096), _log(rng, 128, 4096)
    c = dict(FFBP, nx=nx, ny=ny, P=_log(rng, 256, 8192), K=_log(rng, 256, 4096), squint=rng.choice([0.0, 2.0]))
    if rng.random() < 0.6:
        c.update(T=rng.choice([4, 8, 8, 16]), levels=4, atten=80.0)
    if rng.random() < 0.2:
        c.update(precision='float16')
    elif c['P'] * c['K'] < 1 << 22 and rng.random() < 0.3:
        c.update(history=rng.choice(['cphd16', 'float16', 'bfloat16']))
    return c


# ------------------------------------------------------------------------------------------------ scenes

def _geometry(case):
    """ant [P, 3], fmin, df of the case's collection."""
    P, K = case['P'], case['K']
    lam, psi = C / FC, GRAZE
    ground = R0 * math.cos(psi)
    extent = 1.25 * math.hypot(case['nx'], case['ny']) * case['sp']
    df = min(C / (2.0 * extent), C / (2.0 * case['sp']) / K)
    if case['bandwidth']:
        df = case['bandwidth'] / K
    dy = min(lam * R0 / (2.0 * extent), 2.0 * ground * math.tan(math.radians(3.0)) / (P - 1))
    if case['aperture']:
        dy = 2.0 * ground * math.tan(math.radians(case['aperture'] / 2.0)) / (P - 1)
    y = (np.arange(P) - 0.5 * (P - 1)) * dy + ground * math.tan(math.radians(case['squint']))
    ant = np.stack([np.full(P, -ground), y, np.full(P, R0 * math.sin(psi))], axis=1)
    return ant, FC - (K // 2) * df, df


def _scene(case, seed, ant, fmin, df):
    """The phase history [P, K] complex64 on the GPU: targets over 80 % of the grid, white clutter."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    n, P, K = TARGETS, case['P'], case['K']
    u = torch.rand((n, 2), generator=g, device=DEV, dtype=torch.float64) - 0.5
    amp = torch.randn((n, 2), generator=g, device=DEV, dtype=torch.float64) / math.sqrt(2.0)
    pos = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
    pos[:, 1] = 0.8 * case['nx'] * case['sp'] * u[:, 0]
    pos[:, 0] = 0.8 * case['ny'] * case['sp'] * u[:, 1]
    a = torch.as_tensor(ant, device=DEV)
    rows = max(1, (1 << 25) // K)
    k = torch.arange(K, device=DEV, dtype=torch.float64)
    sigma = math.sqrt(float((amp ** 2).sum()) * 10.0 ** -2.5 / 2.0)
    S = torch.randn((P, K, 2), generator=g, device=DEV, dtype=torch.float32).mul_(sigma)
    for p0 in range(0, P, rows):
        ap = a[p0:p0 + rows]
        dr = (pos[None] - ap[:, None]).norm(dim=2) - ap.norm(dim=1)[:, None]
        for t in range(n):
            cyc = (-2.0 / C) * dr[:, t, None] * (fmin + df * k)[None, :]
            ph = ((cyc - cyc.round()) * (2.0 * math.pi)).float()
            c, s = ph.cos(), ph.sin()
            ar, ai = float(amp[t, 0]), float(amp[t, 1])
            S[p0:p0 + rows, :, 0] += ar * c - ai * s
            S[p0:p0 + rows, :, 1] += ar * s + ai * c
    return torch.view_as_complex(S)


def _weight(ant, case):
    """A mosaic's azimuth window: a raised cosine of each pulse's along-track place relative to the pixel."""
    half = 0.6 * float(np.ptp(ant[:, 1]))
    mid = float(ant[:, 1].mean())

    def weight(points, pulses):
        v = (ant[np.asarray(pulses), 1][:, None] - mid - np.asarray(points)[None, :, 1]) / half
        return 0.5 + 0.5 * np.cos(np.pi * np.clip(v, -1.0, 1.0))
    return weight


class _Memory:
    """The CUDA array interface of a DeviceArray's memory, so that torch sees it without a copy."""

    def __init__(self, d):
        self.keep = d
        self.__cuda_array_interface__ = dict(shape=d.shape, typestr=d.dtype.str, data=(d.ptr, False), version=2, strides=None)


def _device(shape):
    d = _hip.DeviceArray(shape, np.complex64)
    return d, torch.as_tensor(_Memory(d), device=DEV)


def _former(case, ant, fmin, df):
    grid = (ant, fmin, df, case['K'], case['nx'], case['ny'], case['sp'], case['sp'], E1, E2)
    if case['kind'] == 'exact':
        return ExactFormer(*grid, interp=case['interp'], profiles=case['profiles'])
    return ImageFormer(*grid, T=case['T'] or 'auto', levels=case['levels'] or None, atten=case['atten'],
                       precision=case['precision'], range_gate=True if case['gate'] else 'auto',
                       aperture_weight=_weight(ant, case) if case['weighted'] else None)


def _typed(S, kind):
    """The host history S in a stored type."""
    if kind != 'cphd16':
        return pack(S, kind)
    amp = (np.maximum(np.abs(S.real), np.abs(S.imag)).max(1) / 30000.0).astype(np.float32)
    q = np.rint(np.stack([S.real, S.imag], 2) / amp[:, None, None])
    return CphdSignal(q.astype('>i2'), amp)


def _batch_cases(case):
    rng = np.random.default_rng(case['seed'])
    out = []
    for i in range(case['images']):
        side, P, K = (int(round(2.0 ** rng.uniform(math.log2(lo), math.log2(hi)))) for lo, hi in ((256, 2048), (512, 4096), (1024, 4096)))
        out.append(dict(FFBP, nx=side, ny=side, P=P, K=K, squint=2.0 * (i % 2), T=8, levels=4, atten=80.0))
    return out


def prepare(case, seed):
    if case['kind'] == 'batch':
        formers, hists, images, views = [], [], [], []
        for i, c in enumerate(_batch_cases(case)):
            ant, fmin, df = _geometry(c)
            S, t = _device((c['P'], c['K']))
            t.copy_(_scene(c, 1000 * seed + i, ant, fmin, df))
            img, v = _device((c['nx'], c['ny']))
            formers.append(_former(c, ant, fmin, df))
            hists.append(S)
            images.append(img)
            views.append(v)
        torch.cuda.synchronize()
        return dict(kind='batch', batch=Batch(formers, hists, images), views=views)
    ant, fmin, df = _geometry(case)
    former = _former(case, ant, fmin, df)
    hist = _scene(case, seed, ant, fmin, df)
    if case['host']:
        return dict(kind='host', former=former, S=hist.cpu().numpy())
    if case['history'] != 'complex64':
        S = _typed(hist.cpu().numpy(), case['history']).to_device()
    else:
        S, t = _device((case['P'], case['K']))
        t.copy_(hist)
    img, view = _device((case['nx'], case['ny']))
    torch.cuda.synchronize()
    return dict(kind='device', former=former, S=S, img=img, view=view)


def run(state):
    if state['kind'] == 'batch':
        state['batch'].run()
        return state['views']
    if state['kind'] == 'host':
        return state['former'](state['S'])
    state['former'](state['S'], out=state['img'])
    return state['view']


# ------------------------------------------------------------------------------------------------ work

SAMPLE_BYTES = {'complex64': 8, 'cphd16': 4, 'float16': 4, 'bfloat16': 4}


def work(case):
    if case['kind'] == 'batch':
        parts = [work(c) for c in _batch_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ('bytes', 'flops')}
    N, P, K = case['nx'] * case['ny'], case['P'], case['K']
    io = SAMPLE_BYTES[case['history']] * P * K + 8 * N
    if case['kind'] == 'exact':
        # per pixel and pulse: the range (7), its bin and weights (12 cubic, 2 linear), the read (16, 8), the phase's
        # sine and cosine (2) and the complex multiply-add (8); per pulse the transform of the profiles
        nfft = 1 << math.ceil(math.log2(8 * K))
        return dict(bytes=io, flops=(45.0 if case['interp'] == 'cubic' else 27.0) * N * P + 5.0 * P * nfft * math.log2(nfft))
    # the factorization's own counts for the plan these options make: rotations, decimation filters, final products
    ant, fmin, df = _geometry(case)
    col = type('Collection', (), dict(fmin=fmin, df=df, K=K, ant=ant))()
    T, nlev = case['T'], case['levels'] or 3
    if not T:
        T, _ = planner.choose_T(ant, fmin + K * df, case['nx'], case['ny'], case['sp'], case['sp'], E1, E2, -40.0,
                                choices=(32, 16, 8, 4))
    while True:
        try:
            plan = planner.make_plan(col, case['nx'], case['ny'], case['sp'], case['sp'], T=T, nlev=nlev, atten=case['atten'],
                                     e1=E1, e2=E2)
            break
        except ValueError:
            nlev += 1
    return dict(bytes=io, flops=sum(v for (stage, _), v in metrics.stage_flops(plan).items()
                                    if stage in ('rot_fir_k', 'fir_p', 'final_tiles')))


# ------------------------------------------------------------------------------------------------ exact

EXACT_PAIRS = 2.5e10      # pixel-pulse pairs a direct float64 image is formed for (about 10 s)


def _taylor(n, sll=35.0, nbar=4):
    """The Taylor window of n samples (unnormalized), in float32 as the formers hold it."""
    B = 10.0 ** (sll / 20.0)
    A = math.acosh(B) / math.pi
    s2 = nbar ** 2 / (A ** 2 + (nbar - 0.5) ** 2)
    m = np.arange(1, nbar)
    x = (np.arange(n) - n / 2.0 + 0.5) / n
    w = np.ones(n)
    for i in m:
        num = (-1.0) ** (i + 1) * np.prod(1.0 - i ** 2 / s2 / (A ** 2 + (m - 0.5) ** 2))
        den = 2.0 * np.prod([1.0 - i ** 2 / j ** 2 for j in m if j != i])
        w += 2.0 * num / den * np.cos(2.0 * np.pi * i * x)
    return w.astype(np.float32)


def _stored(S, kind):
    """The values a stored history holds, complex128."""
    if kind == 'complex64':
        return S.to(torch.complex128)
    re, im = S.real.contiguous(), S.imag.contiguous()
    if kind == 'bfloat16':
        return torch.complex(re.bfloat16().double(), im.bfloat16().double())
    big = torch.maximum(re.abs(), im.abs()).amax(1, keepdim=True)
    if kind == 'float16':
        g = 2.0 ** (14 - big.double().log2().ceil())
        return torch.complex((re * g.float()).half().double(), (im * g.float()).half().double()) / g
    amp = big / 30000.0
    return torch.complex((re / amp).round().double(), (im / amp).round().double()) * amp.double()


def _backproject(case, seed):
    """The image in complex128 by direct backprojection: profiles oversampled 64 times, cubic reads, exact ranges."""
    ant, fmin, df = _geometry(case)
    nx, ny, P, K = case['nx'], case['ny'], case['P'], case['K']
    S = _stored(_scene(case, seed, ant, fmin, df), case['history'])
    w = torch.as_tensor(_taylor(P), device=DEV)[:, None] * torch.as_tensor(_taylor(K), device=DEV)[None, :]
    S = S * w.double()
    nfft = 1 << math.ceil(math.log2(64 * K))
    h = K // 2
    X = ((torch.arange(nx, device=DEV, dtype=torch.float64) - nx / 2.0) * case['sp'])[:, None].expand(nx, ny)
    Y = ((torch.arange(ny, device=DEV, dtype=torch.float64) - ny / 2.0) * case['sp'])[None, :].expand(nx, ny)
    kcyc, inv_dr = 2.0 * (fmin + h * df) / C, 2.0 * df * nfft / C
    weight = _weight(ant, case) if case.get('weighted') else None
    pts = torch.stack([Y, X, torch.zeros_like(X)], 2).reshape(-1, 3).cpu().numpy() if weight else None
    out = torch.zeros((nx, ny), device=DEV, dtype=torch.complex128)
    pad = torch.zeros(nfft, device=DEV, dtype=torch.complex128)
    for p in range(P):
        pad[:K - h] = S[p, h:]
        pad[nfft - h:] = S[p, :h]
        prof = torch.fft.ifft(pad) * nfft
        ax, ay, az = (float(v) for v in ant[p])
        dR = torch.sqrt((Y - ax) ** 2 + (X - ay) ** 2 + az * az) - math.sqrt(ax * ax + ay * ay + az * az)
        t = dR * inv_dr
        i = t.floor()
        f = t - i
        i = i.long()
        v = prof[(i - 1) % nfft] * (-f * (f - 1) * (f - 2) / 6)
        v += prof[i % nfft] * ((f + 1) * (f - 1) * (f - 2) / 2)
        v += prof[(i + 1) % nfft] * (-(f + 1) * f * (f - 2) / 2)
        v += prof[(i + 2) % nfft] * ((f + 1) * f * (f - 1) / 6)
        ph = kcyc * dR
        v *= torch.polar(torch.ones_like(ph), 2.0 * math.pi * (ph - ph.round()))
        if weight:
            v *= torch.as_tensor(weight(pts, np.array([p]))[0], device=DEV).reshape(nx, ny)
        out += v
    return out


def exact(case, seed):
    if case['kind'] == 'batch':
        # the images of the batch that take a second or less
        got = [_backproject(c, 1000 * seed + i) if c['nx'] * c['ny'] * c['P'] <= 1e9 else None
               for i, c in enumerate(_batch_cases(case))]
        return got if any(g is not None for g in got) else None
    if case['nx'] * case['ny'] * case['P'] > EXACT_PAIRS:
        return None
    out = _backproject(case, seed)
    return out.cpu().numpy() if case['host'] else out
