"""Workloads of scopyon_amd for performance measurement.

``listed()`` holds the fixed cases, ``draw(rng)`` one more of the same ranges;
``prepare(case, seed)`` makes what a program holds before the call (inputs from
the seed, the simulator or model), ``run(state)`` is one pass through the public
entry points, ``work(case)`` the bytes and operations a pass cannot do without
and ``exact(case, seed)`` the outputs in 64 bits where they are computed numbers
(frames drawn from random number streams have none).

Kinds of case:
  frame   ``EPIFMSimulator.form_image`` with a RandomState (the drop-in path)
  movie   ``EPIFMSimulator.generate_images`` with PhiloxRNG, one time point per frame
  walk    ``scopyon_amd.sample`` trajectories
  batch   ``BatchedSimulator`` time steps of many fields of view (2D), eager or
          replayed from a captured graph
  depth   ``BatchedSimulator`` over a depth range: LUT steps, or noise-free frames
          from the 1 nm tables
  render  ``GaussianModel.forward`` in the precision forms
  fit     Gaussian forward + Poisson NLL + backward, raw or through autograd
"""
import math

import numpy
import torch

import scopyon_amd
from scopyon_amd.batched import BatchedSimulator
from scopyon_amd.gauss import GaussianModel, poisson_nll, render


def listed():
    return [
        # one drop-in frame as a script makes it: 512 x 512 EMCCD, 160 nm pixels, dense sample
        {'name': 'frame_10k', 'kind': 'frame', 'nw': 512, 'nh': 512, 'n': 10000, 'mag': 100.0,
         'detector': 'EMCCD', 'dims': 2, 'full': False},
        # a 3D sample at the default magnification on an odd region of interest, with the
        # ground truth returned: most of the emitters meet a depth table of their own
        {'name': 'frame_3d', 'kind': 'frame', 'nw': 201, 'nh': 333, 'n': 120, 'mag': 241.0,
         'detector': 'EMCCD', 'dims': 3, 'full': True},
        # a short movie of moving, bleaching fluorophores on an sCMOS camera, device random numbers
        {'name': 'movie_1k', 'kind': 'movie', 'nw': 512, 'nh': 512, 'n': 1000, 'mag': 100.0,
         'detector': 'CMOS', 'frames': 4},
        # trajectories for such a movie: 1,000 particles, 50 time points, RandomState
        {'name': 'walk_1k', 'kind': 'walk', 'n': 1000, 't': 50, 'ndim': 2, 'states': 1,
         'periodic': True, 'rng': 'state'},
        # the plain configuration, one field of view per eager step: the smallest step
        {'name': 'single_1k', 'kind': 'batch', 'fovs': 1, 'sizes': '512x512', 'n': 1000,
         'spread': 0.0, 'layout': 1, 'mag': 100.0, 'detector': 'EMCCD', 'graph': False},
        # the benchmark's headline: 64 fields of view of 512 x 512 with 10,000 emitters each
        {'name': 'batch_64', 'kind': 'batch', 'fovs': 64, 'sizes': '512x512', 'n': 10000,
         'spread': 0.0, 'layout': 1, 'mag': 100.0, 'detector': 'EMCCD', 'graph': True},
        # 256 fields of view of mixed sizes and lognormal emitter counts
        {'name': 'uneven_256', 'kind': 'batch', 'fovs': 256, 'sizes': '128x128,256x256,512x512',
         'n': 5000, 'spread': 1.0, 'layout': 17, 'mag': 100.0, 'detector': 'EMCCD', 'graph': True},
        # 3D scale-up: 100,000 emitters over +-1 um of depth, 1024 x 1024 at 66.4 nm, LUT PSF
        {'name': 'depth_lut', 'kind': 'depth', 'psf': 'lut', 'nw': 1024, 'nh': 1024, 'n': 100000,
         'mag': 241.0, 'depth': 1.0e-6},
        # the same sample as noise-free images from the 1 nm parity tables
        {'name': 'depth_table', 'kind': 'depth', 'psf': 'table', 'nw': 1024, 'nh': 1024,
         'n': 100000, 'mag': 241.0, 'depth': 1.0e-6},
        # precision study: a million emitters on 2048 x 2048, bfloat16 operands
        {'name': 'render_1m', 'kind': 'render', 'fovs': 1, 'nw': 2048, 'nh': 2048, 'n': 1000000,
         'sigma': 1.2, 'radius': 6, 'method': 'mfma-bf16'},
        # refinement of many frames: the loss and every gradient, float32 operands
        {'name': 'fit_64', 'kind': 'fit', 'fovs': 64, 'nw': 256, 'nh': 256, 'n': 5000,
         'sigma': 1.2, 'radius': 6, 'auto': False},
        # one small odd frame fitted through autograd with an ordinary optimiser
        {'name': 'fit_small', 'kind': 'fit', 'fovs': 1, 'nw': 61, 'nh': 83, 'n': 300,
         'sigma': 1.35, 'radius': 6, 'auto': True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['frame', 'movie', 'walk', 'batch', 'batch', 'depth', 'render', 'fit', 'fit'])
    if kind in ('frame', 'movie'):
        case = {'kind': kind, 'nw': _log(rng, 48, 512), 'nh': _log(rng, 48, 512),
                'mag': rng.choice([100.0, 160.0, 241.0]),
                'detector': rng.choice(['EMCCD', 'EMCCD', 'CMOS', 'CCD'])}
        if kind == 'movie':
            return dict(case, n=_log(rng, 50, 2000), frames=rng.randint(2, 5))
        dims = rng.choice([2, 3])
        return dict(case, n=_log(rng, 30, 10000) if dims == 2 else _log(rng, 20, 150), dims=dims,
                    full=rng.random() < 0.3)
    if kind == 'walk':
        return {'kind': kind, 'n': _log(rng, 100, 20000), 't': rng.randint(10, 60),
                'ndim': rng.choice([2, 3]), 'states': rng.choice([1, 1, 3]),
                'periodic': rng.random() < 0.5, 'rng': rng.choice(['state', 'philox'])}
    if kind == 'batch':
        fovs = _log(rng, 1, 128)
        sizes = ','.join('{}x{}'.format(_log(rng, 96, 512), _log(rng, 96, 512))
                         for _ in range(rng.randint(1, 3)))
        return {'kind': kind, 'fovs': fovs, 'sizes': sizes, 'n': _log(rng, 200, 8000),
                'spread': rng.choice([0.0, 0.5, 1.0]), 'layout': rng.randrange(1, 1000),
                'mag': rng.choice([100.0, 100.0, 160.0]),
                'detector': rng.choice(['EMCCD', 'EMCCD', 'EMCCD', 'CMOS', 'CCD']),
                'graph': rng.random() < 0.7}
    if kind == 'depth':
        psf = rng.choice(['lut', 'lut', 'table'])
        return {'kind': kind, 'psf': psf, 'nw': _log(rng, 200, 1024), 'nh': _log(rng, 200, 1024),
                'n': _log(rng, 1000, 100000), 'mag': rng.choice([150.0, 241.0]),
                'depth': rng.choice([0.2e-6, 0.5e-6, 1.0e-6])}
    sigma = rng.uniform(0.8, 1.8)
    if kind == 'render':
        fovs = rng.choice([1, 1, 2, 7])
        return {'kind': kind, 'fovs': fovs, 'nw': _log(rng, 200, 2048) // fovs + 40,
                'nh': _log(rng, 200, 2048), 'n': _log(rng, 5000, 1000000) // fovs, 'sigma': sigma,
                'radius': rng.choice([5, 6, 7]),
                'method': rng.choice(['mfma-f32', 'mfma-f16', 'mfma-bf16'])}
    fovs = _log(rng, 1, 64)
    return {'kind': kind, 'fovs': fovs, 'nw': _log(rng, 48, 256), 'nh': _log(rng, 48, 256),
            'n': _log(rng, 100, 5000), 'sigma': sigma, 'radius': rng.choice([5, 6, 7]),
            'auto': rng.random() < 0.5}


# ---- what the cases are made of ----

def _config(case, size, exposure, bleach=False, angle=None):
    over = {'magnification': case['mag'],
            'detector': {'type': case.get('detector', 'EMCCD'), 'image_size': list(size),
                         'exposure_time': exposure},
            'effects': {'photo_bleaching': {'switch': bleach}}}
    if angle is not None:
        over['light_source'] = {'angle': angle}
    config = scopyon_amd.DefaultConfiguration()
    config.update({'default': over})
    return config


def _layout(case):
    """Frame sizes and emitter counts of a batch: they belong to the case, not to the seed."""
    rng = numpy.random.Generator(numpy.random.Philox(case['layout']))
    sizes = [tuple(int(v) for v in s.split('x')) for s in case['sizes'].split(',')]
    pick = rng.integers(0, len(sizes), case['fovs'])
    counts = numpy.exp(rng.normal(math.log(case['n']), case['spread'], case['fovs']))
    return [sizes[i] for i in pick], numpy.clip(counts, 100, 50000).round().astype(int)


def _frame_inputs(case, seed):
    """Positions in metres: uniform over the frame, and over +-0.5 um of depth in 3D."""
    rng = numpy.random.RandomState(seed % (1 << 32))
    pl = 16.0e-6 / case['mag']
    half = numpy.array([case['nw'], case['nh']]) * pl / 2
    xy = rng.uniform(-1.0, 1.0, size=(case['n'], 2)) * half
    if case.get('dims', 2) == 2:
        return xy
    return numpy.hstack([xy, rng.uniform(-0.5e-6, 0.5e-6, size=(case['n'], 1))])


def _depth_positions(case, seed):
    rng = numpy.random.Generator(numpy.random.Philox(seed))
    pl = 16.0e-6 / case['mag']
    n = case['n']
    return (rng.uniform(-case['depth'], case['depth'], n),
            rng.uniform(-0.5, 0.5, n) * 0.8 * case['nw'] * pl,
            rng.uniform(-0.5, 0.5, n) * 0.8 * case['nh'] * pl)


def _gauss_inputs(case, seed):
    """Emitters of a Gaussian case, float32 on the GPU: x, y, z, I, frame id."""
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    n = case['n'] * case['fovs']

    def uniform(lo, hi):
        return lo + (hi - lo) * torch.rand(n, generator=g, device='cuda')

    x, y, z = uniform(0, case['nw']), uniform(0, case['nh']), uniform(-0.5, 0.5)
    if case['kind'] == 'render':
        I = -500.0 * torch.log1p(-torch.rand(n, generator=g, device='cuda'))
    else:
        I = uniform(500.0, 1500.0)
    fid = torch.arange(case['fovs'], device='cuda', dtype=torch.int32).repeat_interleave(case['n'])
    return x, y, z, I, fid, g


def _camera_counts(case, x, y, z, I, fid, g):
    """Photon counts of those emitters (whole photons at their pixels, blurred) plus 10
    background photons, Poisson distributed: what the fit is given."""
    F, nw, nh = case['fovs'], case['nw'], case['nh']
    px = x.long().clamp(max=nw - 1)
    py = y.long().clamp(max=nh - 1)
    amp = (I.double() * torch.exp(-z.double().abs() / 0.377)).round().long()
    counts = torch.zeros(F * nw * nh, dtype=torch.int64, device='cuda')
    counts.index_add_(0, (fid.long() * nw + px) * nh + py, amp)
    image = counts.double().view(F, nw, nh)
    R = case['radius']
    for axis in (1, 2):
        size = image.shape[axis]
        out = torch.zeros_like(image)
        for s in range(-R, R + 1):
            k = math.exp(-0.5 * (s / case['sigma']) ** 2) / (math.sqrt(2 * math.pi) * case['sigma'])
            if abs(s) < size:
                out.narrow(axis, max(s, 0), size - abs(s)).add_(
                    image.narrow(axis, max(-s, 0), size - abs(s)), alpha=k)
        image = out
    return torch.poisson((image + 10.0).float(), generator=g).reshape(-1).contiguous()


def _fit_inputs(case, seed):
    x, y, z, I, fid, g = _gauss_inputs(case, seed)
    k = _camera_counts(case, x, y, z, I, fid, g)
    x = x + 0.3 * torch.randn(x.shape, generator=g, device='cuda')
    y = y + 0.3 * torch.randn(y.shape, generator=g, device='cuda')
    return x, y, z, I, fid, k


def _walk_arguments(case):
    args = {'N': [case['n'] // case['states']] * case['states'], 'ndim': case['ndim'],
            'lower': [-15e-6] * case['ndim'], 'upper': [15e-6] * case['ndim'],
            'D': [0.1e-12 * (s + 1) for s in range(case['states'])],
            'periodic': case['periodic']}
    if case['states'] > 1:
        rates = numpy.full((case['states'],) * 2, 0.5)
        numpy.fill_diagonal(rates, 0.0)
        args['transmat'] = rates
    return numpy.arange(case['t']) * 0.033, args


def prepare(case, seed):
    kind = case['kind']
    state = {'case': case}
    if kind == 'frame':
        angle = None if case['dims'] == 2 else 0.0
        config = _config(case, (case['nw'], case['nh']), 0.033, angle=angle)
        state['sim'] = scopyon_amd.create_simulator(
            config, method='default', rng=numpy.random.RandomState((seed + 1) % (1 << 32)))
        state['inputs'] = _frame_inputs(case, seed)
    elif kind == 'movie':
        config = _config(case, (case['nw'], case['nh']), 0.033, bleach=True)
        rng = numpy.random.RandomState(seed % (1 << 32))
        points, inputs = _frame_inputs(case, seed), []
        for k in range(case['frames']):
            rows = numpy.column_stack([points, numpy.arange(case['n']), numpy.ones(case['n'])])
            inputs.append((0.033 * k, rows))
            points = points + rng.normal(0.0, math.sqrt(2 * 0.1e-12 * 0.033), points.shape)
        state['inputs'] = inputs
        state['sim'] = scopyon_amd.create_simulator(config, method='default',
                                                    rng=scopyon_amd.PhiloxRNG(seed))
    elif kind == 'walk':
        state['rng'] = (scopyon_amd.PhiloxRNG(seed) if case['rng'] == 'philox'
                        else numpy.random.RandomState(seed % (1 << 32)))
        state['t'], state['args'] = _walk_arguments(case)
    elif kind == 'batch':
        sizes, counts = _layout(case)
        state['sim'] = BatchedSimulator(_config(case, sizes[0], 0.033), sizes, counts, D=0.1e-12,
                                        dt=0.033, seed=seed)
        if case['graph']:
            state['sim'].capture()
    elif kind == 'depth':
        rng = numpy.random.Generator(numpy.random.Philox(seed + 1))
        D = numpy.exp(rng.normal(math.log(0.5e-12), 1.0, case['n']))
        pl = 16.0e-6 / case['mag']
        size = (case['nw'], case['nh'])
        sim = BatchedSimulator(_config(case, size, 0.01, angle=0.0), [size], case['n'], D=D,
                               dt=0.01, seed=seed, box=(0.8 * size[0] * pl, 0.8 * size[1] * pl),
                               depth_range=(-case['depth'], case['depth']), psf=case['psf'])
        sim.set_positions(*_depth_positions(case, seed))
        if case['psf'] == 'lut':
            sim.capture()
        state['sim'] = sim
    else:
        model = GaussianModel([(case['nw'], case['nh'])] * case['fovs'], sigma=case['sigma'],
                              radius=case['radius'], inv_depth=1.0 / 0.377, background=10.0)
        state['model'] = model
        if kind == 'render':
            x, y, _, I, fid, _ = _gauss_inputs(case, seed)
            state['emitters'] = (x, y, None, I, fid if case['fovs'] > 1 else None)
        else:
            x, y, z, I, fid, k = _fit_inputs(case, seed)
            state['emitters'] = (x, y, z, I, fid)
            state['k'] = k
            if case['auto']:
                state['sigma'] = torch.tensor(case['sigma'], device='cuda')
                state['leaves'] = [t.requires_grad_() for t in (x, y, z, I, state['sigma'])]
            else:
                state['grad_mu'] = torch.empty(model.n_pix, dtype=torch.float32, device='cuda')
                state['outputs'] = [torch.empty_like(x) for _ in range(4)]
    return state


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'frame':
        if not case['full']:
            return [state['sim'].form_image(state['inputs']).as_array()]
        image, info = state['sim'].form_image(state['inputs'], full_output=True)
        return [image.as_array(), info['expectation']]
    if kind == 'movie':
        return [image.as_array() for image in
                state['sim'].generate_images(state['inputs'], case['frames'])]
    if kind == 'walk':
        return scopyon_amd.sample(state['t'], rng=state['rng'], **state['args'])
    if kind == 'depth' and case['psf'] == 'table':
        state['sim'].form()
        return [state['sim'].photons]
    if kind in ('batch', 'depth'):
        sim = state['sim']
        sim.replay()
        return [sim.adc, sim.u, sim.v, sim.depth]
    model = state['model']
    x, y, z, I, fid = state['emitters']
    if kind == 'render':
        return [model.forward(x, y, z, I, fid, method=case['method'])]
    if not case['auto']:
        loss = model.forward_nll(x, y, z, I, state['k'], fid, grad_mu=state['grad_mu'])
        grads = model.backward(x, y, z, I, state['grad_mu'], fid, outputs=state['outputs'])
        return [loss, *grads]
    for t in state['leaves']:
        t.grad = None
    losses = poisson_nll(model, render(model, x, y, z, I, state['sigma'], fid), state['k'])
    losses.sum().backward()
    return [losses.detach(), *(t.grad for t in state['leaves'])]


def work(case):
    """Every emitter read once, every output written once, and a multiply-add per emitter and
    footprint pixel (the contraction's two factors for the Gaussian model)."""
    kind = case['kind']
    if kind in ('frame', 'movie', 'batch', 'depth'):
        foot = (2.0e-6 / (16.0e-6 / case['mag']) + 1) ** 2
        if kind == 'batch':
            sizes, counts = _layout(case)
            n, pixels = float(counts.sum()), float(sum(a * b for a, b in sizes))
        else:
            n, pixels = float(case['n']), float(case['nw'] * case['nh'])
        frames = case['frames'] if kind == 'movie' else 1
        per = {'batch': 32.0, 'depth': 56.0}.get(kind, 40.0)
        out = 8.0 if kind in ('frame', 'movie') or case.get('psf') == 'table' else 4.0
        return {'bytes': frames * (per * n + out * pixels), 'flops': frames * 2.0 * n * foot}
    if kind == 'walk':
        steps = float(case['n']) * case['t'] * case['ndim']
        return {'bytes': 16.0 * steps, 'flops': 2.0 * steps}
    n, pixels = float(case['n']) * case['fovs'], float(case['nw'] * case['nh']) * case['fovs']
    window = (2 * case['radius'] + 1) ** 2
    if kind == 'render':
        return {'bytes': 12.0 * n + 4.0 * pixels, 'flops': 2.0 * n * window}
    return {'bytes': 40.0 * n + 4.0 * pixels, 'flops': 12.0 * n * window}


# ---- the same outputs in 64 bits ----

HC, AVOGADRO = 6.62607015e-34 * 299792458.0, 6.02214076e23
NM = 1.0e-9


def _photon_scale(exposure, angle):
    """Photons per unit of the normalised emission for an emitter at the coverslip, and the
    penetration depth: the defaults of the configuration."""
    flux, wave, QY, absorb, radius = 400000.0, 532.0e-9, 0.61, 83400.0, 20.0e-9
    amplitude, depth = flux / (HC / wave), math.inf
    n1, n2 = 1.46, 1.384
    s2, c2, r2 = math.sin(angle) ** 2, math.cos(angle) ** 2, (n2 / n1) ** 2
    if s2 / r2 >= 1:
        d = r2 ** 2 * c2 + s2 - r2
        amplitude *= (4 * c2 * (s2 - r2) / d + 4 * c2 * s2 / d + 4 * c2 / (1 - r2)) / 2
        depth = wave / (4.0 * math.pi * math.sqrt(n1 ** 2 * s2 - n2 ** 2))
    x_sec = math.log(10) * absorb * 0.1 / AVOGADRO
    A = absorb * 0.1 / AVOGADRO / (4.0 / 3.0 * math.pi * radius ** 3) * 2.0 * radius
    photons = QY * amplitude * x_sec * exposure * (1.0 - 10.0 ** -A)
    return 13564.06122650865 * photons / (4.0 * math.pi), depth


def _summed_kernel(depth):
    """Summed-area table of the Born-Wolf profile (NA 1.4, 578 nm) on 1 nm cells."""
    k = 2.0 * math.pi / 578.0e-9
    nr = 1000
    r = torch.arange(nr, dtype=torch.float64, device='cuda') * NM
    rho = torch.arange(1, 101, dtype=torch.float64, device='cuda') / 100
    J0 = torch.special.bessel_j0((r * (k * 1.4))[:, None] * rho)
    phase = 2.0 * depth * (k * 0.49) * rho * rho
    prof = (((torch.cos(phase) * rho * 0.01) * J0).sum(1) ** 2
            + ((torch.sin(phase) * rho * 0.01) * J0).sum(1) ** 2) * (k * 1.4) ** 2 / math.pi
    c = torch.arange(-(nr - 1), nr, dtype=torch.float64, device='cuda')
    R = torch.sqrt(c[:, None] ** 2 + c ** 2).clamp(max=nr - 1)
    lo = R.floor().long().clamp(max=nr - 2)
    table = prof[lo] + (R - lo) * (prof[lo + 1] - prof[lo])
    S = torch.zeros(2 * nr, 2 * nr, dtype=torch.float64, device='cuda')
    S[1:, 1:] = table.cumsum(0).cumsum(1)
    return S


def _noise_free(nw, nh, mag, depth, u, v, exposure, angle):
    """Photons per pixel, the reference's model: the kernel of each emitter's 1 nm depth key
    summed over the cells of each pixel."""
    depth, u, v = (torch.as_tensor(a, dtype=torch.float64, device='cuda') for a in (depth, u, v))
    pl, cells = 16.0e-6 / mag, 1999
    scale, penetration = _photon_scale(exposure, angle)
    weight = scale * torch.exp(-depth.abs() / penetration) * NM * NM
    keys = torch.where(depth.abs() < 1.0e-6 + NM, (depth.abs() / NM).long(),
                       torch.full_like(depth, 1000).long())
    m = int(math.ceil(1998 * NM / pl)) + 2
    image = torch.zeros(nw * nh, dtype=torch.float64, device='cuda')
    order = torch.argsort(keys)
    sizes = torch.unique_consecutive(keys[order], return_counts=True)
    at = 0
    for key, count in zip(*(t.tolist() for t in sizes)):
        S = _summed_kernel(key * NM)
        mine = order[at:at + count]
        at += count
        for part in mine.split(200000):
            axes = []
            for coord, size in ((u[part], nw), (v[part], nh)):
                o = size * pl * 0.5 + coord - NM * 1998 * 0.5
                first = torch.floor(o / pl)
                idx = first[:, None] + torch.arange(m + 1, dtype=torch.float64, device='cuda')
                edge = torch.ceil((idx * pl - o[:, None]) / NM).clamp(0, cells).long()
                axes.append((idx[:, :-1].long(), edge))
            (i, a), (j, b) = axes
            C = S[a[:, :, None], b[:, None, :]]
            p = C[:, 1:, 1:] - C[:, :-1, 1:] - C[:, 1:, :-1] + C[:, :-1, :-1]
            ok = ((i >= 0) & (i < nw))[:, :, None] & ((j >= 0) & (j < nh))[:, None, :]
            pix = (i[:, :, None] * nh + j[:, None, :]).clamp(0, nw * nh - 1)
            image.index_add_(0, pix.reshape(-1), (p * weight[part, None, None] * ok).reshape(-1))
    return image


def _pixel_factors(c, sigma, R):
    """G, dG/dc and dG/dsigma of the window pixels around c, float64."""
    first = torch.floor(c) - R
    e0 = first[:, None] + torch.arange(2 * R + 1, dtype=torch.float64, device='cuda') - c[:, None]
    e1 = e0 + 1.0
    s = 1.0 / (math.sqrt(2.0) * sigma)
    G = torch.where(e0 >= 0, torch.erfc(e0 * s) - torch.erfc(e1 * s),
                    torch.where(e1 <= 0, torch.erfc(-e1 * s) - torch.erfc(-e0 * s),
                                torch.erf(e1 * s) - torch.erf(e0 * s))) / 2
    norm = 1.0 / (math.sqrt(2 * math.pi) * sigma)
    p0, p1 = norm * torch.exp(-0.5 * (e0 / sigma) ** 2), norm * torch.exp(-0.5 * (e1 / sigma) ** 2)
    return first.long(), (G, p0 - p1, (e0 * p0 - e1 * p1) / sigma)


def _window(case, part, x, y, fid):
    """Pixel indices of each emitter's window, whether they lie in the frame, and the factors."""
    nw, nh, W = case['nw'], case['nh'], 2 * case['radius'] + 1
    sigma = float(numpy.float32(case['sigma']))
    fx, U = _pixel_factors(x[part], sigma, case['radius'])
    fy, V = _pixel_factors(y[part], sigma, case['radius'])
    k = torch.arange(W, device='cuda')
    i, j = fx[:, None] + k, fy[:, None] + k
    ok = ((i >= 0) & (i < nw))[:, :, None] & ((j >= 0) & (j < nh))[:, None, :]
    frame = fid[part].long() if fid is not None else torch.zeros_like(fx)
    pix = ((frame[:, None, None] * nw + i.clamp(0, nw - 1)[:, :, None]) * nh
           + j.clamp(0, nh - 1)[:, None, :])
    return pix, ok, U, V


def _gauss_exact(case, seed):
    if case['kind'] == 'render':
        x, y, _, I, fid, _ = _gauss_inputs(case, seed)
        z, k = None, None
    else:
        x, y, z, I, fid, k = _fit_inputs(case, seed)
    x, y, I = x.double(), y.double(), I.double()
    inv_depth = float(numpy.float32(1.0 / 0.377))
    fade = torch.ones_like(I) if z is None else torch.exp(-z.double().abs() * inv_depth)
    mu = torch.full((case['fovs'] * case['nw'] * case['nh'],), 10.0, dtype=torch.float64,
                    device='cuda')
    parts = torch.arange(x.numel(), device='cuda').split(100000)
    for part in parts:
        pix, ok, U, V = _window(case, part, x, y, fid)
        add = (I * fade)[part, None, None] * U[0][:, :, None] * V[0][:, None, :] * ok
        mu.index_add_(0, pix.reshape(-1), add.reshape(-1))
    if case['kind'] == 'render':
        return [mu]
    k = k.double()
    losses = (mu - k * torch.log(mu)).view(case['fovs'], -1).sum(1)
    dmu = 1.0 - k / mu
    grads, gsigma = [[], [], [], []], torch.zeros((), dtype=torch.float64, device='cuda')
    for part in parts:
        pix, ok, U, V = _window(case, part, x, y, fid)
        g = dmu[pix] * ok

        def total(a, b):
            return (a[:, :, None] * g * b[:, None, :]).sum((1, 2))

        S, f, amp = total(U[0], V[0]), fade[part], (I * fade)[part]
        grads[0].append(amp * total(U[1], V[0]))
        grads[1].append(amp * total(U[0], V[1]))
        grads[2].append(-torch.sign(z[part].double()) * inv_depth * amp * S)
        grads[3].append(f * S)
        gsigma += (amp * (total(U[2], V[0]) + total(U[0], V[2]))).sum()
    gsigma = gsigma if case['auto'] else gsigma.reshape(1)
    return [losses, *(torch.cat(g) for g in grads), gsigma]


def _walk_exact(case, seed):
    t, args = _walk_arguments(case)
    rng = numpy.random.RandomState(seed % (1 << 32))
    n, ndim = args['N'][0], case['ndim']
    x = numpy.stack([rng.uniform(-15e-6, 15e-6, n) for _ in range(ndim)], axis=1)
    out = []
    for k in range(len(t)):
        if k:
            x = x + math.sqrt(2 * 0.1e-12 * (t[k] - t[k - 1])) * rng.standard_normal((n, ndim))
            if case['periodic']:
                x = (x + 15e-6) % 30e-6 - 15e-6
        out.append(numpy.column_stack([x, numpy.zeros(n), numpy.arange(n)]))
    return out


def exact(case, seed):
    kind = case['kind']
    if kind in ('render', 'fit'):
        return _gauss_exact(case, seed)
    if kind == 'walk' and case['rng'] == 'state' and case['states'] == 1:
        return _walk_exact(case, seed)
    if kind == 'frame' and case['full']:
        p = _frame_inputs(case, seed)
        angle = 1.2566370614359172 if case['dims'] == 2 else 0.0
        depth = p[:, 2] if case['dims'] == 3 else numpy.zeros(len(p))
        photons = _noise_free(case['nw'], case['nh'], case['mag'], depth, p[:, 0], p[:, 1], 0.033,
                              angle)
        return [None, (0.92 * (photons + 0.01)).view(case['nw'], case['nh'])]
    if kind == 'depth' and case['psf'] == 'table':
        depth, u, v = _depth_positions(case, seed)
        return [_noise_free(case['nw'], case['nh'], case['mag'], depth, u, v, 0.01, 0.0)]
    return None
