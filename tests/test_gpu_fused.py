"""Splat + EMCCD + ADC in one tile pass (smx_splat_detect_ts) against the two
separate passes (smx_splat_expected_ts, then smx_emccd_philox): the fused
epilogue draws every pixel's numbers from the same Philox stream with the
same code, so ADC counts, expectations and photons are bit-identical, for
tiles of 16, 32 and 64 pixels, uneven frames and several steps."""
import ctypes

import numpy
import pytest
import torch

from conftest import product_config

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64), (48, 80), (128, 128), (16, 16), (200, 72)]
COUNTS = [50, 10, 400, 3, 120]


def _cfg():
    return product_config({'detector': {'image_size': [64, 64], 'exposure_time': 0.033},
                           'magnification': 100.0,
                           'effects': {'photo_bleaching': {'switch': False}}})


def _pair(ts, precision='folded', adc_dtype=torch.float32, keep_photons=True, seed=3, q=16):
    from scopyon_amd.batched import BatchedSimulator
    kw = dict(dt=0.033, seed=seed, table_precision=precision, tile_side=ts, quadrant=q,
              adc_dtype=adc_dtype, keep_expectation=True)
    sep = BatchedSimulator(_cfg(), SHAPES, COUNTS, fuse_detector=False, **kw)
    fus = BatchedSimulator(_cfg(), SHAPES, COUNTS, fuse_detector=True, keep_photons=keep_photons,
                           **kw)
    assert not sep.fused and fus.fused
    return sep, fus


def _bits(t):
    a = t.cpu().numpy()
    return a.view(numpy.uint64 if a.dtype == numpy.float64 else numpy.uint32)


@pytest.mark.parametrize('ts,q', [(16, 16), (32, 16), (64, 16), (32, 32), (64, 32)])
@pytest.mark.parametrize('precision', ['folded', 'float64'])
def test_fused_equals_separate_passes(gpu, ts, q, precision):
    print('fused detector: tile side {} quadrant {} table {}'.format(ts, q, precision), flush=True)
    sep, fus = _pair(ts, precision, q=q)
    for sim in (sep, fus):
        sim.photons.fill_(-1.0)
        sim.adc.fill_(-1.0)
        sim.weights()
    sep.splat()
    sep.emccd()
    fus.splat_detect()
    torch.cuda.synchronize()
    assert sep.status() & ~1 == 0 and fus.status() & ~1 == 0
    assert (sep.adc >= 0).all() and sep.photons.max() > 0
    assert numpy.array_equal(_bits(fus.adc), _bits(sep.adc))
    assert numpy.array_equal(_bits(fus.E), _bits(sep.E))
    assert numpy.array_equal(_bits(fus.photons), _bits(sep.photons))


@pytest.mark.parametrize('ts', [16, 32])
def test_fused_steps_and_graph_replay(gpu, ts):
    """Several steps (Brownian move, weights, fused pass, frame counter), the
    fused simulator replayed from a HIP graph, against eager separate steps;
    no photon image is written in the fused steps."""
    print('fused detector: steps, tile side {}'.format(ts), flush=True)
    sep, fus = _pair(ts, keep_photons=False, adc_dtype=torch.float64, seed=7)
    fus.photons.fill_(-2.0)
    fus.capture()                                # one eager step, then the graph
    outs = []
    sep.step()
    outs.append((sep.adc.clone(), fus.adc.clone()))
    for _ in range(3):
        sep.step()
        fus.replay()
        outs.append((sep.adc.clone(), fus.adc.clone()))
    torch.cuda.synchronize()
    for a, b in outs:
        assert numpy.array_equal(_bits(a), _bits(b))
    assert not torch.equal(outs[0][0], outs[1][0])
    assert (fus.photons == -2.0).all()
    assert torch.equal(sep.u, fus.u) and torch.equal(sep.v, fus.v)


def test_fused_with_adc_maps(gpu):
    """Per-pixel gain and offset maps (fixed-pattern noise) through the C-ABI:
    the fused pass reads them like smx_emccd_philox."""
    from scopyon_amd import _device, _lib
    sep, fus = _pair(32, keep_photons=True, seed=13)
    n = sep.n_pix
    rng = numpy.random.RandomState(5)
    gain = torch.as_tensor(rng.uniform(10.0, 14.0, n), device='cuda')
    offset = torch.as_tensor(numpy.rint(rng.normal(2000.0, 30.0, n)), device='cuda')
    sep.weights()
    sep.splat()
    adc_a = torch.zeros(n, dtype=torch.float32, device='cuda')
    _lib.call('smx_emccd_philox', n, sep.photons.data_ptr(), gain.data_ptr(), offset.data_ptr(),
              sep.det, 99, 4, 0, None, None, adc_a.data_ptr(), 1, _device.stream())
    fus.weights()
    t = fus.tables
    adc_b = torch.zeros(n, dtype=torch.float32, device='cuda')
    _lib.call('smx_splat_detect_ts', fus.n, fus.u.data_ptr(), fus.v.data_ptr(), fus.w.data_ptr(),
              fus.key.data_ptr(), fus.fov_id.data_ptr(), fus.fovs_dev.data_ptr(), fus.nfov,
              fus.n_tiles, t.sat.data_ptr(), t.sat_elems, len(t.slot_of), t.ntab, t.period, 1e-9,
              1e-18, fus.capacity, 0, _device.ptr(fus.Ktab), fus.k_format, t.m, None,
              fus.ws.data_ptr(), fus.ws.numel(), fus.splatter.status.data_ptr(), _device.stream(),
              gain.data_ptr(), offset.data_ptr(), fus.det, 99, 4, 0, None, None, adc_b.data_ptr(),
              1, 32)
    torch.cuda.synchronize()
    assert numpy.array_equal(_bits(adc_a), _bits(adc_b))


def test_fused_refuses_what_it_cannot_do(gpu):
    from scopyon_amd import _device, _lib
    sep, fus = _pair(32)
    t = fus.tables
    args = [fus.n, fus.u.data_ptr(), fus.v.data_ptr(), fus.w.data_ptr(), fus.key.data_ptr(),
            fus.fov_id.data_ptr(), fus.fovs_dev.data_ptr(), fus.nfov, fus.n_tiles,
            t.sat.data_ptr(), t.sat_elems, len(t.slot_of), t.ntab, t.period, 1e-9, 1e-18,
            fus.capacity]
    tail = [fus.ws.data_ptr(), fus.ws.numel(), fus.splatter.status.data_ptr(), _device.stream(),
            None, None, fus.det, 1, 0, 0, None, None, fus.adc.data_ptr(), 1, 32]
    with pytest.raises(ValueError):       # accumulate = 1
        _lib.call('smx_splat_detect_ts', *args, 1, _device.ptr(fus.Ktab), fus.k_format, t.m,
                  None, *tail)
    with pytest.raises(ValueError):       # no phase table
        _lib.call('smx_splat_detect_ts', *args, 0, None, 0, t.m, None, *tail)


@pytest.mark.parametrize('nfov,n', [(1, 1), (1, 63), (1, 257), (1, 2048), (3, 500), (40, 30)])
@pytest.mark.parametrize('kind', ['folded', 'float64', 'lut'])
def test_self_listed_tiles_equal_binned(gpu, nfov, n, kind):
    """Up to 2048 emitters the tile passes list their emitters themselves; with
    emitters of zero weight appended past that they are binned.  Photons and
    counts are the same bits, for interleaved FOV ids, one and several FOVs,
    split bin / accumulate calls and a second (warm) step."""
    from scopyon_amd import _device, _epifm, _lib
    from scopyon_amd.batched import BatchedSimulator
    ov = {'detector': {'image_size': [64, 64], 'exposure_time': 0.033},
          'magnification': 100.0, 'effects': {'photo_bleaching': {'switch': False}}}
    shapes = [(61 + f % 3, 64 - f % 5) for f in range(nfov)]
    rng = numpy.random.RandomState(n)
    half = 0.5 * 64 * 1.6e-7
    total = n * nfov
    place = rng.uniform(-1.2 * half, 1.2 * half, (2, total))
    fov = rng.permutation(numpy.repeat(numpy.arange(nfov), n))
    frames = []
    for extra in (0, 2100):
        for side in (16, 32):
            sim = BatchedSimulator(product_config(ov), shapes, n + (extra + nfov - 1) // nfov,
                                   dt=0.033, seed=5, tile_side=side, keep_photons=True,
                                   psf='lut' if kind == 'lut' else 'table',
                                   table_precision='folded' if kind == 'lut' else kind,
                                   lut_slices=4, lut_bins=512, lut_phases=8)
            m = sim.n
            pos = numpy.zeros((2, m))
            pos[:, :total] = place
            ids = numpy.zeros(m, dtype=numpy.int32)
            ids[:total] = fov
            sim.fov_id.copy_(torch.as_tensor(ids))
            sim.set_positions(numpy.zeros(m), pos[0], pos[1])
            sim.w[total:] = 0.0
            for step in range(2):
                sim.splat_detect()
                frames.append((sim.photons.clone(), sim.adc.clone()))
            sim.photons.zero_()
            sim.splat('smx_splat_bin')
            sim.splat('smx_splat_accumulate')
            frames.append((sim.photons.clone(), frames[-1][1]))
            assert sim.status() == 0
    assert frames[0][0].abs().sum() > 0
    for photons, adc in frames[1:]:
        assert torch.equal(photons, frames[0][0]) and torch.equal(adc, frames[0][1])


@pytest.mark.parametrize('clustered,spread', [(0, 1.0), (6000, 0.08), (6000, 0.4), (60000, 0.5)])
def test_heavy_tiles_first(gpu, clustered, spread):
    """Launches of 4,096 tiles and more start their heaviest tiles first, as many as
    their list holds (256 of 4,099 here: none are heavy, some, or more than it
    holds); fewer, larger tiles note none.  Photons and counts are the same bits."""
    from scopyon_amd.batched import BatchedSimulator
    ov = {'detector': {'image_size': [64, 64], 'exposure_time': 0.033},
          'magnification': 100.0, 'effects': {'photo_bleaching': {'switch': False}}}
    shapes = [(1024, 1024), (33, 16)]
    rng = numpy.random.RandomState(clustered)
    n = 500 + clustered // 2
    x = rng.uniform(-512, 512, (2, 2 * n)) * 1.6e-7
    x[:, :clustered] *= spread
    fov = numpy.zeros(2 * n, dtype=numpy.int32)
    fov[-100:] = 1
    frames = []
    for side in (16, 32, 64):
        sim = BatchedSimulator(product_config(ov), shapes, n, dt=0.033, seed=5, tile_side=side,
                               keep_photons=True, psf='table', table_precision='folded')
        sim.fov_id.copy_(torch.as_tensor(fov))
        sim.set_positions(numpy.zeros(2 * n), x[0], x[1])
        for step in range(2):
            sim.splat_detect()
            frames.append((sim.photons.clone(), sim.adc.clone()))
        assert sim.status() == 0
    assert frames[0][0].abs().sum() > 0
    for photons, adc in frames[1:]:
        assert torch.equal(photons, frames[0][0]) and torch.equal(adc, frames[0][1])


@pytest.mark.parametrize('nfov,n', [(1, 300), (3, 200), (1, 2100)])
def test_workspace_across_call_forms(gpu, nfov, n):
    """A workspace binned by a call that lists its emitters itself (few of them)
    serves the calls that the interface allows on it: warm calls without phase
    tables or with the other quadrant, and the tile pass with the other quadrant.
    Same bits as each call on a workspace of its own."""
    from scopyon_amd import _device, _lib
    from scopyon_amd.batched import BatchedSimulator
    q32, warm = 0x100, 0x200
    sim = BatchedSimulator(_cfg(), [(61 + f, 64 - f) for f in range(nfov)], n, dt=0.033, seed=2,
                           tile_side=32, table_precision='float64')
    sim.weights()
    t = sim.tables

    def fresh():
        return torch.full_like(sim.ws, 0x55)

    def call(entry, tile, ws, phase=True):
        out = torch.zeros_like(sim.photons)
        _lib.call('smx_splat_{}_ts'.format(entry), sim.n, sim.u.data_ptr(), sim.v.data_ptr(),
                  sim.w.data_ptr(), sim.key.data_ptr(), sim.fov_id.data_ptr(),
                  sim.fovs_dev.data_ptr(), sim.nfov, sim.n_tiles, t.sat.data_ptr(), t.sat_elems,
                  len(t.slot_of), t.ntab, t.period, 1e-9, 1e-18, sim.capacity, 0,
                  _device.ptr(sim.Ktab if phase else None), sim.k_format, t.m, out.data_ptr(),
                  ws.data_ptr(), ws.numel(), sim.splatter.status.data_ptr(), _device.stream(), tile)
        return out

    listed, general = call('expected', 32, fresh()), call('expected', 32, fresh(), phase=False)
    assert listed.abs().sum() > 0
    torch.testing.assert_close(listed, general, rtol=1e-12, atol=0)
    for tile in (32, 32 | q32):
        for then in (32, 32 | q32):
            ws = fresh()
            assert torch.equal(call('expected', tile, ws), listed)
            assert torch.equal(call('accumulate', then, ws), listed)
            assert torch.equal(call('expected', then | warm, ws), listed)
            ws = fresh()
            call('bin', tile, ws)
            assert torch.equal(call('accumulate', then, ws), listed)
            assert torch.equal(call('expected', 32 | warm, ws, phase=False), general)
            assert torch.equal(call('expected', then | warm, ws), listed)
    assert sim.status() == 0


def test_heavy_tiles_of_a_large_frame(gpu):
    """65,536 tiles and more: the counters are scanned by the device scan, and the
    heavy tiles noted beside it, again in a second step.  Same bits as from fewer,
    larger tiles, which one workgroup scans."""
    from scopyon_amd.batched import BatchedSimulator
    n = 20000
    rng = numpy.random.RandomState(1)
    x = rng.uniform(-0.5, 0.5, (2, n)) * numpy.array([[4096], [4112]]) * 1.6e-7
    x[:, :n // 2] *= 0.03
    frames = []
    for side, tiles in ((16, 65792), (32, 16512)):
        sim = BatchedSimulator(_cfg(), [(4096, 4112)], n, dt=0.033, seed=5, tile_side=side,
                               keep_photons=True, table_precision='folded')
        assert sim.n_tiles == tiles
        sim.set_positions(numpy.zeros(n), x[0], x[1])
        for step in range(2):
            sim.splat_detect()
            frames.append((sim.photons.clone(), sim.adc.clone()))
        assert sim.status() == 0
    assert frames[0][0].abs().sum() > 0
    for photons, adc in frames[1:]:
        assert torch.equal(photons, frames[0][0]) and torch.equal(adc, frames[0][1])
