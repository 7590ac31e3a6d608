"""End-to-end parity: scopyon_amd.form_image / generate_images vs the oracle
on the same inputs and the same RandomState stream."""
import numpy
import pytest

from oracle import epifm as O
from conftest import oracle_params, product_config, PRE

pytestmark = pytest.mark.gpu


def _oracle_frames(overrides, inputs, seed, nframes=None, exposure=None):
    rng = numpy.random.RandomState(seed)
    p = oracle_params(overrides, rng)
    data = list(O.format_inputs(inputs, PRE))
    psf = O.PSFCache(p)
    if nframes is None:
        return [O.output_frame(p, psf, data, rng=rng, exposure_time=exposure)]
    return list(O.generate_frames(p, psf, data, nframes, rng=rng, exposure_time=exposure))


@pytest.mark.parametrize('mag,shape,n', [(100.0, (48, 48), 30), (241.0, (40, 56), 25)])
def test_form_image_matches_oracle(gpu, mag, shape, n):
    import scopyon_amd
    ov = {'detector': {'image_size': list(shape), 'exposure_time': 0.033}, 'magnification': mag}
    pl = 16e-6 / mag
    rng = numpy.random.RandomState(42)
    inputs = rng.uniform(-0.5 * shape[0] * pl, 0.5 * shape[0] * pl, size=(n, 2))
    img, info = scopyon_amd.form_image(inputs, config=product_config(ov),
                                       rng=numpy.random.RandomState(5), full_output=True)
    (cam, oinfo), = _oracle_frames(ov, inputs, 5)
    numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-10, atol=0)
    assert numpy.array_equal(img.as_array(), cam[:, :, 1])
    assert sorted(info['true_data']) == sorted(oinfo['true_data'])
    for m in oinfo['true_data']:
        numpy.testing.assert_allclose(info['true_data'][m], oinfo['true_data'][m], rtol=1e-12)


def test_form_image_3d_inputs(gpu):
    import scopyon_amd
    ov = {'detector': {'image_size': [32, 32], 'exposure_time': 0.05}, 'magnification': 241.0,
          'light_source': {'angle': 0.0}}
    rng = numpy.random.RandomState(3)
    pl = 16e-6 / 241.0
    inputs = numpy.column_stack([rng.uniform(-16 * pl, 16 * pl, (12, 2)),
                                 rng.uniform(-6e-7, 6e-7, 12)])
    # 3-column input -> (depth = z, u = x, v = y) through the unit vectors
    img, info = scopyon_amd.form_image(inputs, config=product_config(ov),
                                       rng=numpy.random.RandomState(1), full_output=True)
    (cam, _), = _oracle_frames(ov, inputs, 1)
    numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-10)
    assert numpy.array_equal(img.as_array(), cam[:, :, 1])


def test_generate_images_bleaching_matches_oracle(gpu):
    import scopyon_amd
    from oracle import sampling as S
    ov = {'detector': {'image_size': [32, 32], 'exposure_time': 0.033}, 'magnification': 100.0,
          'effects': {'photo_bleaching': {'switch': True, 'half_life': 0.05}}}
    pl = 16e-6 / 100.0
    dt = 0.033
    t = numpy.arange(0, 7) * dt / 2          # two sub-steps per frame
    inputs = S.sample_inputs(t, N=20, lower=-14 * pl, upper=14 * pl, ndim=2, D=0.1e-12,
                             rng=numpy.random.RandomState(2))
    frames = list(scopyon_amd.generate_images(inputs, 3, config=product_config(ov),
                                              rng=numpy.random.RandomState(9), full_output=True))
    ref = _oracle_frames(ov, inputs, 9, nframes=3)
    for (img, info), (cam, oinfo) in zip(frames, ref):
        numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-10)
        assert numpy.array_equal(img.as_array(), cam[:, :, 1])
        st, ost = info['fluorescence_states'], oinfo['fluorescence_states']
        assert sorted(st) == sorted(ost)
        for m in ost:
            assert st[m] == pytest.approx(ost[m], rel=1e-12, abs=0)


def test_bleaching_with_molecules_coming_and_going(gpu):
    """Molecule sets that stay, shrink, come back in another order and grow over
    the sub-steps: budgets are drawn in order of first sight and follow the ids."""
    import scopyon_amd
    ov = {'detector': {'image_size': [24, 24], 'exposure_time': 0.033}, 'magnification': 100.0,
          'effects': {'photo_bleaching': {'switch': True, 'half_life': 0.03}}}
    pl = 16e-6 / 100.0
    rng = numpy.random.RandomState(4)
    xy = rng.uniform(-10 * pl, 10 * pl, (30, 2))
    sets = [range(12), range(12), [3, 1, 7], [7, 3, 1], [29, 1, 5], list(range(30)),
            list(range(30))[::-1], range(12)]
    inputs = [(0.011 * k, numpy.column_stack([xy[list(ids)], list(ids), numpy.ones(len(ids))]))
              for k, ids in enumerate(sets)]
    frames = list(scopyon_amd.generate_images(inputs, 2, config=product_config(ov),
                                              rng=numpy.random.RandomState(6), full_output=True))
    for (img, info), (cam, oinfo) in zip(frames, _oracle_frames(ov, inputs, 6, nframes=2)):
        numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-10)
        assert numpy.array_equal(img.as_array(), cam[:, :, 1])
        st, ost = info['fluorescence_states'], oinfo['fluorescence_states']
        assert list(st) == list(ost)
        for m in ost:
            assert st[m] == pytest.approx(ost[m], rel=1e-12, abs=0)
        for m in oinfo['true_data']:
            numpy.testing.assert_allclose(info['true_data'][m], oinfo['true_data'][m], rtol=1e-12)
    bad = numpy.column_stack([xy, numpy.full(30, numpy.nan), numpy.ones(30)])
    with pytest.raises(ValueError):
        list(scopyon_amd.generate_images([(0.0, bad)], 1, config=product_config(ov),
                                         rng=numpy.random.RandomState(6)))


def test_form_image_errors(gpu):
    import scopyon_amd
    cfg = product_config({'detector': {'image_size': [8, 8]}})
    with pytest.raises(ValueError):
        scopyon_amd.form_image(numpy.zeros((3, 6)), config=cfg, rng=numpy.random.RandomState(0))
    with pytest.raises(ValueError):
        scopyon_amd.form_image(numpy.zeros(3), config=cfg, rng=numpy.random.RandomState(0))
    with pytest.raises(TypeError):
        scopyon_amd.form_image(3.0, config=cfg, rng=numpy.random.RandomState(0))


def _cmos_table():
    import os
    import scopyon_amd
    path = os.path.join(os.path.dirname(scopyon_amd.__file__), 'catalog', 'detector',
                        'RNDist_F40.csv')
    return numpy.loadtxt(path, delimiter=',')


@pytest.mark.parametrize('kind', ['CCD', 'CMOS'])
def test_ccd_and_cmos_match_oracle(gpu, kind):
    """CCD / CMOS detectors (_epifm.py:329-353, 418-433, 1443-1469): same ADC
    counts as the oracle for the same RandomState stream."""
    import scopyon_amd
    ov = {'detector': {'type': kind, 'image_size': [40, 36], 'exposure_time': 0.033},
          'magnification': 100.0}
    pl = 16e-6 / 100.0
    rng = numpy.random.RandomState(9)
    inputs = rng.uniform(-18 * pl, 18 * pl, size=(20, 2))
    img, info = scopyon_amd.form_image(inputs, config=product_config(ov),
                                       rng=numpy.random.RandomState(8), full_output=True)
    orng = numpy.random.RandomState(8)
    p = oracle_params(ov, orng)
    data = list(O.format_inputs(inputs, PRE))
    cam, _ = O.output_frame(p, O.PSFCache(p), data, rng=orng,
                            cmos_table=_cmos_table() if kind == 'CMOS' else None)
    numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-10, atol=0)
    assert numpy.array_equal(img.as_array(), cam[:, :, 1])


@pytest.mark.parametrize('kind', ['CCD', 'CMOS'])
def test_ccd_and_cmos_philox_moments(gpu, kind):
    """Philox CCD / CMOS: photo-electrons Poisson(E) plus readout noise
    (normal of the configured sigma, or the CMOS table's distribution):
    mean and variance of the ADC counts with gain 1."""
    import torch
    from scopyon_amd import _lib, _device
    n = 512 * 512
    det = _lib.DetectorParamsT()
    det.qe, det.background, det.background_switch, det.emgain = 1.0, 0.0, 0, 1
    det.readout_noise = 3.0 if kind == 'CCD' else 0.0
    det.fullwell, det.adc_max, det.offset, det.gain = 1e300, 1e300, 100.0, 1.0
    if kind == 'CMOS':
        t = _cmos_table()
        p = t[:, 1] / t[:, 1].sum()
        cdf = p.cumsum()
        cdf /= cdf[-1]
        tv, tc = (torch.as_tensor(a, dtype=torch.float64, device=gpu) for a in (t[:, 0], cdf))
        nmean, nvar = float((t[:, 0] * p).sum()), float((t[:, 0] ** 2 * p).sum() - ((t[:, 0] * p).sum()) ** 2)
        targs = (tv.data_ptr(), tc.data_ptr(), len(cdf))
    else:
        nmean, nvar = 0.0, 9.0
        targs = (None, None, 0)
    for E in (0.3, 5.0, 40.0):
        photons = torch.full((n,), E, dtype=torch.float64, device=gpu)
        adc = torch.empty(n, dtype=torch.float32, device=gpu)
        _lib.call('smx_photon_detector_philox', n, photons.data_ptr(), None, None, det, *targs,
                  77, 1, 0, None, None, adc.data_ptr(), 1, _device.stream())
        x = adc.cpu().numpy().astype(float) - 100.0
        var = E + nvar
        assert abs(x.mean() - (E + nmean)) < 5 * numpy.sqrt(var / n), (kind, E, x.mean())
        assert abs(x.var() / var - 1.0) < 0.03, (kind, E, x.var(), var)


def test_filter_switches_follow_the_reference(gpu):
    """_epifm.py:1308-1313: an emission filter switched on without a type
    zeroes every weight (background only, same frame as the oracle); a
    dichroic mirror switched on with a catalog type raises TypeError."""
    import scopyon_amd
    pl = 16e-6 / 100.0
    inputs = numpy.random.RandomState(2).uniform(-10 * pl, 10 * pl, size=(15, 2))
    ov = {'detector': {'image_size': [24, 24], 'exposure_time': 0.033}, 'magnification': 100.0,
          'emission_filter': {'switch': True}}
    img, info = scopyon_amd.form_image(inputs, config=product_config(ov),
                                       rng=numpy.random.RandomState(4), full_output=True)
    (cam, _), = _oracle_frames(ov, inputs, 4)
    assert numpy.array_equal(img.as_array(), cam[:, :, 1])
    numpy.testing.assert_allclose(info['expectation'], cam[:, :, 0], rtol=1e-12)
    assert numpy.allclose(cam[:, :, 0], cam[0, 0, 0])
    ov = {'detector': {'image_size': [24, 24], 'exposure_time': 0.033}, 'magnification': 100.0,
          'dichroic_mirror': {'switch': True}}
    with pytest.raises(TypeError):
        scopyon_amd.form_image(inputs, config=product_config(ov), rng=numpy.random.RandomState(4))
    with pytest.raises(TypeError):
        _oracle_frames(ov, inputs, 4)


def test_reference_example_images(gpu):
    """The drop-in path run exactly as the reference's examples/tirf.py and
    examples/twocolor.py (same calls, same RandomState(123)) reproduces their
    committed output images (tests/golden/*_u8.npz, from examples/*.png) on
    the background-only pixels: > 99% equal after the 8-bit rescale, all
    within one grey level.  (Pixels under emitters depend on the uniforms
    and noise of each pixel as well as its expectation; their brightness is
    pinned through the oracle, whose expectation this path equals to 1e-10,
    in test_oracle_png.test_tirf_png_emitter_brightness.)"""
    import os
    import scopyon_amd
    from test_oracle_png import GOLDEN, _background_agreement

    def agree(img, info, png):
        return _background_agreement(info['expectation'], img.as_array(), png)

    config = scopyon_amd.DefaultConfiguration()
    config.default.detector.exposure_time = 33.0e-3
    pl = config.default.detector.pixel_length / config.default.magnification
    L_2 = config.default.detector.image_size[0] * pl * 0.5
    rng = numpy.random.RandomState(123)
    inputs = rng.uniform(-L_2, +L_2, size=(100, 2))
    img, info = scopyon_amd.form_image(inputs, config=config, rng=rng, full_output=True)
    exact, worst, n_bg = agree(img, info, numpy.load(os.path.join(GOLDEN, 'tirf_000_u8.npz'))['image'])
    assert n_bg > 150_000 and exact > 0.99 and worst <= 1, (exact, worst, n_bg)

    config = scopyon_amd.DefaultConfiguration()
    rng = numpy.random.RandomState(123)
    inputs = rng.uniform(-L_2, +L_2, size=(250, 2))
    png = numpy.load(os.path.join(GOLDEN, 'twocolor_000_u8.npz'))['image']
    for ch, part in enumerate((inputs[: 200], inputs[150:])):
        img, info = scopyon_amd.form_image(part, config=config, rng=rng, full_output=True)
        exact, worst, n_bg = agree(img, info, png[:, :, ch])
        assert n_bg > 100_000 and exact > 0.99 and worst <= 1, (ch, exact, worst, n_bg)


def test_uploads_are_complete_for_other_streams(gpu):
    """What an object keeps on the device is there for work on any stream when the
    upload returns, however busy the stream it was made on; staged copies are
    ordered on the caller's stream, in every type, small and large."""
    import torch
    from scopyon_amd import _device
    side = torch.cuda.Stream()
    a = numpy.random.RandomState(1).uniform(1.0, 2.0, 4000)
    for _ in range(3):
        with torch.cuda.stream(side):
            torch.cuda._sleep(50000000)
            up = _device.upload(a)
        seen = up.clone()            # on the default stream
        torch.cuda.synchronize()
        assert numpy.array_equal(seen.cpu().numpy(), a)
        side.synchronize()
    for n in (0, 1, 4000, 100000):
        for dtype in (torch.float64, torch.int32, torch.int64):
            want = (numpy.arange(n) * 1.5).astype(numpy.float64)
            with torch.cuda.stream(side):
                torch.cuda._sleep(5000000)
                twice = _device.stage(want, dtype=dtype, device=gpu) * 2
                got = twice.cpu()
            assert torch.equal(got, torch.as_tensor(want).to(dtype) * 2)


@pytest.mark.parametrize('detector', ['EMCCD', 'CCD', 'CMOS'])
@pytest.mark.parametrize('kind', ['state', 'plain', 'philox'])
def test_failing_frame_leaves_the_generator(gpu, detector, kind):
    """A splat that reports an overflow, and a bad molecule id with ground truth,
    raise with the generator as it was, also one whose state cannot be put back."""
    import scopyon_amd
    from scopyon_amd import _epifm
    ov = {'detector': {'type': detector, 'image_size': [24, 20], 'exposure_time': 0.033},
          'magnification': 100.0}
    sim = _epifm._EPIFMSimulator(_epifm.EPIFMConfigs(product_config(ov).default,
                                                     rng=numpy.random.RandomState(0)))
    source = numpy.random.RandomState(5)

    class Plain:    # no state to read
        def __getattr__(self, name):
            if name in ('normal', 'random_sample', 'poisson', 'standard_normal'):
                return getattr(source, name)
            raise AttributeError(name)

    rng = {'state': source, 'plain': Plain(), 'philox': scopyon_amd.PhiloxRNG(5)}[kind]
    rows = numpy.column_stack([numpy.zeros(9), numpy.linspace(-1e-6, 1e-6, 9), numpy.zeros(9),
                               numpy.arange(9), numpy.ones(9)])

    def states():
        return [x.tolist() if hasattr(x, 'tolist') else x for x in source.get_state()]

    good, _ = sim.output_frame([(0.0, rows)], rng=rng)
    before, frame = states(), sim._philox_frame
    splat = sim.splatter.splat

    def overflowing(*args, **kwargs):
        splat(*args, **kwargs)
        sim.splatter.status |= 2

    sim.splatter.splat = overflowing
    for full in (False, True):
        with pytest.raises(RuntimeError, match='capacity'):
            sim.output_frame([(0.0, rows)], rng=rng, full_output=full)
        assert states() == before and sim._philox_frame == frame
    sim.splatter.splat = splat
    bad = rows.copy()
    bad[4, 3] = numpy.nan
    with pytest.raises(ValueError):
        sim.output_frame([(0.0, bad)], rng=rng, full_output=True)
    assert states() == before and sim._philox_frame == frame
    again, _ = sim.output_frame([(0.0, rows)], rng=rng)
    assert not numpy.array_equal(again[:, :, 1], good[:, :, 1])
    if kind != 'philox':
        assert states() != before
    else:
        assert sim._philox_frame == frame + 1


def test_readout_noise_that_is_not_a_number(gpu):
    """An EMCCD readout noise of NaN is drawn like any other (numpy gives NaN), so
    that it shows in the counts; the generator advances as for a number."""
    import scopyon_amd
    frames, ends = [], []
    for noise in (100.0, numpy.nan):
        ov = {'detector': {'type': 'EMCCD', 'image_size': [16, 16], 'readout_noise': noise,
                           'exposure_time': 0.033}, 'magnification': 100.0}
        rng = numpy.random.RandomState(3)
        frames.append(scopyon_amd.form_image(numpy.zeros((1, 2)), config=product_config(ov),
                                             rng=rng).as_array())
        ends.append(rng.random_sample())
    assert numpy.isfinite(frames[0]).all() and ends[0] == ends[1]
    assert not numpy.array_equal(*frames)
