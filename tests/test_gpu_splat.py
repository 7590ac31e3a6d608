"""GPU weights + splat vs the oracle's overlay loop (same positions)."""
import numpy
import pytest
import torch

from oracle import epifm as O
from conftest import oracle_params, product_config

pytestmark = pytest.mark.gpu


def _oracle_expected(p, particles, unit_time):
    psf = O.PSFCache(p)
    nw, nh = p.image_size
    exp, _, _ = O.molecule_plane(p, psf, particles, (nw, nh), numpy.asarray(p.focal_point),
                                 unit_time, {}, None, None)
    return exp


def _gpu_expected(gpu, overrides, particles, unit_time):
    from scopyon_amd import _epifm
    cfg = product_config(overrides)
    sim = _epifm._EPIFMSimulator(_epifm.EPIFMConfigs(cfg.default, rng=numpy.random.RandomState(0)))
    nw, nh = sim.configs.detector_image_size
    camera = torch.zeros(nw * nh, dtype=torch.float64, device=gpu)
    sim._substep(particles, unit_time, camera, None, None, {}, False)
    _epifm._status_check(sim.splatter.status)
    return camera.cpu().numpy().reshape(nw, nh)


def _particles(rng, n, half, depth=None):
    xy = rng.uniform(-half, half, size=(n, 2))
    d = numpy.zeros(n) if depth is None else depth
    return numpy.column_stack([d, xy, numpy.arange(n), numpy.ones(n)])


CASES = [
    # (overrides, n, half-extent factor, depth spread [m])
    ({'detector': {'image_size': [64, 64]}, 'magnification': 100.0}, 40, 0.6, None),
    ({'detector': {'image_size': [48, 80]}, 'magnification': 241.0}, 30, 0.7, None),
    ({'detector': {'image_size': [40, 40]}, 'magnification': 100.0}, 25, 1.2, None),  # edges/outside
    ({'detector': {'image_size': [32, 48]}, 'magnification': 241.0}, 12, 0.6, 1.5e-6),  # 3D keys
    ({'detector': {'image_size': [33, 17]}, 'magnification': 60.0}, 10, 0.8, 2e-7),
]


@pytest.mark.parametrize('case', range(len(CASES)))
def test_splat_matches_oracle(gpu, case):
    ov, n, f, dz = CASES[case]
    rng = numpy.random.RandomState(100 + case)
    p = oracle_params(ov)
    pl = p.pixel_length / p.magnification
    half = f * 0.5 * max(p.image_size) * pl
    depth = None if dz is None else rng.uniform(-dz, dz, n)
    parts = _particles(rng, n, half, depth)
    ref = _oracle_expected(p, parts, 0.033)
    got = _gpu_expected(gpu, ov, parts, 0.033)
    scale = ref.max()
    assert scale > 0
    numpy.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-13 * scale)


def test_splat_gaussian_psf(gpu):
    ov = {'detector': {'image_size': [40, 40]}, 'magnification': 100.0,
          'fluorophore': {'type': 'Gaussian', 'radial_width': 1.5e-7, 'wave_length': 6.0e-7}}
    rng = numpy.random.RandomState(5)
    p = oracle_params(ov)
    parts = _particles(rng, 15, 0.5 * 40 * 1.6e-7)
    ref = _oracle_expected(p, parts, 0.05)
    got = _gpu_expected(gpu, ov, parts, 0.05)
    numpy.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-13 * ref.max())


def test_splat_empty_and_zero_weight(gpu):
    ov = {'detector': {'image_size': [32, 32]}, 'magnification': 100.0}
    parts = numpy.array([[0.0, 0.0, 0.0, 0, 0.0],        # p_state 0 -> weight 0, skipped
                         [0.0, 1e-3, 1e-3, 1, 1.0]])     # far outside the frame
    got = _gpu_expected(gpu, ov, parts, 0.033)
    assert not got.any()
    got = _gpu_expected(gpu, ov, numpy.zeros((0, 5)), 0.033)
    assert not got.any()


def test_splat_deterministic(gpu):
    ov = {'detector': {'image_size': [64, 64]}, 'magnification': 100.0}
    rng = numpy.random.RandomState(9)
    parts = _particles(rng, 400, 0.5 * 64 * 1.6e-7)
    a = _gpu_expected(gpu, ov, parts, 0.033)
    b = _gpu_expected(gpu, ov, parts, 0.033)
    assert numpy.array_equal(a, b)


@pytest.mark.parametrize('mag,shape,n,spread', [(241.0, (70, 45), 300, 0.6), (60.0, (33, 64), 40, 1.3),
                                                (150.0, (16, 200), 1500, 0.55),
                                                (23.7, (31, 31), 1, 0.1)])
def test_sorted_tables_equal_plain_layout(gpu, mag, shape, n, spread):
    """Pixels that are not whole cells: the splat from sorted tables (any number
    of entries per tile, footprints across frame and quadrant edges) gives the
    bits of the splat from the plain layout, added to what the image holds."""
    from scopyon_amd import _device, _epifm, _lib
    cfg = product_config({'detector': {'image_size': list(shape)}, 'magnification': mag})
    sim = _epifm._EPIFMSimulator(_epifm.EPIFMConfigs(cfg.default, rng=numpy.random.RandomState(0)))
    t = sim.tables
    assert t.places is not None
    rng = numpy.random.RandomState(int(mag))
    t.ensure(numpy.array([0, 3, 250, -1]))
    half = 0.5 * numpy.array(shape) * 16e-6 / mag
    u = _device.upload(rng.uniform(-1, 1, n) * 2 * spread * half[0], device=gpu)
    v = _device.upload(rng.uniform(-1, 1, n) * 2 * spread * half[1], device=gpu)
    w = _device.upload(rng.uniform(0.0, 50.0, n), device=gpu)
    key = _device.upload(rng.randint(0, 4, n), dtype=torch.int32, device=gpu)
    start = _device.upload(rng.uniform(0.0, 1.0, shape), device=gpu)
    got = start.clone()
    sim.splatter.splat(u, v, w, key, sim.fovs_dev, 1, sim.geom.n_tiles, got)
    ref = start.clone()
    cap = n * _epifm.tiles_per_emitter(sim.configs.pixel_length, t.ntab)
    ws = torch.empty(_lib.lib().smx_splat_workspace_bytes(n, sim.geom.n_tiles, cap),
                     dtype=torch.uint8, device=gpu)
    _lib.call('smx_splat_expected', n, u.data_ptr(), v.data_ptr(), w.data_ptr(), key.data_ptr(),
              None, sim.fovs_dev.data_ptr(), 1, sim.geom.n_tiles, t.sat.data_ptr(), t.sat_elems, 4,
              t.ntab, t.period, 1e-9, 1e-18, cap, 1, None, 0, t.m, ref.data_ptr(), ws.data_ptr(),
              ws.numel(), sim.splatter.status.data_ptr(), _device.stream())
    assert int(sim.splatter.status.item()) == 0
    assert not torch.equal(got, start)
    assert torch.equal(got, ref)
    with pytest.raises(ValueError):      # no detector epilogue on the general path
        _lib.call('smx_splat_detect_ts', n, u.data_ptr(), v.data_ptr(), w.data_ptr(),
                  key.data_ptr(), None, sim.fovs_dev.data_ptr(), 1, sim.geom.n_tiles,
                  *t.splat_tables()[:2], 4, t.ntab, t.period, 1e-9, 1e-18, cap, 0,
                  *t.splat_tables()[2:], t.m, None, ws.data_ptr(), ws.numel(),
                  sim.splatter.status.data_ptr(), _device.stream(), None, None, sim.det, 0, 0, 0,
                  None, None, got.data_ptr(), 0, 32)


@pytest.mark.parametrize('nr', [11600, 33000])
def test_splat_from_wide_tables(gpu, nr):
    """Tables of more than 2^29 corners (4 GB) and of more than 2^32, whose
    offsets need 64 bits: 23 and 66 um across on 66.4 cells a pixel.  Corner
    (a, b) holds f(a) f(b) with whole f, so every pixel integral is an exact whole
    number, and the frame lies at the table's last corner or its first."""
    from scopyon_amd import _device, _epifm, _lib
    side, ntab = 2 * nr, 2 * nr - 1
    pl, shape = 66.39e-9, (40, 33)
    period = 66
    lib = _lib.lib()
    f = numpy.arange(side) + numpy.arange(side) % 7
    place = numpy.arange(side) % period * (-(-side // period)) + numpy.arange(side) // period
    for a in (0, 1, 65, 66, side - 1):
        assert lib.smx_sat_index_host(side, period, 0, a) == place[a]
    width = period * -(-side // period)
    assert int(lib.smx_psf_sat_elems(nr, period)) == width * width
    axis = numpy.zeros(width)
    axis[place] = f
    axis = torch.as_tensor(axis, device=gpu)
    table = torch.empty((width, width), dtype=torch.float64, device=gpu)
    for rows in range(0, width, 1024):
        torch.outer(axis[rows:rows + 1024], axis, out=table[rows:rows + 1024])
    geom = _epifm.FrameGeometry(*shape, pl, 0.0, 0.0)
    fovs = torch.from_numpy(numpy.frombuffer(bytes(geom.fov), dtype=numpy.uint8).copy()).to(gpu)
    half, res = 1e-9 * (ntab - 1) * 0.5, 1e-9
    # centres that put the frame at the end of the footprint, at its start, and
    # once across its last corner
    at = numpy.array([[-half + 15 * pl, -half + 12 * pl], [half - 14.3 * pl, half - 11.6 * pl],
                      [-half + 1.7 * pl, half - 3.2 * pl]])
    n = len(at)
    u, v = (_device.upload(at[:, k], device=gpu) for k in (0, 1))
    w = torch.tensor([1.0, 2.0, 4.0], dtype=torch.float64, device=gpu)
    key = torch.zeros(n, dtype=torch.int32, device=gpu)
    cap = n * geom.n_tiles
    ws = torch.empty(lib.smx_splat_workspace_bytes(n, geom.n_tiles, cap), dtype=torch.uint8,
                     device=gpu)
    status = torch.zeros(1, dtype=torch.int32, device=gpu)
    out = torch.empty(shape, dtype=torch.float64, device=gpu)
    _lib.call('smx_splat_expected', n, u.data_ptr(), v.data_ptr(), w.data_ptr(), key.data_ptr(),
              None, fovs.data_ptr(), 1, geom.n_tiles, table.data_ptr(), table.numel(), 1, ntab,
              period, res, 1.0, cap, 0, None, 0, 0, out.data_ptr(), ws.data_ptr(), ws.numel(),
              status.data_ptr(), _device.stream())
    got = out.cpu().numpy()
    del table
    torch.cuda.empty_cache()
    assert int(status.item()) == 0
    want = numpy.zeros(shape)
    for (x, y), weight in zip(at, (1.0, 2.0, 4.0)):
        sums = []
        for c, size in ((x, shape[0]), (y, shape[1])):
            o = size * pl * 0.5 + c - half
            # the footprint's pixels, and its table cells cut at their edges
            # (_epifm.py:241-263)
            k = numpy.arange(size)
            inside = (k >= numpy.floor(o / pl)) & (k < numpy.ceil((size * pl * 0.5 + c + half) / pl))
            edge = numpy.ceil((numpy.arange(size + 1) * pl - o) / res)
            sums.append(inside * numpy.diff(f[numpy.clip(edge, 0, ntab).astype(int)]))
        want += weight * numpy.outer(*sums)
    assert (want > 0).mean() > 0.5
    assert numpy.array_equal(got, want)
