"""GPU PSF tables vs the oracle: radial profiles and SAT pixel sums."""
import numpy
import pytest
import torch

from oracle import epifm as O

pytestmark = pytest.mark.gpu


def _tables(gpu, wl=5.780000000000062e-07, kind='TRITC', width=None, pl=1.6e-7):
    from scopyon_amd._psf import PSFTables
    return PSFTables('Gaussian' if kind == 'Gaussian' else kind, wl, 1000e-9, 1000e-9,
                     width, pl, gpu)


@pytest.mark.parametrize('depth_nm', [0, 1, 137, 500, 999])
def test_born_wolf_radial_matches_oracle(gpu, depth_nm):
    t = _tables(gpu)
    key = depth_nm
    t.ensure([key])
    r = O.radial_grid(1000e-9)
    ref = O.born_wolf_radial(r, key * 1e-9, 5.780000000000062e-07)
    got = t.radial_last[0].cpu().numpy()
    # float64 with independent j0/sincos: absolute agreement relative to the peak
    assert numpy.abs(got - ref).max() <= 1e-12 * ref.max()


def test_gaussian_radial_matches_oracle(gpu):
    t = _tables(gpu, kind='Gaussian', width=1.0e-7)
    t.ensure([0])
    r = O.radial_grid(1000e-9)
    ref = O.gaussian_radial(r, 1.0e-7)
    got = t.radial_last[0].cpu().numpy()
    numpy.testing.assert_allclose(got, ref, rtol=1e-14, atol=1e-300)


@pytest.mark.parametrize('period,pl', [(66, 6.639004149377593e-08), (160, 1.6e-7)])
def test_sat_pixel_sums_match_bruteforce(gpu, period, pl):
    from scopyon_amd import _lib
    t = _tables(gpu, pl=pl)
    assert t.period == period and t.use_phase == (period == 160)
    t.ensure([0])
    r = O.radial_grid(1000e-9)
    prof = t.radial_last[0].cpu().numpy()
    table = O.radial_to_cartesian(r, prof)          # oracle cartesian table from the GPU profile
    sat = t.sat[t.slot_of[0]].cpu().numpy()
    lib = _lib.lib()
    rng = numpy.random.RandomState(0)
    side = t.ntab + 1
    for _ in range(200):
        a0, a1 = sorted(rng.randint(0, side, 2))
        b0, b1 = sorted(rng.randint(0, side, 2))
        S = lambda a, b: sat[lib.smx_sat_index_host(side, period, int(a), int(b))]
        got = S(a1, b1) - S(a0, b1) - S(a1, b0) + S(a0, b0)
        ref = table[a0:a1, b0:b1].sum()
        assert abs(got - ref) <= 1e-12 * table.sum() + 1e-13 * abs(ref)


@pytest.mark.parametrize('nr,nz,period', [(2, 1, 1), (3, 2, 5), (33, 1, 7), (65, 3, 1), (129, 5, 160),
                                          (500, 2, 9000), (1000, 66, 66), (1025, 2, 160),
                                          (2048, 2, 267), (2049, 1, 160)])
def test_sat_build_sizes(gpu, nr, nz, period):
    """Corner prefix sums for narrow and wide tables, one to many depths (both
    segment heights, depth groups with a remainder), layouts padded beyond the
    row and beyond LDS, and the widest table of the blocked form and the first
    beyond it.  Bound: each corner is a sum of at most ntab^2 positive cells
    in some order, each partial sum rounded once and at most ~2 ntab + 64 of
    them on any path, so 2e-12 of the corner covers ntab = 4097."""
    from scopyon_amd import _device, _lib
    lib = _lib.lib()
    rng = numpy.random.RandomState(nr + nz)
    prof = numpy.exp(-numpy.linspace(0.0, 3.0, nr)) * rng.uniform(0.5, 1.5, (nz, nr))
    ntab = 2 * nr - 1
    elems = int(lib.smx_psf_sat_elems(nr, period))
    dprof = _device.upload(prof, device=gpu)
    ws = torch.empty(int(lib.smx_psf_sat_workspace_bytes(nr, nz)), dtype=torch.uint8, device=gpu)
    sat = torch.full((nz, elems), numpy.nan, dtype=torch.float64, device=gpu)
    _lib.call('smx_psf_sat_build', dprof.data_ptr(), nz, nr, 1e-9, period, ws.data_ptr(),
              sat.data_ptr(), _device.stream())
    place = numpy.array([lib.smx_sat_index_host(ntab + 1, period, 0, b) for b in range(ntab + 1)])
    rows = numpy.array([lib.smx_sat_index_host(ntab + 1, period, a, 0) for a in range(ntab + 1)])
    for z in {0, nz - 1, nz // 2}:
        table = O.radial_to_cartesian(numpy.arange(nr) * 1e-9, prof[z])
        ref = numpy.zeros((ntab + 1, ntab + 1))
        ref[1:, 1:] = table.cumsum(axis=0).cumsum(axis=1)
        got = sat[z].cpu().numpy()[rows[:, None] + place[None, :]]
        numpy.testing.assert_allclose(got, ref, rtol=2e-12, atol=0)


@pytest.mark.parametrize('nr', [33, 1000])
@pytest.mark.parametrize('layout', ['plain', 'sorted'])
def test_sat_bits_do_not_depend_on_the_batch(gpu, nr, layout):
    """A depth's table built alone and among any others is the same bits."""
    from scopyon_amd import _device, _lib
    lib = _lib.lib()
    rng = numpy.random.RandomState(nr)
    nz = 67
    prof = _device.upload(rng.uniform(0.1, 1.0, (nz, nr)), device=gpu)
    if layout == 'plain':
        elems = int(lib.smx_psf_sat_elems(nr, 1))
    else:
        elems = int(lib.smx_psf_sat_sorted_elems(nr))
        places = numpy.empty(2 * nr, dtype=numpy.int32)
        _lib.call('smx_sat_sorted_places', nr, 6.639, places.ctypes.data)
        places = _device.upload(places, dtype=torch.int32, device=gpu)

    def build(first, count):
        ws = torch.empty(int(lib.smx_psf_sat_workspace_bytes(nr, count)), dtype=torch.uint8,
                         device=gpu)
        sat = torch.empty((count, elems), dtype=torch.float64, device=gpu)
        args = (prof[first].data_ptr(), count, nr, 1e-9)
        if layout == 'plain':
            _lib.call('smx_psf_sat_build', *args, 1, ws.data_ptr(), sat.data_ptr(),
                      _device.stream())
        else:
            _lib.call('smx_psf_sat_build_sorted', *args, places.data_ptr(), ws.data_ptr(),
                      sat.data_ptr(), _device.stream())
        return sat

    alone = torch.cat([build(z, 1) for z in range(nz)])
    assert alone.isfinite().all() and alone.any(dim=1).all()
    for count in (2, 4, 5, 16, 66, 67):
        assert torch.equal(build(0, count), alone[:count])


def test_tables_do_not_depend_on_how_they_were_asked_for(gpu):
    """Depth keys met one after another, and in one call: the same tables, also
    in the copy in the plain layout."""
    from scopyon_amd import _lib
    from scopyon_amd._psf import PSFTables
    keys = [0, 3, 250, 17, 40, 41, 999, -1]
    kw = dict(pixel_length=16e-6 / 241.0, device=gpu)
    one = PSFTables('Alexa 647', 6.6e-7, 4.0e-7, 1.0e-6, **kw)
    for k in keys:
        one.ensure(numpy.array([k]))
    all_ = PSFTables('Alexa 647', 6.6e-7, 4.0e-7, 1.0e-6, **kw)
    all_.ensure(numpy.array(keys))
    assert one.places is not None and set(one.slot_of) == set(all_.slot_of)
    lib, side = _lib.lib(), one.ntab + 1     # the plain layout has places without a corner
    rows = torch.tensor([lib.smx_sat_index_host(side, one.period, a, 0) for a in range(side)])
    cols = torch.tensor([lib.smx_sat_index_host(side, one.period, 0, b) for b in range(side)])
    corners = (rows[:, None] + cols).to(gpu)
    for k in one.slot_of:
        a, b = one.slot_of[k], all_.slot_of[k]
        assert torch.equal(one._sat[a], all_._sat[b])
        assert torch.equal(one.sat[a][corners], all_.sat[b][corners])
