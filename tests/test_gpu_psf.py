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
