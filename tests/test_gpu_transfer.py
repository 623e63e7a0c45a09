"""Populations, masks and fields between the device and halo-padded host
arrays: sizes of one transfer slot and of several, rows that cross a slot's
end, fields small enough to be written straight to the host."""
import numpy as np
import pytest

from dlbc_amd.lattice import _padded_shape


@pytest.fixture(scope="module")
def D():
    import dlbc_amd
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    return dlbc_amd


@pytest.mark.gpu
@pytest.mark.parametrize("dq,n", [((3, 19), (70, 61, 67)), ((3, 19), (5, 4, 6)),
                                  ((2, 9), (601, 523)), ((2, 9), (9, 17)), ((1, 3), (70001,)),
                                  ((1, 5), (40,))], ids=str)
@pytest.mark.parametrize("halo", [0, 1, 3])
def test_round_trip(D, dq, n, halo):
    d, q = dq
    rng = np.random.default_rng(7)
    inner = tuple(slice(halo, halo + v) for v in n)
    lat = D.Lattice(d, q, 2, n)
    lat.set_params([1.0, 1.0])
    mask = np.full(_padded_shape(n, halo), 7, np.int32)  # halo values are not looked at
    mask[inner] = rng.random(n) < 0.2
    lat.upload_mask(mask, halo=halo)
    assert np.array_equal(lat.mask(halo)[inner], mask[inner])
    pops = [rng.random(_padded_shape(n, halo) + (q,)) for _ in range(2)]
    for f in range(2):
        lat.upload_population(f, pops[f], halo=halo)
    for f in range(2):
        back = lat.population(f, halo)
        assert np.array_equal(back[inner], pops[f][inner])
        back[inner] = 0.0
        assert not back.any()  # the halo is left alone
        rho = lat.density(f)
        np.testing.assert_allclose(rho, pops[f][inner].sum(-1), rtol=1e-14)
        padded = np.full(_padded_shape(n, halo), -1.0)
        lat._check(D.lib().dlbc_gpu_density(lat.h, f, padded.reshape(-1), halo), "density")
        assert np.array_equal(padded[inner], rho)
        u = np.zeros(_padded_shape(n, halo) + (d,))
        lat._check(D.lib().dlbc_gpu_velocity(lat.h, f, u.reshape(-1), halo), "velocity")
        assert np.array_equal(u[inner], lat.velocity(f))
    colour = lat.colour()
    assert np.array_equal(colour, np.where(mask[inner] != 0, 0.0, lat.density(0) - lat.density(1)))
