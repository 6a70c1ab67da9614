"""Uploads and downloads of state, nonlinear term, forcing and spectra: the same bits come back, for
fields smaller and larger than a transfer chunk (2 MB) and planes that are no multiple of a tile."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,ny", [(32, 32, 9), (48, 32, 66), (64, 96, 97)])
def test_round_trips_keep_every_bit(require_gpu, nx, nz, ny):
    from littleharsh_amd.solver import Channel
    s = make_setup(nx=nx, nz=nz, ny_total=ny, dsty=2 if ny < 20 else 5, re=180.0, posth=0.15, dyq=4.0, ntilex=4,
                   ntilez=4, dstx=3, dstz=4)
    rng = np.random.default_rng(3)
    c = lambda n: rng.standard_normal((s.ncol, n)) + 1j * rng.standard_normal((s.ncol, n))
    st = c(s.nyu), c(s.nyv), c(s.nyu), c(s.nyp)
    st[0][3, 4] = np.nan
    nl = c(s.nyu - 2), c(s.nyv - 2), c(s.nyu - 2)
    ch = Channel(s)
    print(f"case {nx}x{ny}x{nz}", flush=True)
    ch.set_state(*st)
    ch.set_nonlinear(*nl)
    ch.set_forcing(nl[2], None, nl[0])
    for a, b in zip(ch.get_state(), st):
        assert np.array_equal(a, b, equal_nan=True)
    for a, b in zip(ch.get_nonlinear(), nl):
        assert np.array_equal(a, b)
    f = ch.get_forcing()
    assert np.array_equal(f[0], nl[2]) and not np.any(f[1]) and np.array_equal(f[2], nl[0])
    u, v, w, p = c(s.nyu), c(s.nyv), c(s.nyu), c(s.nyp)
    ch.set_state(u, v, w, p)
    ch.spectra_accumulate()
    sp = ch.spectra()
    for q, a in ((0, u), (1, v), (2, w), (4, p)):
        assert np.allclose(sp[q, :, :a.shape[1]], a.real ** 2 + a.imag ** 2, rtol=4e-16, atol=0)
        assert not np.any(sp[q, :, a.shape[1]:])
    ch.close()
