"""The canopy forcing of whole planes (transform lengths up to 144) against the oracle: every length in
x and in z, square and uneven planes, tip planes and the ones below, through whole substeps."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(32, 32), (32, 96), (48, 64), (64, 48), (64, 64), (48, 96), (96, 48), (96, 96)])
def test_canopy_planes_match_oracle(require_gpu, nx, nz):
    from littleharsh_amd.initial import laminar_plus_noise
    from littleharsh_amd.solver import Channel
    from oracle.oracle import Oracle
    s = make_setup(nx=nx, nz=nz, ny_total=33, dsty=5, re=180.0, posth=0.15, dyq=4.0, ntilex=4, ntilez=2, dstx=3,
                   dstz=5)
    st = laminar_plus_noise(s, seed=11)
    g, o = Channel(s), Oracle(s)
    g.set_state(*st)
    o.set_state(*st)
    print(f"case nx={nx} nz={nz}", flush=True)
    for k in (1, 2, 3):
        g.substep(k, 2e-4)
        o.substep(k, 2e-4)
    for a, b in zip(g.get_state(), o.get_state()):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()
    g.close()
