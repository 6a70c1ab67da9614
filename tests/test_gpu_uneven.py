"""Planes whose x and z lengths differ widely (the one-wavefront x pass at 576 collocation points
with short z lines, and the reverse) against the oracle, one step each."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(384, 48), (48, 384)])
def test_uneven_plane_step_matches_oracle(require_gpu, nx, nz):
    from littleharsh_amd.initial import laminar_plus_noise
    from littleharsh_amd.solver import Channel
    from oracle.oracle import Oracle
    s = make_setup(nx=nx, nz=nz, ny_total=33, dsty=5, re=180.0, posth=0.15, dyq=4.0, ntilex=6, ntilez=6, dstx=3,
                   dstz=4)
    st = laminar_plus_noise(s, seed=5)
    g, o = Channel(s), Oracle(s)
    g.set_state(*st)
    o.set_state(*st)
    print(f"case nx={nx} nz={nz}", flush=True)
    g.step(2e-5)
    o.step(2e-5)
    for a, b in zip(g.get_state(), o.get_state()):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()
    g.close()
