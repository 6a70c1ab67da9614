"""Nu_new against the oracle over the x lengths whose lines share a wavefront (and 384, one line per
wavefront): row pairs that leave the last wavefront partly empty, and every kind of level chunk."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(32, 48), (48, 32), (64, 96), (96, 32), (96, 64), (256, 48)])
def test_x_pass_matches_oracle(require_gpu, nx, nz):
    from littleharsh_amd.initial import laminar_plus_noise
    from littleharsh_amd.solver import Channel
    from oracle.oracle import Oracle
    s = make_setup(nx=nx, nz=nz, ny_total=34, dsty=5, re=180.0, posth=0.15, dyq=4.0, ntilex=4, ntilez=4, dstx=3,
                   dstz=4)
    st = laminar_plus_noise(s, seed=5)
    g, o = Channel(s), Oracle(s)
    g.set_state(*st)
    o.set_state(*st)
    o.nonlinear(1)
    ref, dt = o.get_nonlinear(), None
    first = g.get_launch()
    for lc in (first["xraw_lc"], 1, 5, 64):
        g.set_launch(lc, first["zasm_lc"], first["col_bs"])
        print(f"case nx={nx} nz={nz} levels per wave {lc}", flush=True)
        g.nonlinear(1)
        # some 1e3 roundings of values up to the cell count times the result's
        for a, b in zip(g.get_nonlinear(), ref):
            assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
        # the CFL maximum does not depend on how the levels are shared out
        d = g.cfl_dt(0.5)
        assert dt is None or d == dt
        dt = d
    g.close()
