"""Nu_new of planes of 576 x 576 and 384 x 384 collocation points (their own z assembly and product layout) against
the oracle, over the levels per block: one, a remainder, the default, all of them."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(384, 13), (384, 34), (256, 13), (256, 34)])
def test_assembly_of_large_planes_matches_oracle(require_gpu, nx, ny):
    from littleharsh_amd.initial import laminar_plus_noise
    from littleharsh_amd.solver import Channel
    from oracle.oracle import Oracle
    s = make_setup(nx=nx, nz=nx, ny_total=ny, dsty=3, re=180.0, posth=0.15, dyq=4.0, ntilex=6, ntilez=6, dstx=3,
                   dstz=4)
    st = laminar_plus_noise(s, seed=5)
    g, o = Channel(s), Oracle(s)
    g.set_state(*st)
    o.set_state(*st)
    o.nonlinear(1)
    ref = o.get_nonlinear()
    first = g.get_launch()
    for lc in (first["zasm_lc"], 1, 5, 64):
        g.set_launch(first["xraw_lc"], lc, first["col_bs"])
        print(f"case nx={nx} ny={ny} levels per block {lc}", flush=True)
        g.nonlinear(1)
        # the bound: 2 x 576-point transforms each way and a difference over one cell, some 1e3 roundings
        # of values up to the cell count times the result's
        for a, b in zip(g.get_nonlinear(), ref):
            assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
    g.close()
