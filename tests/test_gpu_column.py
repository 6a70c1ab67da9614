"""The column stage's kernels at the edges of their block shapes, one step each against the oracle
(1e-10 relative, the bound of the other parity tests): levels that are one short of, equal to and
one past a multiple of a thread's levels, channels of a few levels, of more levels than one block
of the widest shape holds, and of more than any holds; both mean-flow modes."""
import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

pytestmark = pytest.mark.gpu

# (nx, nz, planes): 544 columns take 4 levels per thread (up to 256 levels), 2112 columns 9; 300
# levels need the narrower blocks, 619 levels the one-thread sweeps
SHAPES = [(32, 32, 9), (32, 32, 45), (32, 32, 257), (32, 32, 258), (64, 64, 28), (64, 64, 29), (64, 64, 27), (32, 32, 301),
          (32, 32, 620)]


@pytest.mark.parametrize("flag", [1, 0])
@pytest.mark.parametrize("nx,nz,ny", SHAPES)
def test_column_shapes_match_oracle(require_gpu, nx, nz, ny, flag):
    from littleharsh_amd.initial import laminar_plus_noise
    from littleharsh_amd.solver import Channel
    from oracle.oracle import Oracle
    s = make_setup(nx=nx, nz=nz, ny_total=ny, dsty=2 if ny < 20 else 5, re=180.0, posth=0.15, dyq=4.0, ntilex=4,
                   ntilez=4, dstx=3, dstz=4, flag_ctpress=flag, qxt=120.0)
    st = laminar_plus_noise(s, seed=6)
    g, o = Channel(s), Oracle(s)
    g.set_state(*st)
    o.set_state(*st)
    print(f"case {nx}x{ny}x{nz} flag {flag}", flush=True)
    g.step(2e-5)
    o.step(2e-5)
    for a, b in zip(g.get_state(), o.get_state()):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()
    g.close()
