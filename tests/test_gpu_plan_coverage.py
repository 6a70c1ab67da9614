"""The kernels that only mixed-precision channels, and FP64 channels with one short and one long
length, still run: the canopy stage from job tables (k_zinv, k_xpass_ib and k_zfwd in FP64), the
one-thread-per-column velocity sweeps, the FP32 x pass, and the alternative x plans of all of them.
Mixed precision solves for the velocities in FP64, so that from an uploaded state and nonlinear term
they are held to the FP64 oracle at 1e-10; the FP32 nonlinear term to the bound that its rounding has
against the same oracle at production size."""
import numpy as np
import pytest

from littleharsh_amd import capi
from littleharsh_amd.channel import make_setup, random_instance
from littleharsh_amd.initial import laminar_plus_noise
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-10
TOL32 = 3e-5          # relative, max norm: FP32 transforms and products (test_gpu_mixed.py)


def rel(a, b):
    den = np.abs(b).max()
    return np.abs(a - b).max() / (den if den > 0 else 1.0)


def channel(nx, nz, ny=33):
    return make_setup(nx=nx, nz=nz, ny_total=ny, dsty=4, re=180.0, alp=1.0, bet=2.0, mpgx=-1.0, posth=0.2, dyq=4.0,
                      ntilex=4, ntilez=4, dstx=3, dstz=4)


# every length up to 144 in x and in z, with both plans
@pytest.mark.parametrize("plans", [(0, 0), (1, 1)], ids=["plan0", "plan1"])
@pytest.mark.parametrize("nx,nz", [(32, 96), (48, 32), (64, 48), (96, 64)])
def test_mixed_solve_and_nonlinear_against_oracle(require_gpu, nx, nz, plans):
    from littleharsh_amd.solver import Channel
    s = channel(nx, nz)
    st = laminar_plus_noise(s, seed=11)
    g, o, on = Channel(s, precision=capi.LH_PREC_MIXED), Oracle(s), Oracle(s)
    print(f"{s.px}x{s.nyv}x{s.pz} plans {plans}", flush=True)
    g.set_plans(*plans)
    for x in (g, o, on):
        x.set_state(*st)
    # the nonlinear term in FP32
    g.nonlinear(2)
    on.nonlinear(2)
    nu = on.get_nonlinear()
    e32 = [rel(a, b) for a, b in zip(g.get_nonlinear(), nu)]
    # canopy, velocities and pressure in FP64, from the oracle's term (as Nu_old too)
    g.set_nonlinear(*nu)
    o.set_nonlinear(*nu)
    g.solve_u(2, 2e-4)
    o.substep_vel(2, 2e-4)
    e64 = [rel(a, b) for a, b in zip(g.get_state(), o.get_state())]
    g.solve_p(2, 2e-4)
    o.substep_pres(2, 2e-4)
    e64 += [rel(a, b) for a, b in zip(g.get_state(), o.get_state())]
    print("Nu", " ".join(f"{e:.1e}" for e in e32), "| u v w p", " ".join(f"{e:.1e}" for e in e64), flush=True)
    assert max(e32) < TOL32
    assert max(e64) < TOL


# a short x and a long z: the canopy x pass by value, on both plans
@pytest.mark.parametrize("xplan", [0, 1])
@pytest.mark.parametrize("nx", [32, 48, 64, 96])
def test_short_x_long_z_matches_oracle(require_gpu, nx, xplan):
    from littleharsh_amd.solver import Channel
    s = channel(nx, 256, 25)
    st = laminar_plus_noise(s, seed=13)
    g, o = Channel(s), Oracle(s)
    print(f"{s.px}x{s.nyv}x{s.pz} x plan {xplan}", flush=True)
    g.set_plans(xplan, 0)
    g.set_state(*st)
    o.set_state(*st)
    dt = g.cfl_dt(0.4)
    g.step(dt)
    o.step(dt)
    errs = [rel(a, b) for a, b in zip(g.get_state(), o.get_state())]
    print(" ".join(f"{e:.1e}" for e in errs), flush=True)
    assert max(errs) < TOL


def test_batch_of_both_precisions(require_gpu):
    """FP64 and mixed members of several lengths and both plans: the FP64 members' whole planes beside
    the mixed members' passes, column kernels of every kind beside each other; each member
    bit-identical to its single steps."""
    from littleharsh_amd.solver import Batch, Channel
    members = [(random_instance(0), False, 0), (random_instance(1), True, 1), (random_instance(3), True, 0),
               (channel(32, 32), False, 1), (channel(48, 48), True, 1), (random_instance(11), False, 0),
               (channel(256, 256, 17), True, 0), (channel(96, 64, 21), True, 1)]
    chans, refs = [], []
    for i, (s, mixed, plan) in enumerate(members):
        st = laminar_plus_noise(s, seed=150 + i)
        pair = [Channel(s, precision=capi.LH_PREC_MIXED if mixed else capi.LH_PREC_FP64) for _ in range(2)]
        for x in pair:
            n = x.get_plans()
            x.set_plans(min(plan, n["xcount"] - 1), min(plan, n["zcount"] - 1))
            x.set_state(*st)
        chans.append(pair[0])
        refs.append(pair[1])
    b = Batch(chans)
    for _ in range(2):
        b.step_cfl(0.5)
        for r in refs:
            r.step_cfl(0.5)
    for i, (c, r) in enumerate(zip(chans, refs)):
        for x, y in zip(c.get_state(), r.get_state()):
            assert np.array_equal(x, y), i
    b.close()
