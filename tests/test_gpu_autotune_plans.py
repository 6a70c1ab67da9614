"""The autotuner leaves the x plan alone where no kernel of the channel's step reads it: the trials
of two x plans then time the same code, and a choice between them is noise."""
import pytest

from littleharsh_amd.initial import laminar_plus_noise

from cases import tiny

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ib", [True, False], ids=["canopy", "plain"])
def test_autotune_keeps_an_x_plan_nothing_reads(require_gpu, ib):
    from littleharsh_amd.solver import Channel
    s = tiny(ib=ib)
    g = Channel(s)
    g.set_state(*laminar_plus_noise(s, seed=43))
    for _ in range(3):
        for xplan in (0, 1):
            g.set_plans(xplan, 0)
            p = g.autotune(1)
            print("x plan", xplan, "tuned", p, flush=True)
            assert p["xplan"] == xplan
