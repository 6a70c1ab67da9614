"""Transfers from several threads at once, beside channels that are created and closed: every state
comes back as it went."""
import threading

import numpy as np
import pytest

from littleharsh_amd.channel import make_setup

from cases import small, tiny

pytestmark = pytest.mark.gpu


def test_threads_get_their_own_state(require_gpu):
    from littleharsh_amd.solver import Channel
    # 1.4 MB, 6 MB and 44 MB of state: part of a chunk, a few chunks, many
    setups = [tiny(), small(), make_setup(nx=96, nz=96, ny_total=145, dsty=12, re=180.0, alp=1.0, bet=2.0, mpgx=-1.0)]
    errors = []

    def transfers(s, seed):
        try:
            rng = np.random.default_rng(seed)
            ch = Channel(s)
            for _ in range(6):
                st = [rng.standard_normal((s.ncol, n)) + 1j * rng.standard_normal((s.ncol, n))
                      for n in (s.nyu, s.nyv, s.nyu, s.nyp)]
                ch.set_state(*st)
                for a, b in zip(ch.get_state(), st):
                    assert np.array_equal(a, b)
            ch.close()
        except Exception as e:
            errors.append(e)

    def handles():
        try:
            for _ in range(6):
                Channel(setups[0]).close()
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=transfers, args=(s, i)) for i, s in enumerate(setups)]
    threads.append(threading.Thread(target=handles))
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
