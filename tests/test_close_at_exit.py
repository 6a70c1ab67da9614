"""Handles left to the interpreter's exit: each is destroyed once, although the modules' globals
may be gone by then (another object's finaliser closes the handle, then its own runs)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# a stub of the library that prints every destroy call, and a global owner that closes its handle
SCRIPT = """
import ctypes, os, sys
import torch
from littleharsh_amd.closure_les import DeviceClosure
from littleharsh_amd.mlp import MLP
from littleharsh_amd.solver import Batch, Channel


class Lib:
    def __getattr__(self, name, write=os.write):
        def call(*args):
            if name.endswith("destroy"):
                write(1, f"{name} {args[0].value}\\n".encode())
            return 0
        return call


class Owner:
    def __init__(self, h):
        self.h = h

    def __del__(self):
        self.h.close()


def handle(cls, lib, attr):
    h = cls.__new__(cls)
    setattr(h, lib, Lib())
    setattr(h, attr, ctypes.c_void_p(1))
    return h


owner = Owner({make})
"""


@pytest.mark.parametrize("make, destroy", [
    ('handle(Channel, "_lib", "_h")', "lh_destroy"),
    ('handle(Batch, "_lib", "_b")', "lh_batch_destroy"),
    ('handle(MLP, "lib", "h")', "lh_mlp_destroy"),
    ('handle(DeviceClosure, "lib", "h")', "lh_closure_destroy"),
], ids=["Channel", "Batch", "MLP", "DeviceClosure"])
def test_a_handle_left_to_exit_is_destroyed_once(make, destroy):
    r = subprocess.run([sys.executable, "-c", SCRIPT.replace("{make}", make)], cwd=ROOT, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert r.stdout.splitlines() == [f"{destroy} 1"], r.stdout + r.stderr


@pytest.mark.parametrize("status, left", [(0, False), (1, True)], ids=["destroyed", "refused"])
def test_a_refused_handle_stays_open(status, left):
    """lh_destroy refuses a member of a batch: the channel then keeps its handle."""
    import ctypes
    from littleharsh_amd.solver import Channel

    class Lib:
        calls = 0

        def lh_destroy(self, h):
            Lib.calls += 1
            return status

    c = Channel.__new__(Channel)
    c._lib, c._h = Lib(), ctypes.c_void_p(1)
    c.close()
    assert (c._h is not None) == left and Lib.calls == 1
    c._h = None
