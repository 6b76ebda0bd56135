"""get_state() forms the virtual state on the device: against the oracle's
get_state where the affine map has fewer address bits than qubits, is
permuted and shifted, and where the output takes more than one chunk (22
bits) of the device buffer."""
import subprocess
import sys

import numpy as np
import pytest

import oracle_py as O
from conftest import ROOT
from zxh_adae_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,hs,eager", [(1, 0, False), (3, 1, False), (9, 9, True), (16, 5, False), (18, 5, False), (19, 6, False), (21, 20, False),
                                        (22, 3, False), (23, 4, False), (24, 6, False), (23, 2, True)])
def test_get_state(gpu_engine, n, hs, eager, prec):
    """hs qubits in superposition, then X, CX, Rz and Z gates (the rows mix,
    the offsets and the global phase are set); the other amplitudes are zero."""
    r = W.SplitMix64(90 + n)
    gates = [(W.U3, 0, r.below(n), r.uniform() * 3, r.uniform(), r.uniform()) for _ in range(hs)]
    for _ in range(3 * n):
        q = r.below(n)
        gates.append((W.X, 0, q, 0, 0, 0) if r.uniform() < 0.3 else (W.RZ, 0, q, r.uniform(), 0, 0))
        if n > 1:
            gates.append((W.CX, (q + 1 + r.below(n - 1)) % n, q, 0, 0, 0))
    o = O.OracleSim(n, False, eager)
    o.gates(gates)
    o.execute()
    want = o.get_state()
    s = gpu_engine.ZXH(n, False, eager, precision=prec)
    s.gates(gates)
    s.execute()
    got = s.get_state_array()
    # complex64: a few roundings of 6e-8 on amplitudes of at most 1
    assert np.max(np.abs(got - want)) < (1e-12 if prec == "c128" else 2e-6)
    assert np.array_equal(got == 0, want == 0)


WRITER = """
import torch
import numpy as np
import zxh_adae_amd as Z
from zxh_adae_amd import workloads as W
torch.cuda.init()
Z.init()
s = Z.ZXH(18, False, True)
s.gates(W.random_layers(18, 1, 3))
s.execute()
ptr, m = s.device_state()
class Memory:
    __cuda_array_interface__ = {"shape": (2 << m,), "typestr": "<f8", "data": (ptr, False), "version": 2}
psi = torch.as_tensor(Memory(), device="cuda")
before = s.get_state_array()
a = torch.ones(4096, 4096, device="cuda")
torch.cuda.synchronize()
for _ in range(100):  # some tens of milliseconds on the default stream, then the write
    a = torch.tanh(a @ a)
psi.neg_()
got = s.get_state_array()
torch.cuda.synchronize()
assert np.array_equal(got, -before)
print("ordered", flush=True)
"""


def test_get_state_after_the_default_stream():
    """get_state() sees what torch's default stream was given before it, on
    memory taken from device_state(): a process of its own, since torch has to
    be imported first for one HIP runtime."""
    r = subprocess.run([sys.executable, "-c", WRITER], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "ordered" in r.stdout, r.stderr[-2000:]
