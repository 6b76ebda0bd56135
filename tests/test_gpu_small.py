"""Circuits on states that fit one compute unit's LDS (complex128 to 13
address bits, complex64 to 14) run in one launch: against the oracle, at the
edges of that range and of the kernel's step chunks, parameter slots and
windows."""
import numpy as np
import pytest

import oracle_py as O
from zxh_adae_amd import workloads as W

pytestmark = pytest.mark.gpu

# complex128: the engine's 1e-12; complex64: 6e-8 per rounding, a few
# roundings per gate adding as a random walk over at most 3000 gates
TOL = {"c128": 1e-12, "c64": 2e-5}
MODES = {"lazy": (False, False), "plain": (False, True), "nox": (True, True), "nox_lazy": (True, False)}


def check(Z, n, gates, prec, mode):
    dx, eager = MODES[mode]
    o = O.OracleSim(n, dx, eager)
    o.gates(gates)
    o.execute()
    want = o.get_state()
    s = Z.ZXH(n, dx, eager, precision=prec)
    s.gates(gates)
    for _ in range(2):  # the second run starts from a written state
        s.execute()
        assert np.max(np.abs(s.get_state_array() - want)) < TOL[prec], (n, mode)
    return s


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 11, 12, 13, 14])
def test_soups(gpu_engine, n, mode, prec):
    """Every gate kind; 13 is complex128's widest state here and 14
    complex64's, and one more qubit leaves the range."""
    check(gpu_engine, n, W.random_mixed(n, 40 + 20 * n, 700 + n), prec, mode)


@pytest.mark.parametrize("prec,n", [("c128", 13), ("c64", 14)])
def test_no_gates_and_one_gate(gpu_engine, prec, n):
    s = check(gpu_engine, n, [], prec, "plain")
    assert s.get_state_array()[0] == 1 and np.count_nonzero(s.get_state_array()) == 1
    check(gpu_engine, n, [(W.H, 0, n - 1, 0, 0, 0)], prec, "plain")
    check(gpu_engine, n, [(W.CP, 0, n - 1, 0.3, 0, 0)], prec, "plain")


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,layers", [(4, 120), (7, 700), (13, 60)])
def test_many_steps(gpu_engine, n, layers, prec):
    """More steps than one chunk of the kernel's table (112), than one
    parameter slot (about 1000, with the state written and read between the
    runs), and window tables beyond one run's share (32 MiB at 13 bits)."""
    gates = W.random_layers(n, layers, 40 + n)
    if n == 13:
        # windows that do not merge: one gate between each two
        r = W.SplitMix64(9)
        for k in range(300):
            gates += [(W.H, 0, k % n, 0, 0, 0), (W.CP, k % n, (k + 1) % n, r.uniform(), 0, 0)]
    check(gpu_engine, n, gates, prec, "plain")


def test_a_window_larger_than_its_share_of_a_slot(gpu_engine):
    """9000 gates in one window.  Their angles are scaled by 1e-3: the sum of
    a window's angles rounds by half an ulp of the partial sum per gate, and
    with whole angles (partial sums to 14000: 9e-13 each, a random walk of
    9000 of them) that alone passes 1e-12; below 32 they are 1.8e-15 each,
    1.7e-13 in all."""
    n = 6
    window = [g[:3] + (g[3] * 1e-3, 0.0, 0.0) for g in W.diag_batch(n, 9000, 3)]
    check(gpu_engine, n, W.hadamard_all(n) + window + W.hadamard_all(n), "c128", "plain")
