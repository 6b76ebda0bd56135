"""Products of several runs on one qubit, held until they are applied: against
the oracle, where other gates lie between the runs (diagonal gates that
commute with the qubit and that do not, X and CX that change its descriptor
and that do not) and where a run's own product is within 1e-5 of the identity
(the reference skips it, whatever the other runs' products are)."""
import numpy as np
import pytest

import oracle_py as O
from zxh_adae_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(Z, n, gates):
    for eager in (True, False):
        o = O.OracleSim(n, False, eager)
        o.gates(gates)
        o.execute()
        want = o.get_state()
        for prec, tol in (("c128", 1e-12), ("c64", 2e-5)):
            s = Z.ZXH(n, False, eager, precision=prec)
            s.gates(gates)
            s.execute()
            assert np.max(np.abs(s.get_state_array() - want)) < tol, (n, eager, prec)


def u3(q, r):
    return (W.U3, 0, q, r.uniform() * 6, r.uniform() * 6, r.uniform() * 6)


@pytest.mark.parametrize("n", [6, 13, 16])
@pytest.mark.parametrize("seed", range(4))
def test_runs_between_other_gates(gpu_engine, n, seed):
    r = W.SplitMix64(1000 * n + seed)
    gates = W.hadamard_all(n)
    for _ in range(120):
        k = r.below(10)
        q, p = r.below(n), r.below(n - 1)
        p += p >= q
        if k < 5:
            gates += [u3(q, r) for q in [r.below(n) for _ in range(1 + r.below(4))]]
        elif k < 7:
            gates.append((W.CP, p, q, r.uniform(), 0, 0))
        elif k == 7:
            gates.append((W.P, 0, q, r.uniform(), 0, 0))
        elif k == 8:
            gates.append((W.CX, p, q, 0, 0, 0))
        else:
            gates.append((W.X, 0, q, 0, 0, 0))
    check(gpu_engine, n, gates)


@pytest.mark.parametrize("n", [5, 15])
def test_identity_products_of_one_run(gpu_engine, n):
    """On every qubit: a run, a phase elsewhere, a run whose own product is
    the identity to 5e-6, a phase elsewhere, a run that undoes the first to
    5e-6 (not skipped: it is not the identity by itself)."""
    r = W.SplitMix64(n)
    gates = W.hadamard_all(n) + [(W.BARRIER, 0, 0, 0, 0, 0)]
    for q in range(n - 1):
        e = (W.CP, (q + 1) % n, n - 1 if q + 1 < n - 1 else 0, 0.3 + q, 0, 0)
        gates += [(W.U3, 0, q, 0.3, 0, 0), e, (W.U3, 0, q, 0.7, 0, 0), (W.U3, 0, q, -0.7 + 5e-6, 0, 0), e,
                  (W.U3, 0, q, -0.3 + 5e-6, 0, 0)]
    check(gpu_engine, n, gates)


def test_qft_on_a_product_state_takes_as_many_sweeps_as_a_qft(gpu_engine):
    n = 20
    r = W.SplitMix64(3)
    sweeps = []
    for gates in (W.qft(n), [u3(q, r) for q in range(n)] + W.qft(n)):
        s = gpu_engine.ZXH(n, False, True)
        s.gates(gates)
        s.set_timing(True)
        s.execute()
        s.set_timing(False)
        sweeps.append(sum(s.timing(f)["launches"] for f in ("u3_tile", "u3_pair", "fused", "diag")))
    assert sweeps[0] == sweeps[1]
