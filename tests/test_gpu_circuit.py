"""Circuits executed out of LDS (knobs circuit.bits.<prec>): states of one tile
(complex128 to 13 address bits, complex64 to 14) and tiles of wider ones,
against the oracle at the edges of both ranges and of a pass's steps, gates,
windows, window tables and tiles; and the tile passes, which take the same
circuits when the knob is 0."""
import numpy as np
import pytest

import oracle_py as O
from zxh_adae_amd import autotune as A
from zxh_adae_amd import workloads as W

pytestmark = pytest.mark.gpu

# complex128: the engine's 1e-12; complex64: 6e-8 per rounding, a few
# roundings per gate adding as a random walk over at most 3000 gates
TOL = {"c128": 1e-12, "c64": 2e-5}
MODES = {"lazy": (False, False), "plain": (False, True), "nox": (True, True), "nox_lazy": (True, False)}


def check(Z, n, gates, prec, mode, knobs=(None,)):
    dx, eager = MODES[mode]
    o = O.OracleSim(n, dx, eager)
    o.gates(gates)
    o.execute()
    want = o.get_state()
    name = f"circuit.bits.{prec}"
    old = A.tune_get(name)
    try:
        for k in knobs:
            if k is not None:
                A.tune_set(name, k)
            s = Z.ZXH(n, dx, eager, precision=prec)
            s.gates(gates)
            for _ in range(2):  # the second run starts from a written state
                s.execute()
                assert np.max(np.abs(s.get_state_array() - want)) < TOL[prec], (n, mode, k)
    finally:
        A.tune_set(name, old)
    return s


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 11, 12, 13, 14, 15, 16, 18])
def test_soups(gpu_engine, n, mode, prec):
    """Every gate kind; 13 is complex128's widest one-tile state and 14
    complex64's."""
    check(gpu_engine, n, W.random_mixed(n, 40 + 20 * n, 700 + n), prec, mode, (None, 0) if n > 11 else (None,))


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("kind", ["z", "rz", "p", "cp", "cx_cp", "unset", "many"])
@pytest.mark.parametrize("n", [1, 2, 3, 5])
def test_no_superposition(gpu_engine, n, kind, prec):
    """Default mode without U3 or H: a state of no address bits, whose phase
    gates on set qubits have constant selectors."""
    a, b = 0, n - 1
    if n == 1 and kind in ("cp", "cx_cp"):
        pytest.skip("needs two qubits")
    gates = {"z": [(W.X, 0, b, 0, 0, 0), (W.Z, 0, b, 0, 0, 0)],
             "rz": [(W.X, 0, b, 0, 0, 0), (W.RZ, 0, b, 0.3, 0, 0)],
             "p": [(W.X, 0, b, 0, 0, 0), (W.P, 0, b, 0.3, 0, 0), (W.X, 0, b, 0, 0, 0), (W.P, 0, b, 0.5, 0, 0)],
             "cp": [(W.X, 0, a, 0, 0, 0), (W.X, 0, b, 0, 0, 0), (W.CP, a, b, 0.3, 0, 0)],
             "cx_cp": [(W.X, 0, a, 0, 0, 0), (W.CX, a, b, 0, 0, 0), (W.CP, a, b, 0.3, 0, 0)],
             "unset": [(W.P, 0, b, 0.3, 0, 0)],
             # (a circuit of up to 24 gates takes a launch of its own for the window)
             "many": [(W.X, 0, a, 0, 0, 0)] + [(W.X, 0, b, 0, 0, 0), (W.P, 0, b, 0.3, 0, 0)] * 40}[kind]
    s = check(gpu_engine, n, gates, prec, "lazy", (None, 0))
    s.set_seed(5)
    s.measure(7)
    at = np.flatnonzero(s.get_state_array())
    assert at.size == 1 and np.all(s.results_bits() == [(at[0] >> (n - 1 - q)) & 1 for q in range(n)])


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,gates", [(2, [(W.X, 0, 1, 0, 0, 0), (W.P, 0, 1, 0.3, 0, 0)] * 13), (5, W.hadamard_all(5))])
def test_knob_at_zero_is_never(gpu_engine, n, gates, prec):
    """Also for a state of no address bits."""
    name = f"circuit.bits.{prec}"
    old = A.tune_get(name)
    s = gpu_engine.ZXH(n, False, False, precision=prec)
    s.gates(gates)
    s.set_timing(True)
    try:
        for knob, launches in ((0, 0), (old, 1)):
            A.tune_set(name, knob)
            s.reset_timing()
            s.execute()
            assert s.timing("fused")["launches"] == launches
    finally:
        A.tune_set(name, old)


@pytest.mark.parametrize("prec,n", [("c128", 13), ("c64", 14), ("c128", 14), ("c64", 15), ("c128", 17)])
def test_no_gates_and_one_gate(gpu_engine, prec, n):
    s = check(gpu_engine, n, [], prec, "plain")
    assert s.get_state_array()[0] == 1 and np.count_nonzero(s.get_state_array()) == 1
    check(gpu_engine, n, [(W.H, 0, n - 1, 0, 0, 0)], prec, "plain")
    check(gpu_engine, n, [(W.CP, 0, n - 1, 0.3, 0, 0)], prec, "plain")
    check(gpu_engine, n, [(W.U3, 0, q, 0.3, 0.2, 0.1) for q in (0, n // 2, n - 1)] + [(W.P, 0, n - 1, 0.3, 0, 0)],
          prec, "plain")


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,layers", [(4, 120), (7, 700), (13, 60)])
def test_many_steps(gpu_engine, n, layers, prec):
    """More steps than one pass takes (about 500, with the state written and
    read between the passes), and window tables beyond one pass's share (32 MiB
    at 13 bits)."""
    gates = W.random_layers(n, layers, 40 + n)
    if n == 13:
        # windows that do not merge: one gate between each two
        r = W.SplitMix64(9)
        for k in range(300):
            gates += [(W.H, 0, k % n, 0, 0, 0), (W.CP, k % n, (k + 1) % n, r.uniform(), 0, 0)]
    check(gpu_engine, n, gates, prec, "plain")


def test_a_window_larger_than_a_pass_takes(gpu_engine):
    """9000 gates in one window.  Their angles are scaled by 1e-3: the sum of
    a window's angles rounds by half an ulp of the partial sum per gate, and
    with whole angles (partial sums to 14000: 9e-13 each, a random walk of
    9000 of them) that alone passes 1e-12; below 32 they are 1.8e-15 each,
    1.7e-13 in all."""
    for n in (6, 14):
        window = [g[:3] + (g[3] * 1e-3, 0.0, 0.0) for g in W.diag_batch(n, 9000, 3)]
        check(gpu_engine, n, W.hadamard_all(n) + window + W.hadamard_all(n), "c128", "plain")


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n", [7, 14, 15])
def test_a_window_of_more_different_gates_than_a_pass_takes(gpu_engine, n, prec):
    """4000 gates, each under another map (a CX before it), of which a pass
    takes 2560; a whole state, and tables of every tile.  Angles to 1e-3: see
    the test above."""
    r = W.SplitMix64(5 * n)
    gates = W.hadamard_all(n)
    for k in range(4000):
        a, b, c, d = r.below(n), r.below(n - 1), r.below(n), r.below(n - 1)
        gates.append((W.CX, a, b + (b >= a), 0, 0, 0))
        gates.append((W.CP, c, d + (d >= c), 1e-3 * r.uniform(), 0, 0))
    check(gpu_engine, n, gates + W.hadamard_all(n), prec, "lazy", (None, 0))


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("mode", ["plain", "lazy"])
@pytest.mark.parametrize("n,count", [(1, 65), (2, 200), (5, 64), (7, 128), (13, 129), (14, 300), (15, 1000), (18, 300)])
def test_windows_of_equal_gates(gpu_engine, n, count, mode, prec):
    """Windows above 64 gates, whose equal ones become one: P and CP gates on
    random qubits in both orders, with X gates between them (selectors of
    either sign) and, in the last window, after CX transport.  Angles to 0.01:
    see the test above."""
    r = W.SplitMix64(1000 * n + count)
    gates = W.hadamard_all(n)
    for part in range(3):
        if part == 2 and n > 1:
            gates += [(W.CX, q, (q + 1) % n, 0, 0, 0) for q in range(n)]
        for k in range(count):
            a, b = r.below(n), r.below(n)
            if k % 7 == 3:
                gates.append((W.X, 0, a, 0, 0, 0))
            gates.append((W.P, 0, a, 0.01 * r.uniform(), 0, 0) if a == b else (W.CP, a, b, 0.01 * r.uniform(), 0, 0))
        gates += [(W.U3, 0, q, r.uniform() * 6, r.uniform() * 6, r.uniform() * 6) for q in range(n)]
    check(gpu_engine, n, gates, prec, mode, (None, 0))


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,layers", [(14, 20), (17, 9), (20, 6), (21, 3), (22, 2)])
def test_layers_over_tiles(gpu_engine, n, layers, prec):
    """Layers with CP ladders: passes that carry parts of several layers, up
    to eight windows; every state width up to ten
    address bits outside a tile (the knob at its largest), and more tiles
    than workgroups at a time."""
    top = {"c128": 22, "c64": 23}[prec]
    check(gpu_engine, n, W.random_layers(n, layers, 50 + n), prec, "plain", (top, 0))


@pytest.mark.parametrize("prec,n", [("c128", 14), ("c128", 18), ("c128", 19), ("c64", 15), ("c64", 20), ("c64", 21)])
@pytest.mark.parametrize("mode", ["plain", "lazy"])
def test_windows_of_both_kinds(gpu_engine, n, mode, prec):
    """Windows that split by tile and coordinate and windows that do not, in
    one pass and in turn, at both ends of the states whose tables hold every
    tile, and one bit above."""
    r = W.SplitMix64(31 * n)
    gates = W.hadamard_all(n)
    for layer in range(4):
        if layer % 2:
            gates += [(W.CX, q, (q + 3) % n, 0, 0, 0) for q in range(n)]
        for k in range(2 * n):
            a, b = r.below(n), r.below(n - 1)
            gates.append((W.CP, a, b + (b >= a), r.uniform(), 0, 0))
        if layer % 2:
            gates += [(W.CX, q, (q + 3) % n, 0, 0, 0) for q in reversed(range(n))]
        gates += [(W.U3, 0, q, r.uniform() * 6, r.uniform() * 6, r.uniform() * 6) for q in range(0, n, 1 + layer % 2)]
        gates += [(W.CP, q, q + 1, r.uniform(), 0, 0) for q in range(n - 1)]
        gates += [(W.H, 0, q, 0, 0, 0) for q in range(3)]
    check(gpu_engine, n, gates, prec, mode, (None, 0))


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n", [14, 17, 20])
@pytest.mark.parametrize("kind", ["chain", "reverse", "soup", "windows", "qft"])
def test_transported_circuits_over_tiles(gpu_engine, n, kind, prec):
    """Lazy mode: offsets and selectors of many bits (tiles that are cosets
    of wide offsets), windows whose selectors do not split by tile and
    coordinate, and a QFT (windows over every bit)."""
    r = W.SplitMix64(n)
    gates = []
    if kind == "qft":
        gates = [(W.U3, 0, q, r.uniform() * 6, r.uniform() * 6, r.uniform() * 6) for q in range(n)] + W.qft(n)
        gates += W.qft(n)
    else:
        for layer in range(3):
            gates += [(W.U3, 0, q, r.uniform() * 6, r.uniform() * 6, r.uniform() * 6) for q in range(n)]
            if kind == "chain":
                gates += [(W.CX, q, q + 1, 0, 0, 0) for q in range(n - 1)]
            elif kind == "reverse":
                gates += [(W.CX, q + 1, q, 0, 0, 0) for q in range(n - 1)]
            else:
                for _ in range(2 * n):
                    a, b = r.below(n), r.below(n - 1)
                    gates.append((W.CX, a, b + (b >= a), 0, 0, 0))
            if kind == "windows":
                gates += [(W.P, 0, q, r.uniform(), 0, 0) for q in range(n)]
                gates += [(W.CP, q, (q + 2) % n, r.uniform(), 0, 0) for q in range(n)]
        gates += [(W.H, 0, q, 0, 0, 0) for q in range(n)]
    check(gpu_engine, n, gates, prec, "lazy", (None, 0))
