"""Sweeps of two rounds (the last targets of a layer, its window and the first
targets of the next one on the same tiles): energies, norms and gradients of
single circuits and batches against an adjoint differentiation in numpy, at
widths of one, two and three chunks of targets and for circuits whose layers
leave qubits out, share parameters and carry three rotations on a qubit."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# complex128: roundings of 1e-16 over a few hundred gates, on sums of up to
# twelve terms.  complex64: 6e-8 each.
TOL = {"c128": 1e-12, "c64": 2e-5}


def ragged(rng, n, layers):
    """Layers on random halves of the qubits; parameter 0 is shared by many."""
    from zxh_adae_amd.ansatz import RX, RY, RZ, H, CZ, CP
    ops, count = [], 1
    for _ in range(layers):
        for q in range(n):
            if rng.random() < 0.4:
                continue
            for _ in range(int(rng.integers(1, 4))):
                kind = int(rng.choice([RX, RY, RZ]))
                if rng.random() < 0.2:
                    ops.append((kind, q, 0, -1, float(rng.uniform(-3, 3))))
                elif rng.random() < 0.2:
                    ops.append((kind, q, 0, 0, 0.0))
                else:
                    ops.append((kind, q, 0, count, 0.0))
                    count += 1
            if rng.random() < 0.2:
                ops.append((H, q, 0, -1, 0.0))
        for _ in range(int(rng.integers(0, n))):
            a, b = (int(x) for x in rng.choice(n, 2, replace=False))
            ops.append((CZ, a, b, -1, 0.0) if rng.random() < 0.5 else (CP, a, b, -1, float(rng.uniform(-3, 3))))
    return ops, count


def matrix(kind, t):
    from zxh_adae_amd.ansatz import RX, RY, RZ
    c, s = math.cos(t / 2), math.sin(t / 2)
    if kind == RX:
        return np.array([[c, -1j * s], [-1j * s, c]])
    if kind == RY:
        return np.array([[c, -s], [s, c]], dtype=complex)
    if kind == RZ:
        return np.diag([c - 1j * s, c + 1j * s])
    return np.array([[1, 1], [1, -1]], dtype=complex) / math.sqrt(2.0)


def generator(kind):
    from zxh_adae_amd.ansatz import RX, RY
    return np.array([[0, 1], [1, 0]] if kind == RX else [[0, -1j], [1j, 0]] if kind == RY else [[1, 0], [0, -1]])


def apply(psi, q, u):
    v = psi.reshape(-1, 2, 1 << q)
    out = np.empty_like(v)
    out[:, 0] = u[0, 0] * v[:, 0] + u[0, 1] * v[:, 1]
    out[:, 1] = u[1, 0] * v[:, 0] + u[1, 1] * v[:, 1]
    return out.reshape(-1)


def reference(n, ops, params, terms):
    from zxh_adae_amd.ansatz import CP, CZ
    x = np.arange(1 << n, dtype=np.int64)

    def phase(o, sign):
        a = sign * (math.pi if o[0] == CZ else o[4])
        return np.where(((x >> o[1]) & (x >> o[2]) & 1) != 0, np.exp(1j * a), 1.0)

    def angle(o):
        return params[o[3]] if o[3] >= 0 else o[4]

    psi = np.zeros(1 << n, dtype=complex)
    psi[0] = 1.0
    for o in ops:
        psi = psi * phase(o, 1) if o[0] in (CZ, CP) else apply(psi, o[1], matrix(o[0], angle(o)))
    h = np.zeros(1 << n)
    for t in terms:
        z = 1.0 - 2.0 * ((x >> t[1]) & 1)
        if len(t) > 2:
            z = z * (1.0 - 2.0 * ((x >> t[2]) & 1))
        h += t[0] * z
    e = float(np.sum(np.abs(psi) ** 2 * h))
    lam = h * psi
    g = np.zeros(len(params))
    for o in reversed(ops):
        if o[0] in (CZ, CP):
            w = phase(o, -1)
            psi, lam = psi * w, lam * w
            continue
        if o[3] >= 0:
            # dU/dt = -i/2 G U: 2 Re <lam| -i/2 G |psi>
            g[o[3]] += np.imag(np.vdot(lam, apply(psi, o[1], generator(o[0]))))
        u = matrix(o[0], angle(o)).conj().T
        psi, lam = apply(psi, o[1], u), apply(lam, o[1], u)
    return e, g


def circuit(rng, n, kind, layers):
    from zxh_adae_amd.ansatz import two_local
    return two_local(n, layers) if kind == "two_local" else ragged(rng, n, layers)


def terms_of(rng, n):
    out = []
    for _ in range(12):
        i, j = (int(q) for q in rng.choice(n, 2, replace=False))
        out.append((float(rng.normal()), i) if rng.random() < 0.5 else (float(rng.normal()), i, j))
    return out


@pytest.mark.parametrize("kind", ["two_local", "ragged"])
@pytest.mark.parametrize("prec,n", [("c128", 12), ("c128", 13), ("c128", 16), ("c64", 13), ("c64", 14), ("c64", 17)])
def test_single_circuits(gpu_engine, prec, n, kind):
    from zxh_adae_amd.ansatz import Ansatz
    rng = np.random.default_rng(n)
    layers = 4
    ops, count = circuit(rng, n, kind, layers)
    params, terms = rng.uniform(-math.pi, math.pi, count), terms_of(rng, n)
    e, g = reference(n, ops, params, terms)
    a = Ansatz(n, ops, count, prec)
    a.set_observable(terms)
    if kind == "two_local":
        # one chunk: a sweep per layer; two: the last of a layer and the
        # first of the next are one
        assert a.tile_passes() == (layers if n == (12 if prec == "c128" else 13) else layers + 1)
    scale = sum(abs(t[0]) for t in terms)
    for _ in range(2):
        got, norm = a.forward(params)
        grads, back = a.backward(params)
        assert abs(got - e) < TOL[prec] * scale and abs(back - e) < TOL[prec] * scale
        assert abs(norm - 1.0) < TOL[prec]
        assert np.max(np.abs(grads - g)) < TOL[prec] * scale * (1 if kind == "two_local" else 4 * layers)
    a.close()


@pytest.mark.parametrize("seg", [0, 3, 6])
@pytest.mark.parametrize("prec,widths", [("c128", [14, 16, 19, 15]), ("c64", [20, 15, 16])])
def test_batches(gpu_engine, prec, widths, seg):
    """Geometry 6 leaves six targets above the low ones to a tile: 19 and 20
    qubits take three chunks (of twelve, a sweep joins only one)."""
    from zxh_adae_amd.ansatz import AnsatzBatch
    rng = np.random.default_rng(seg)
    b = AnsatzBatch(prec)
    sets = []
    for k, n in enumerate(widths):
        ops, count = circuit(rng, n, "two_local" if k % 2 == 0 else "ragged", 2 + k % 2)
        terms = terms_of(rng, n)
        b.set_geometry(n, seg)
        b.add(n, ops, count, terms)
        sets.append((n, ops, rng.uniform(-math.pi, math.pi, count), terms))
    b.finalize()
    want = [reference(*s) for s in sets]
    for _ in range(3):
        e, norms, grads = b.run([s[2] for s in sets])
        only, _, _ = b.run([s[2] for s in sets], gradients=False)
        for k, s in enumerate(sets):
            # (the ragged circuits add up to a dozen entries into parameter 0)
            tol = TOL[prec] * sum(abs(t[0]) for t in s[3])
            assert abs(e[k] - want[k][0]) < tol and abs(only[k] - want[k][0]) < tol
            assert abs(norms[k] - 1.0) < TOL[prec]
            assert np.max(np.abs(grads[k] - want[k][1])) < 12 * tol
    b.close()


def layered(n, kind, layers, seed):
    from zxh_adae_amd import workloads as W
    rng = np.random.default_rng(seed)
    gates = []
    for _ in range(layers):
        qs = range(n) if kind != "part" else [q for q in range(n) if rng.random() < 0.8]
        gates += [(W.U3, 0, q, *rng.uniform(0, 6, 3)) for q in qs]
        if kind == "flipped":
            gates += [(W.X, 0, int(q), 0, 0, 0) for q in rng.choice(n, n // 2, replace=False)]
        gates += [(W.CP, q, q + 1, float(rng.uniform(0, 6)), 0, 0) for q in range(n - 1)]
        gates += [(W.P, 0, q, float(rng.uniform(0, 6)), 0, 0) for q in range(n)]
    return gates


@pytest.mark.parametrize("kind", ["whole", "part", "flipped"])
@pytest.mark.parametrize("plain", [True, False])
@pytest.mark.parametrize("prec,n", [("c128", 12), ("c128", 13), ("c128", 17), ("c128", 21), ("c64", 13), ("c64", 14),
                                    ("c64", 18), ("c64", 22)])
def test_engine_layers(gpu_engine, prec, n, plain, kind):
    """The engine's batches behind a window (flipped: after X gates, whose
    affine bit swaps the sides of a gate's pair), in tile passes; one and two
    passes a layer, all targets below the tile and some left to a second."""
    import oracle_py as O
    from zxh_adae_amd import autotune as A
    layers = 3
    gates = layered(n, kind, layers, n)
    o = O.OracleSim(n, False, plain)
    o.gates(gates)
    o.execute()
    old = A.tune_get(f"circuit.bits.{prec}")
    A.tune_set(f"circuit.bits.{prec}", 0)
    try:
        s = gpu_engine.ZXH(n, False, plain, precision=prec)
        s.gates(gates)
        s.set_timing(True)
        s.execute()
        launches = sum(s.timing(f)["launches"] for f in ("u3_tile", "fused"))
        assert np.max(np.abs(s.get_state_array() - o.get_state())) < (1e-12 if prec == "c128" else 5e-6)
    finally:
        A.tune_set(f"circuit.bits.{prec}", old)
    if plain and kind == "whole" and n in (17, 18):
        assert launches == layers + 1  # two a layer, the end of one with the start of the next
