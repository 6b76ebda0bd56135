"""Complex64 pair offsets that flip address bit 0 together with other bits
ride tile passes from 20 address bits on: batches and whole circuits against
the oracle, on the tile kernel and the upper kernel, with per-pair selectors
that see bit 0, with the in-unit gate in the batch, and with a window after it."""
import numpy as np
import pytest

import oracle_py as O
from test_gpu_kernels import TOL64, dev, oracle_u3, pack, rand_state, rand_u, random_affine
from zxh_adae_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 18, 64], ids=lambda u: f"upper{u}")
def upper(request, gpu_engine):
    from zxh_adae_amd import autotune as A
    old = {k: A.tune_get(k) for k in ("tile.upper.c64", "circuit.bits.c64")}
    A.tune_set("tile.upper.c64", request.param)
    A.tune_set("circuit.bits.c64", 0)
    yield
    for k, v in old.items():
        A.tune_set(k, v)


@pytest.mark.parametrize("n,cx,seed", [(20, 5, 1), (20, 60, 2), (21, 200, 3), (22, 12, 4)])
def test_batches(gpu_engine, upper, n, cx, seed):
    from zxh_adae_amd import kernels as K
    rng = np.random.default_rng(seed)
    rows, deltas = random_affine(rng, n, cx)
    psi = rand_state(rng, n)
    descs = [(pack(rows[q], bool(rng.random() < 0.5)), deltas[q], rand_u(rng)) for q in range(n)]
    cross = [d for _, d, _ in descs if d & 1 and d != 1]
    want = oracle_u3(psi, n, descs)
    d = dev(gpu_engine, psi.astype(np.complex64), "c64")
    K.set_timing(True)
    K.reset_timing()
    try:
        d.u3_batch(descs)
        pair = K.timing("u3_pair")["launches"]
    finally:
        K.set_timing(False)
    assert np.max(np.abs(d.download().astype(np.complex128) - want)) < TOL64
    assert pair == 0, (pair, len(cross))


@pytest.mark.parametrize("n,kind", [(20, "chain"), (20, "reverse"), (21, "soup"), (20, "window")])
def test_circuits(gpu_engine, upper, n, kind):
    """Lazy mode: a CX chain up, a chain down (every offset then reaches bit
    0), random CX, and windows that ride the passes as tables."""
    r = W.SplitMix64(n)
    gates = []
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
        if kind == "window":
            gates += [(W.P, 0, q, r.uniform(), 0, 0) for q in range(4)]
    gates += [(W.H, 0, q, 0, 0, 0) for q in range(n)]
    o = O.OracleSim(n, False, False)
    o.gates(gates)
    o.execute()
    s = gpu_engine.ZXH(n, precision="c64")
    s.gates(gates)
    s.execute()
    assert np.max(np.abs(s.get_state_array() - o.get_state())) < 2e-5


@pytest.mark.parametrize("sel,delta", [(2, 3), (1, 3), (1 << 19, (1 << 19) | 1)])
def test_a_gate_by_itself_takes_a_sweep(gpu_engine, sel, delta):
    from zxh_adae_amd import kernels as K
    rng = np.random.default_rng(sel)
    psi = rand_state(rng, 20)
    descs = [(sel, delta, rand_u(rng))]
    d = dev(gpu_engine, psi.astype(np.complex64), "c64")
    K.set_timing(True)
    K.reset_timing()
    try:
        d.u3_batch(descs)
        assert K.timing("u3_pair")["launches"] == 1
    finally:
        K.set_timing(False)
    assert np.max(np.abs(d.download().astype(np.complex128) - oracle_u3(psi, 20, descs))) < TOL64
