"""How a circuit is split into passes that execute it out of LDS
(zxh_circuit_plan; host only, no device).  The plan is this engine's own (the
reference applies one sweep per gate, zxh.cpp:390-428), so the checks are its
contract: every operation once, operations that do not commute in the
circuit's order, a pass's pair offsets within one tile."""
import time

import numpy as np
import pytest

from zxh_adae_amd import _lib
from zxh_adae_amd._lib import check

NO_SEL = (1 << 64) - 1
ALPHA = (1 << 63) - 1
TOP = 1 << 63
TILE = {"c128": 12, "c64": 13}
WHOLE = {"c128": 13, "c64": 14}
RUN = {"c128": 3, "c64": 4}


def plan(prec, nbits, ops):
    """ops: (kind, delta, sel0, sel1)."""
    lib = _lib.load()
    kind = np.array([o[0] for o in ops], np.uint32)
    cols = [np.array([o[k] for o in ops], np.uint64) for k in (1, 2, 3)]
    order, pass_of = np.empty(len(ops), np.uint32), np.empty(len(ops), np.uint32)
    check(lib.zxh_circuit_plan(_lib.ZXH_C128 if prec == "c128" else _lib.ZXH_C64, nbits, kind.ctypes.data,
                               *(c.ctypes.data for c in cols), len(ops), order.ctypes.data, pass_of.ctypes.data))
    return order, pass_of


def parity(x):
    return bin(x).count("1") & 1


def commute(a, b):
    if 1 in (a[0], b[0]):
        return False
    if a[0] == 2 and b[0] == 2:
        return True
    if a[0] == 2:
        a, b = b, a
    if b[0] == 2:
        return not parity(b[2] & ALPHA & a[1]) and (b[3] == NO_SEL or not parity(b[3] & ALPHA & a[1]))
    return not parity(a[2] & ALPHA & b[1]) and not parity(b[2] & ALPHA & a[1])


def rank(vs):
    rows = []
    for v in vs:
        for r in rows:
            v = min(v, v ^ r)
        if v:
            rows.append(v)
    return len(rows)


def check_plan(prec, nbits, ops):
    order, pass_of = plan(prec, nbits, ops)
    assert sorted(order.tolist()) == list(range(len(ops)))
    assert np.all(np.diff(pass_of.astype(np.int64)) >= 0)
    place = np.empty(len(ops), np.int64)
    place[order] = np.arange(len(ops))
    for i in range(len(ops)):
        for j in range(i + 1, len(ops)):
            assert place[i] < place[j] or commute(ops[i], ops[j]), (i, j)
    if nbits > WHOLE[prec]:
        for p in range(int(pass_of.max()) + 1 if len(ops) else 0):
            vs = [ops[o][1] for o in order[pass_of == p] if ops[o][0] != 2]
            assert rank([1 << b for b in range(RUN[prec])] + vs) <= TILE[prec]
    return order, pass_of


def random_ops(rng, nbits, nops, kinds):
    ops = []
    for _ in range(nops):
        k = kinds[int(rng.integers(len(kinds)))]
        beta = TOP if rng.random() < 0.3 else 0
        sel = lambda: int(rng.integers(1 << nbits)) | (TOP if rng.random() < 0.3 else 0)
        if k == "bit":
            d = 1 << int(rng.integers(nbits))
            ops.append((0, d, d | beta, 0))
        elif k == "diag":
            s = [1 << int(rng.integers(nbits)) for _ in range(2)]
            ops.append((2, 0, s[0] | beta, s[1] if rng.random() < 0.5 else NO_SEL))
        elif k == "wide diag":
            ops.append((2, 0, sel(), sel() if rng.random() < 0.5 else NO_SEL))
        else:  # an offset and a selector of several bits, of odd parity over it
            d = int(rng.integers(1, 1 << nbits))
            s = int(rng.integers(1 << nbits))
            s ^= 0 if parity(s & d) else d & -d
            ops.append((1, d, s | beta, sel()) if k == "control" else (0, d, s | beta, 0))
    return ops


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("ops", [[(2, 0, TOP, NO_SEL)], [(2, 0, TOP, TOP)], [(2, 0, TOP, NO_SEL)] * 3000, []])
def test_no_address_bits(prec, ops):
    """Circuits without a superposition: phase gates with constant selectors
    on a state of one amplitude."""
    order, pass_of = plan(prec, 0, ops)
    assert sorted(order.tolist()) == list(range(len(ops)))
    assert np.all(np.diff(pass_of.astype(np.int64)) >= 0)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("nbits", [1, 2, 5, 13, 14, 15, 17, 22])
@pytest.mark.parametrize("kinds", [("bit",), ("bit", "diag"), ("bit", "diag", "diag", "diag"), ("wide", "wide diag"),
                                   ("bit", "wide", "diag", "control")], ids="+".join)
def test_random_circuits(prec, nbits, kinds):
    rng = np.random.default_rng(nbits)
    check_plan(prec, nbits, random_ops(rng, nbits, 150, kinds))


def plan_seconds(nbits, nops):
    """Gates whose offsets take two random bits, on the host clock."""
    rng = np.random.default_rng(1)
    b = rng.integers(nbits, size=nops)
    sel = np.uint64(1) << b.astype(np.uint64)
    delta = sel | np.uint64(1) << ((b + 1 + rng.integers(nbits - 1, size=nops)) % nbits).astype(np.uint64)
    kind, zero = np.zeros(nops, np.uint32), np.zeros(nops, np.uint64)
    order, pass_of = np.empty(nops, np.uint32), np.empty(nops, np.uint32)
    t = time.perf_counter()
    check(_lib.load().zxh_circuit_plan(_lib.ZXH_C128, nbits, kind.ctypes.data, delta.ctypes.data, sel.ctypes.data,
                                       zero.ctypes.data, nops, order.ctypes.data, pass_of.ctypes.data))
    return time.perf_counter() - t


def test_time_grows_with_the_length():
    """Sixteen times the operations: 16 times the time when a pass touches
    only the operations it looks at, 195 times when it moved all that follow.
    The bound is three times the first, the least of three runs each."""
    small = min(plan_seconds(16, 50_000) for _ in range(3))
    large = min(plan_seconds(16, 800_000) for _ in range(3))
    assert large < 48 * small, (small, large)


def test_bad_arguments():
    lib = _lib.load()
    a = np.zeros(1, np.uint64)
    k = np.array([2], np.uint32)
    p = [k.ctypes.data, a.ctypes.data, a.ctypes.data, a.ctypes.data]
    o = np.zeros(1, np.uint32).ctypes.data
    assert lib.zxh_circuit_plan(7, 3, *p, 1, o, o) == 1
    assert lib.zxh_circuit_plan(_lib.ZXH_C128, 23, *p, 1, o, o) == 1
    assert lib.zxh_circuit_plan(_lib.ZXH_C64, 24, *p, 1, o, o) == 1
    assert lib.zxh_circuit_plan(_lib.ZXH_C128, 3, *p, 1, None, o) == 1
    k[0] = 3
    assert lib.zxh_circuit_plan(_lib.ZXH_C128, 3, *p, 1, o, o) == 1
    k[0] = 0  # no pair offset
    assert lib.zxh_circuit_plan(_lib.ZXH_C128, 3, *p, 1, o, o) == 1
