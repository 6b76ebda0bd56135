"""Performance cases of the state-vector engine: what its users run.

Three ways into the engine are covered, each over the sizes it is used at:

  circ    the drop-in ZXH object: a recorded circuit executed from |0...0>,
          then shots or the whole state read out, as the application needs.
          Circuits: U3 + CP-ladder + P layers, QFT on a product state, QAOA
          (CX-Rz-CX edges and Rx mixers), and the hardware-efficient SU2 form
          (U3 on every qubit, a CX chain); in the default mode (CX as an
          affine update of the addresses) and in the plain method.
  sample  ZXH.sample_real: a multinomial draw from a state already there
  diag    DeviceState.diag: one batch of P / CP gates on a resident state
  layer   one layer of the dense-block circuit on a resident state: 5-qubit
          unitaries on a random qubit order, a diagonal batch, a cascade of
          multi-controlled X
  grad    expectation value and adjoint gradient of the two-local ansatz
          (torch autograd, or the ansatz object itself for complex64)
  batch   many ansatz circuits of uneven width and depth in one run

A circuit's gates are recorded in prepare(): a program records them once and
executes many times.  Kernel-level calls change the state in place, so a
second pass over the same state continues from the first one's result.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import zxh_adae_amd as Z
from zxh_adae_amd import ansatz as A
from zxh_adae_amd import kernels as K
from zxh_adae_amd.torch_ext import expectation

# gate codes of ZXH.gate (code, cq, q, theta, lambda, phi)
P, CP, CX, H, U3, RZ, RX = 4, 6, 8, 9, 10, 3, 11
TWO_PI = 2.0 * math.pi


def listed():
    return [
        # a small variational circuit: ten qubits, latency and launches
        {"name": "su2_n10_c128_shots", "kind": "circ", "circuit": "su2", "n": 10, "depth": 3, "plain": False,
         "c64": False, "read": "shots", "shots": 1024},
        # the 20-qubit random circuit of 1180 gates and 1024 shots, plain method
        {"name": "layers_n20_c128_shots", "kind": "circ", "circuit": "layers", "n": 20, "depth": 20, "plain": True,
         "c64": False, "read": "shots", "shots": 1024},
        # a circuit whose whole state vector goes back to the caller
        {"name": "layers_n17_c128_state", "kind": "circ", "circuit": "layers", "n": 17, "depth": 4, "plain": False,
         "c64": False, "read": "state", "shots": 0},
        # the 30-qubit QFT in the plain method, 16 GiB of state
        {"name": "qft_n30_c128", "kind": "circ", "circuit": "qft", "n": 30, "depth": 1, "plain": True,
         "c64": False, "read": "", "shots": 0},
        # QAOA in the default mode, an everyday size
        {"name": "qaoa_n25_c128", "kind": "circ", "circuit": "qaoa", "n": 25, "depth": 2, "plain": False,
         "c64": False, "read": "", "shots": 0},
        # a hardware-efficient circuit in single precision, default mode
        {"name": "su2_n27_c64", "kind": "circ", "circuit": "su2", "n": 27, "depth": 3, "plain": False,
         "c64": True, "read": "", "shots": 0},
        # a million shots from a 30-qubit state
        {"name": "sample_n30_c128", "kind": "sample", "n": 30, "c64": False, "shots": 1000000},
        # 64 phase gates as one sweep over a 30-qubit state
        {"name": "diag_n30_c128", "kind": "diag", "n": 30, "c64": False, "gates": 64},
        # one dense-block layer, six 5-qubit blocks
        {"name": "layer_n30_c64", "kind": "layer", "n": 30, "c64": True, "gates": 64, "mcx": 8},
        # the 28-qubit two-local ansatz, 448 parameters, 200 terms
        {"name": "grad_n28_c64", "kind": "grad", "n": 28, "depth": 8, "terms": 200, "c64": True},
        # a gradient at a size that optimisers iterate at
        {"name": "grad_n16_c128", "kind": "grad", "n": 16, "depth": 4, "terms": 50, "c64": False},
        # 128 circuits of 16..24 qubits and 2..10 layers
        {"name": "batch_128_c64", "kind": "batch", "sets": 128, "lo": 16, "hi": 24, "dlo": 2, "dhi": 10,
         "terms": 50, "c64": True},
    ]


def _log(rng, lo, hi):
    """An integer in lo..hi, uniform over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["circ", "circ", "circ", "circ", "circ", "sample", "diag", "layer", "grad", "grad", "batch"])
    c64 = rng.random() < 0.4
    if kind == "circ":
        circuit = rng.choice(["layers", "qft", "qaoa", "su2"])
        n = rng.randint(4, 28)
        depth = {"layers": _log(rng, 1, 20), "qft": 1, "qaoa": rng.randint(1, 3), "su2": rng.randint(1, 5)}[circuit]
        if n > 24:
            depth = min(depth, 4)
        read = rng.choice(["", "shots", "state"] if n <= 18 else ["", "shots"])
        return {"kind": kind, "circuit": circuit, "n": n, "depth": depth, "plain": rng.random() < 0.4, "c64": c64,
                "read": read, "shots": _log(rng, 100, 20000) if read == "shots" else 0}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(10, 29), "c64": c64, "shots": _log(rng, 100, 1000000)}
    if kind == "diag":
        return {"kind": kind, "n": rng.randint(10, 29), "c64": c64, "gates": _log(rng, 1, 256)}
    if kind == "layer":
        return {"kind": kind, "n": rng.randint(11, 29), "c64": c64, "gates": _log(rng, 8, 128),
                "mcx": rng.randint(1, 8)}
    if kind == "grad":
        n = rng.randint(13, 26)
        return {"kind": kind, "n": n, "depth": rng.randint(1, 8), "terms": _log(rng, 5, 200), "c64": rng.random() < 0.6}
    lo = rng.randint(16, 20)
    dlo = rng.randint(1, 4)
    return {"kind": kind, "sets": _log(rng, 4, 64), "lo": lo, "hi": lo + rng.randint(0, 3), "dlo": dlo,
            "dhi": dlo + rng.randint(0, 5), "terms": _log(rng, 5, 50), "c64": c64 or rng.random() < 0.5}


# ---- inputs ----

def _gates(case, seed):
    """The circuit's gate tuples; every angle comes from the seed."""
    r = random.Random(seed * 7919 + 17)
    n, depth = case["n"], case["depth"]

    def ang():
        return r.uniform(0.0, TWO_PI)

    def u3(q):
        return (U3, 0, q, ang(), ang(), ang())
    gs = []
    if case["circuit"] == "layers":
        for _ in range(depth):
            gs += [u3(q) for q in range(n)]
            gs += [(CP, q, q + 1, ang(), 0.0, 0.0) for q in range(n - 1)]
            gs += [(P, 0, q, ang(), 0.0, 0.0) for q in range(n)]
    elif case["circuit"] == "qft":
        gs += [u3(q) for q in range(n)]
        for t in range(n):
            gs.append((H, 0, t, 0.0, 0.0, 0.0))
            gs += [(CP, j, t, math.pi / 2 ** (t - j), 0.0, 0.0) for j in range(t)]
    elif case["circuit"] == "qaoa":
        # a ring and n random chords, one weight per round
        edges = [(q, (q + 1) % n) for q in range(n)]
        for _ in range(n):
            a = r.randrange(n)
            edges.append((a, (a + 1 + r.randrange(n - 1)) % n))
        gs += [(H, 0, q, 0.0, 0.0, 0.0) for q in range(n)]
        for _ in range(depth):
            g = ang()
            for a, b in edges:
                gs += [(CX, a, b, 0.0, 0.0, 0.0), (RZ, 0, b, g, 0.0, 0.0), (CX, a, b, 0.0, 0.0, 0.0)]
            beta = ang()
            gs += [(RX, 0, q, beta, 0.0, 0.0) for q in range(n)]
    else:
        for _ in range(depth):
            gs += [u3(q) for q in range(n)]
            gs += [(CX, q - 1, q, 0.0, 0.0, 0.0) for q in range(n - 1, 0, -1)]
        gs += [u3(q) for q in range(n)]
    return gs


def _diag_gates(r, n, count):
    """count P (half of them) and CP gates on random qubits: (sel0, sel1, theta)."""
    out = []
    for _ in range(count):
        a = r.randrange(n)
        b = (a + 1 + r.randrange(n - 1)) % n
        out.append((1 << a, K.NO_SEL if r.random() < 0.5 else 1 << b, r.uniform(0.0, TWO_PI)))
    return out


def _layer(case, seed):
    """Targets and unitaries of n // 5 blocks, the diagonal batch, the (controls, target) cascade."""
    r = random.Random(seed * 6271 + 3)
    g = np.random.default_rng(seed)
    n = case["n"]
    order = list(range(n))
    r.shuffle(order)
    blocks = []
    for b in range(n // 5):
        z = g.standard_normal((32, 32)) + 1j * g.standard_normal((32, 32))
        q, rr = np.linalg.qr(z)
        blocks.append((order[5 * b:5 * b + 5], q * (np.diag(rr) / np.abs(np.diag(rr)))[None, :]))
    cascade = []
    for _ in range(case["mcx"]):
        qs = r.sample(range(n), 3 + r.randrange(5))
        cascade.append((sum(1 << q for q in qs[1:]), qs[0]))
    return blocks, _diag_gates(r, n, case["gates"]), cascade


def _terms(r, n, count):
    """Z and ZZ terms with N(0, 1) coefficients."""
    out = []
    for _ in range(count):
        a = r.randrange(n)
        b = (a + 1 + r.randrange(n - 1)) % n
        out.append((r.gauss(0.0, 1.0), a) if r.random() < 0.5 else (r.gauss(0.0, 1.0), min(a, b), max(a, b)))
    return out


def _sets(case, seed):
    """(qubits, layers, terms, parameters) of each circuit of a batch."""
    # widths and depths belong to the workload, angles and terms to the seed
    shape = random.Random(case["sets"] * 131 + case["lo"])
    r = random.Random(seed * 131 + 5)
    out = []
    for _ in range(case["sets"]):
        n, layers = shape.randint(case["lo"], case["hi"]), shape.randint(case["dlo"], case["dhi"])
        out.append((n, layers, _terms(r, n, case["terms"]), _angles(r, 2 * n * layers)))
    return out


def _angles(r, count):
    return np.array([r.uniform(-math.pi, math.pi) for _ in range(count)])


def _amplitudes(case, seed):
    """A normalised random state as 2^n rows (re, im), in the case's precision."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dt = torch.float32 if case["c64"] else torch.float64
    x = torch.empty(1 << case["n"], 2, dtype=dt, device="cuda").normal_(generator=g)
    return x.mul_(1.0 / torch.linalg.vector_norm(x).item())


def _prec(case):
    return "c64" if case["c64"] else "c128"


class _Memory:
    """A simulator's device state, as torch takes it over without a copy.  The
    tensor holds this object and with it the simulator that owns the memory."""

    def __init__(self, sim, ptr, rows, c64):
        self.sim = sim
        self.__cuda_array_interface__ = {"shape": (rows, 2), "typestr": "<f4" if c64 else "<f8", "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(sim, case):
    ptr, m = sim.device_state()
    return torch.as_tensor(_Memory(sim, ptr, 1 << m, case["c64"]), device="cuda")


def prepare(case, seed):
    Z.init()
    kind = case["kind"]
    s = {"case": case}
    if kind == "circ":
        sim = Z.ZXH(case["n"], False, case["plain"], precision=_prec(case))
        sim.gates(_gates(case, seed))
        sim.set_seed(seed)
        s["sim"] = sim
    elif kind == "sample":
        sim = Z.ZXH(case["n"], False, True, precision=_prec(case))
        sim.execute()
        sim.set_seed(seed)
        _view(sim, case).copy_(_amplitudes(case, seed))
        s["sim"] = sim
    elif kind in ("diag", "layer"):
        s["psi"] = _amplitudes(case, seed)
        s["state"] = K.DeviceState.wrap(s["psi"].data_ptr(), case["n"], _prec(case))
        if kind == "diag":
            gs = _diag_gates(random.Random(seed), case["n"], case["gates"])
            s["gates"] = [np.array([g[0] for g in gs], dtype=np.uint64), np.array([g[1] for g in gs], dtype=np.uint64),
                          np.array([g[2] for g in gs])]
        else:
            s["layer"] = _layer(case, seed)
    elif kind == "grad":
        r = random.Random(seed)
        ops, count = A.two_local(case["n"], case["depth"])
        a = A.Ansatz(case["n"], ops, count, _prec(case))
        a.set_observable(_terms(r, case["n"], case["terms"]))
        s["ansatz"] = a
        s["params"] = _angles(r, count)
        if not case["c64"]:
            s["theta"] = torch.tensor(s["params"], dtype=torch.float64, requires_grad=True)
    else:
        b = A.AnsatzBatch(_prec(case))
        params = []
        for n, layers, terms, p in _sets(case, seed):
            ops, count = A.two_local(n, layers)
            b.add(n, ops, count, terms)
            params.append(p)
        b.finalize()
        s["batch"], s["params"] = b, np.concatenate(params)
    torch.cuda.synchronize()  # the engine works on streams of its own
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "circ":
        sim = state["sim"]
        sim.execute()
        if case["read"] == "state":
            return sim.get_state_array()
        out = {"state": _view(sim, case)}
        if case["read"] == "shots":
            sim.measure(case["shots"])
            out["bits"] = sim.results_bits()
        return out
    if kind == "sample":
        return state["sim"].sample_real(case["shots"]).astype(np.int64)
    if kind == "diag":
        state["state"].diag(*state["gates"])
        return state["psi"]
    if kind == "layer":
        st = state["state"]
        blocks, gates, cascade = state["layer"]
        for targets, u in blocks:
            st.block5(targets, u)
        st.diag([g[0] for g in gates], [g[1] for g in gates], [g[2] for g in gates])
        for controls, target in cascade:
            st.mcx(controls, target)
        return state["psi"]
    if kind == "grad":
        if "theta" in state:
            theta = state["theta"]
            theta.grad = None
            e = expectation(theta, state["ansatz"])
            e.backward()
            return {"energy": e.detach(), "grad": theta.grad}
        e, norm = state["ansatz"].forward(state["params"])
        g, _ = state["ansatz"].backward(state["params"])
        return {"energy": e, "norm": norm, "grad": g}
    e, norms, grads = state["batch"].run(state["params"])
    return {"energy": e, "norm": norms, "grad": np.concatenate(grads)}


def work(case):
    """Bytes of inputs and outputs, and the arithmetic of the gates: 14
    operations per amplitude for a U3 (two complex products and a sum per
    amplitude), 6 for a window of diagonal gates, 256 for a 5-qubit block."""
    kind = case["kind"]
    size = 8 if case["c64"] else 16
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for n, layers, terms, p in _sets(case, 0):
            w = work({"kind": "grad", "n": n, "depth": layers, "terms": case["terms"], "c64": case["c64"]})
            total = {k: total[k] + w[k] for k in total}
        return total
    n = case["n"]
    amps = float(1 << n)
    if kind == "circ":
        gates = _gates(case, 0)
        u3s = sum(g[0] in (U3, H, RX) for g in gates)
        windows = {"layers": case["depth"], "qft": n - 1, "qaoa": case["depth"], "su2": 0}[case["circuit"]]
        return {"bytes": size * amps + 8 * case["shots"], "flops": amps * (14 * u3s + 6 * windows)}
    if kind == "sample":
        return {"bytes": size * amps + 8 * case["shots"], "flops": 4 * amps}
    if kind == "diag":
        return {"bytes": 2 * size * amps, "flops": 6 * amps}
    if kind == "layer":
        return {"bytes": 2 * size * amps, "flops": amps * (256 * (n // 5) + 6)}
    # forward, the observable, and each gate undone on two states with its
    # two gradient entries (6 operations each)
    return {"bytes": 2 * size * amps, "flops": amps * case["depth"] * n * (14 * 3 + 12)}


def tolerance(case):
    """About four times the error against exact(): 1e-14 (twenty layers,
    complex128) and 4e-7 to 1e-6 (complex64) of a state, 4e-14 and 6e-7 of a
    gradient case's energy, a sum of terms that cancel and so the least exact
    of its outputs."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "circ":
        # a rounding of the state may move a shot across a boundary
        return {"rel": 5e-6 if case["c64"] else 1e-13, "max": 5e-5 if case["c64"] else 2e-12, "differ": 1e-3}
    if kind in ("diag", "layer"):
        return {"rel": 3e-6 if case["c64"] else 1e-13, "max": 3e-5 if case["c64"] else 2e-12}
    return {"rel": 2e-5 if case["c64"] else 1e-12, "max": 2e-4 if case["c64"] else 1e-11}


# ---- the same in 64 bits, in plain torch ----

def _apply(psi, n, q, u):
    """A 2x2 matrix on address bit q of a complex128 state, in place."""
    v = psi.view(1 << (n - 1 - q), 2, 1 << q)
    a, b = v[:, 0], v[:, 1]
    new = a * u[0] + b * u[1]
    v[:, 1].mul_(u[3]).add_(a, alpha=u[2])
    v[:, 0].copy_(new)


def _phase(psi, n, qs, theta):
    """exp(i theta) on the amplitudes whose bits qs (one or two) are all one."""
    p = complex(math.cos(theta), math.sin(theta))
    if len(qs) == 1:
        psi.view(1 << (n - 1 - qs[0]), 2, 1 << qs[0])[:, 1].mul_(p)
        return
    hi, lo = max(qs), min(qs)
    psi.view(1 << (n - 1 - hi), 2, 1 << (hi - 1 - lo), 2, 1 << lo)[:, 1, :, 1].mul_(p)


def _u3(theta, lam, phi):
    c, s = math.cos(theta / 2), math.sin(theta / 2)
    e = lambda t: complex(math.cos(t), math.sin(t))  # noqa: E731
    return [complex(c), -e(lam) * s, e(phi) * s, e(phi + lam) * c]


def _flip(psi, n, controls, target):
    """Swap the amplitudes of address bit target where every control bit is one."""
    dims = sorted(set(controls) | {target}, reverse=True)
    shape, at = [], n
    for d in dims:
        shape += [1 << (at - 1 - d), 2]
        at = d
    v = psi.view(shape + [1 << at])
    i0, i1 = [], []
    for d in dims:
        i0 += [slice(None), 1 if d in controls else 0]
        i1 += [slice(None), 1]
    a = v[tuple(i0)].clone()
    v[tuple(i0)] = v[tuple(i1)]
    v[tuple(i1)] = a


def _exact_circuit(case, seed):
    """The virtual state, its global phase, and the affine address map
    (rows, b, width) of the default mode: a qubit gets a new address bit at
    its first U3 unless a combination of the present bits already flips it
    alone."""
    n = case["n"]
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1.0
    rows, b, m = [0] * n, [0] * n, 0
    if case["plain"]:
        rows, m = [1 << q for q in range(n)], n
    turn = 0.0
    for code, cq, q, th, la, ph in _gates(case, seed):
        if code in (H, U3, RX):
            if code == H:
                th, la, ph = math.pi / 2, math.pi, 0.0
            elif code == RX:
                la, ph = math.pi / 2, -math.pi / 2
            if not case["plain"] and not _spans(rows, m, q):
                rows[q] |= 1 << m
                m += 1
            _apply(psi, n, q, _u3(th, la, ph))
        elif code == CX:
            if not case["plain"] or cq != q:
                rows[q] ^= rows[cq]
                b[q] ^= b[cq]
            _flip(psi, n, [cq], q)
        elif code == CP:
            _phase(psi, n, [cq, q], th)
        else:
            _phase(psi, n, [q], th)
            if code == RZ:
                turn -= 0.5 * th
    return psi, complex(math.cos(turn), math.sin(turn)), rows, b, m


def _spans(rows, m, q):
    """Whether some combination of the m address bits flips qubit q alone
    (e_q is in the span of the columns): no combination of the rows that
    takes in row q is zero."""
    basis = {}
    for k, r in enumerate(rows):
        if k == q:
            continue
        while r:
            top = r.bit_length() - 1
            if top not in basis:
                basis[top] = r
                break
            r ^= basis[top]
    r = rows[q]
    while r:
        top = r.bit_length() - 1
        if top not in basis:
            return True
        r ^= basis[top]
    return False


def _addressed(psi, rows, b, m):
    """psi_phys[x] = psi_virt[A x ^ b], a slice at a time."""
    n = len(rows)
    out = torch.empty(1 << m, dtype=torch.complex128, device="cuda")
    step = min(1 << m, 1 << 24)
    const = sum(b[q] << q for q in range(n))
    cols = [sum(((rows[q] >> c) & 1) << q for q in range(n)) for c in range(m)]
    for x0 in range(0, 1 << m, step):
        x = torch.arange(x0, x0 + step, dtype=torch.int64, device="cuda")
        v = torch.full_like(x, const)
        for c in range(m):
            v ^= ((x >> c) & 1) * cols[c]
        out[x0:x0 + step] = psi[v]
    return out


def _grad(n, layers, terms, params):
    """Energy, norm and gradient of the two-local ansatz (RY, RZ on every
    qubit, then the CZ chain), undoing the gates one qubit at a time."""
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1.0
    sign = torch.ones(1 << n, dtype=torch.float64, device="cuda")
    for q in range(n - 1):
        sign.view(1 << (n - 2 - q), 2, 2, 1 << q)[:, 1, 1].mul_(-1.0)

    def mats(k):
        t, f = params[k] / 2, params[k + 1] / 2
        c, s = math.cos(t), math.sin(t)
        z = complex(math.cos(f), math.sin(f))
        return np.array([[c, -s], [s, c]], dtype=complex), np.diag([z.conjugate(), z])
    k = 0
    for _ in range(layers):
        for q in range(n):
            ry, rz = mats(k)
            _apply(psi, n, q, [complex(v) for v in (rz @ ry).reshape(-1)])
            k += 2
        psi.mul_(sign)
    diag = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
    for t in terms:
        if len(t) == 2:
            v = diag.view(1 << (n - 1 - t[1]), 2, 1 << t[1])
            v[:, 0] += t[0]
            v[:, 1] -= t[0]
        else:
            v = diag.view(1 << (n - 1 - t[2]), 2, 1 << (t[2] - 1 - t[1]), 2, 1 << t[1])
            v[:, 0, :, 0] += t[0]
            v[:, 1, :, 1] += t[0]
            v[:, 0, :, 1] -= t[0]
            v[:, 1, :, 0] -= t[0]
    lam = psi * diag
    del diag
    energy, norm = torch.vdot(psi, lam).real.item(), torch.vdot(psi, psi).real.item()
    grad = torch.zeros(len(params), dtype=torch.float64)
    y = np.array([[0, -1j], [1j, 0]])
    for _ in range(layers):
        psi.mul_(sign)
        lam.mul_(sign)
        for q in range(n - 1, -1, -1):
            k -= 2
            ry, rz = mats(k)
            shape = (1 << (n - 1 - q), 2, 1 << q)
            p, l = psi.view(shape), lam.view(shape)
            # <lam| |a><b| |psi> on qubit q: dE/dtheta = Im <lam| G |psi>
            m = np.array([[_dot(l[:, i], p[:, j]) for j in range(2)] for i in range(2)])
            grad[k] = float(np.sum((rz @ y @ rz.conj().T) * m).imag)
            grad[k + 1] = float((m[0, 0] - m[1, 1]).imag)
            und = [complex(v) for v in (rz @ ry).conj().T.reshape(-1)]
            _apply(psi, n, q, und)
            _apply(lam, n, q, und)
    return energy, norm, grad


def _dot(a, b):
    return torch.vdot(a.reshape(-1), b.reshape(-1)).item()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # whole numbers
    if kind == "circ":
        n = case["n"]
        if n >= 28 and case["depth"] * n > 100:
            return None
        psi, turn, rows, b, m = _exact_circuit(case, seed)
        if case["read"] == "state":
            back = torch.arange(1 << n, dtype=torch.int64, device="cuda")
            rev = torch.zeros_like(back)
            for q in range(n):
                rev |= ((back >> q) & 1) << (n - 1 - q)
            return torch.view_as_real(psi[rev] * turn).cpu().numpy().reshape(-1).view(np.complex128)
        if not case["plain"]:
            psi = _addressed(psi, rows, b, m)
        out = {"state": torch.view_as_real(psi)}
        if case["read"] == "shots":
            out["bits"] = None
        return out
    if kind in ("diag", "layer"):
        n = case["n"]
        psi = torch.view_as_complex(_amplitudes(case, seed).double())
        if kind == "diag":
            blocks, gates, cascade = [], _diag_gates(random.Random(seed), n, case["gates"]), []
        else:
            blocks, gates, cascade = _layer(case, seed)
        for targets, u in blocks:
            # the targets' axes to the front, most significant index bit first
            axes = [n - 1 - t for t in reversed(targets)]
            rest = [a for a in range(n) if a not in axes]
            x = psi.view([2] * n).permute(axes + rest).reshape(32, -1)
            x = torch.from_numpy(u).cuda() @ x
            back = np.argsort(axes + rest).tolist()
            psi = x.view([2] * n).permute(back).reshape(-1)
        for s0, s1, th in gates:
            qs = [s0.bit_length() - 1] + ([] if s1 == K.NO_SEL else [s1.bit_length() - 1])
            _phase(psi, n, qs, th)
        for controls, target in cascade:
            _flip(psi, n, [q for q in range(n) if (controls >> q) & 1], target)
        return torch.view_as_real(psi)
    if kind == "grad":
        r = random.Random(seed)
        terms = _terms(r, case["n"], case["terms"])
        e, norm, g = _grad(case["n"], case["depth"], terms, _angles(r, 2 * case["n"] * case["depth"]))
        if case["c64"]:
            return {"energy": e, "norm": norm, "grad": g.numpy()}
        return {"energy": torch.tensor(e, dtype=torch.float64), "grad": g}
    if case["sets"] * (case["dlo"] + case["dhi"]) > 600 and case["hi"] > 20:
        return None  # over 20 seconds
    res = [_grad(n, layers, terms, p) for n, layers, terms, p in _sets(case, seed)]
    return {"energy": np.array([x[0] for x in res]), "norm": np.array([x[1] for x in res]),
            "grad": np.concatenate([x[2].numpy() for x in res])}
