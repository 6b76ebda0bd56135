"""The sampler's descent, its pieces and its packing at their edges, exact
against the oracle: segments below, at and above the lowest stored tree level,
one segment, 4096 and 8192 segments (the single-workgroup tails and the
general ones), draws of one shot, one piece (2^17) and just over, virtual
words of up to and over 64 qubits."""
import numpy as np
import pytest

import oracle_py as O
from zxh_adae_amd import kernels as K

pytestmark = pytest.mark.gpu


def state(m, prec, seed):
    rng = np.random.default_rng(seed)
    psi = rng.normal(size=1 << m) + 1j * rng.normal(size=1 << m)
    psi[rng.random(psi.size) < 0.4] = 0
    if m:
        psi[: 1 << (m - 1)][rng.random(1 << (m - 1)) < 0.5] *= 1e-9
    return psi.astype(np.complex64 if prec == "c64" else np.complex128)


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("m,seg,shots", [(1, 1, 50), (2, 18, 50), (5, 3, 300), (6, 4, 300), (7, 5, 300), (8, 6, 1),
                                         (13, 18, 4096), (14, 2, 131072), (15, 2, 131073), (17, 5, 300000),
                                         (18, 18, 20000), (19, 18, 20000)])
def test_draws(gpu_engine, m, seg, shots, prec):
    psi = state(m, prec, 10 * m + seg)
    d = K.DeviceState(m, prec)
    d.upload(psi)
    want = O.oracle_sample_state(psi.astype(np.complex128), seg, O.mix_seed(m, 0), shots)
    assert np.array_equal(d.sample(seg, O.mix_seed(m, 0), shots), want)
    # the segments' values are those of the kernel-level measure as well
    for nq in (1, 64, 65, 130):
        rng = np.random.default_rng(nq)
        rows = rng.integers(0, 1 << m, size=nq, dtype=np.uint64)
        b = rng.integers(0, 2, size=nq).astype(np.uint8)
        packed, real = d.measure(seg, rows, b, shots, seed=m)
        assert np.array_equal(real, want)
        for q in {0, nq - 1, nq // 2}:
            par = np.zeros(shots, dtype=np.uint64)
            for c in range(m):
                if (int(rows[q]) >> c) & 1:
                    par ^= (real >> np.uint64(c)) & np.uint64(1)
            got = (packed[:, q >> 6] >> np.uint64(q & 63)) & np.uint64(1)
            assert np.array_equal(got, par ^ np.uint64(b[q])), (nq, q)
    d.free()
