"""Per-chunk coefficients of a diagonal window at the edge between the two
kernels that form them (1024 chunks: 20 or 21 address bits under the flat
sweep's 1024-unit chunks, and wider), with one gate, gates on low or high bits
only, and hundreds, against phases summed in numpy."""
import numpy as np
import pytest

from test_gpu_kernels import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n", [17, 18, 19, 20, 21, 22, 23])
@pytest.mark.parametrize("bits", ["all", "high", "low"])
def test_windows(gpu_engine, prec, n, bits):
    from zxh_adae_amd import kernels as K
    rng = np.random.default_rng(n)
    x = np.arange(1 << n, dtype=np.int64)
    lo, hi = {"all": (0, n), "high": (n - 6, n), "low": (0, 10)}[bits]
    for count in (1, 40, 300 if n == 20 else 7):
        s0, s1, th = [], [], []
        angle = np.zeros(1 << n)
        for _ in range(count):
            a, b = (int(q) for q in lo + rng.choice(hi - lo, 2, replace=False))
            pair = rng.random() < 0.6
            t = float(rng.uniform(-3, 3))
            s0.append(1 << a)
            s1.append(1 << b if pair else K.NO_SEL)
            th.append(t)
            on = (x >> a) & ((x >> b) if pair else 1) & 1
            angle += np.where(on, t, 0.0)
        psi = np.exp(1j * rng.uniform(0, 6, 1 << n))
        d = dev(gpu_engine, psi if prec == "c128" else psi.astype(np.complex64), prec)
        d.diag(s0, s1, th)
        want = psi * np.exp(1j * angle)
        # angles of a few hundred radians, sums of as many terms: 1e-13 each way
        assert np.max(np.abs(d.download() - want)) < (2e-12 if prec == "c128" else 1e-6)
