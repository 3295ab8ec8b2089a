"""GPU: sdbe_pfb_inverse against 80-bit banded Cholesky, branch by branch, for
prototypes on both sides of the rule that admits a plan to the constant-coefficient
solve: smooth windows with two or three zeros together near z = -1, whose solve
amplifies rounding, and flat taps of the same kind.

The spectra hold bin 0 only, a float per row, so that the inverse FFT gives that
float / 32768 in every branch without rounding, and the solve alone is compared.
Bar, of a branch's rms: 2^-24, what FP32 rounding of the samples may be, and 2^-26 of
the solve's own; for prototypes that may go to the FP64 factor rows, 8 x 2^-53 times
the condition of P P^T where that is more than 2^-26."""
import sys

import numpy as np
import pytest
from scipy.linalg import eigvals_banded

from oracle import sdbe_oracle as O

pytestmark = pytest.mark.gpu
LB = 32768


def _window(kind):
    m = 4 * LB - 1
    k = np.arange(4 * LB, dtype=np.float64)
    u = 2.0 * k / m - 1.0
    name, _, par = kind.partition(" ")
    if name == "hann_sinc":
        w = O.pfb_window_hann_sinc()
    elif name == "hamming":
        w = O.pfb_window_hamming()
    elif name == "gauss":
        w = np.exp(-0.5 * ((k - m / 2.0) / (float(par) * LB)) ** 2)
    elif name == "kaiser":
        w = np.i0(float(par) * np.sqrt(1.0 - u * u)) / np.i0(float(par))
    elif name == "triangle":
        w = float(par) + (1.0 - float(par)) * (1.0 - np.abs(u))
    else:
        w = np.repeat([float(t) for t in par.split()], LB)
    return w.astype(np.float32)


def _solve(taps, y):
    """x = P^T (P P^T)^-1 y for all columns of taps [4][b], in long double."""
    t = taps.astype(np.longdouble)
    n, b = len(y), taps.shape[1]
    a = [(t[d:] * t[:4 - d]).sum(0) for d in range(4)]
    L = np.zeros((n, 4, b), dtype=np.longdouble)       # L(i, i - d)
    u = np.zeros((n, b), dtype=np.longdouble)
    for i in range(n):
        r = np.full(b, y[i], dtype=np.longdouble)
        for d in range(min(i, 3), -1, -1):
            s = a[d].copy()
            for k in range(max(i - 3, 0), i - d):
                s -= L[i, i - k] * L[i - d, i - d - k]
            L[i, d] = s / L[i - d, 0] if d else np.sqrt(s)
            if d:
                r -= L[i, d] * u[i - d]
        u[i] = r / L[i, 0]
    for i in range(n - 1, -1, -1):
        for d in range(1, min(4, n - i)):
            u[i] -= L[i + d, d] * u[i + d]
        u[i] /= L[i, 0]
    x = np.zeros((n + 3, b), dtype=np.longdouble)
    for k in range(4):
        x[k:k + n] += t[k] * u
    return x


def _condition(taps, n):
    t = taps.astype(np.float64)
    out = []
    for b in range(t.shape[1]):
        band = np.zeros((min(4, n), n))
        for d in range(min(4, n)):
            band[d, :n - d] = (t[d:, b] * t[:4 - d, b]).sum()
        lo = eigvals_banded(band, lower=True, select="i", select_range=(0, 0))[0]
        # the smallest eigenvalue is known to the rounding of the largest; at 1 / eps there is no digit left
        out.append(min(np.abs(t[:, b]).sum() ** 2 / max(lo, 1e-300), 2.0 ** 53))
    return np.array(out)


@pytest.mark.parametrize("kind,exact,rows", [
    ("hann_sinc", True, (1, 2, 3, 33, 255, 256, 257, 511, 4097)),
    ("hamming", True, (1, 2, 3, 20, 31, 32, 33, 64, 128, 225, 255, 256, 257, 289, 511, 512, 1000, 4096, 4097)),
    ("kaiser 5", True, (128, 300)),
    ("gauss 0.954", False, (64, 128, 300, 512)),
    ("gauss 0.955", False, (64, 256, 512)),
    ("kaiser 4.27", False, (64, 255, 512)),
    ("triangle 0.001", False, (255, 512)),
    ("flat 0.3334 1 1 0.3334", False, (300,)),
    ("flat 1 1 1 0.5", True, (3, 300)),
])
def test_inverse_of_prototype(kind, exact, rows):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd.pfb import Pfb
    w = _window(kind)
    if kind.startswith("flat"):
        branches = np.array([0, 1, LB - 1])
    else:
        branches = np.unique(np.concatenate([np.arange(0, LB, 1171), [LB - 1], 4036 + np.arange(-64, 65, 32),
                                             28731 + np.arange(-64, 65, 32), 16384 + np.arange(-1200, 1201, 150)]))
    taps = w.reshape(4, LB)[:, branches]
    idx = torch.from_numpy(branches).cuda()
    for n in rows:
        y = np.random.default_rng(n).normal(size=n).astype(np.float32)
        spec = torch.zeros((n, LB // 2 + 1), dtype=torch.complex64, device="cuda")
        spec.real[:, 0] = torch.from_numpy(y).cuda()
        p = Pfb(w, max_spectra=n)
        print("[pfb] inverse %s n=%d" % (kind, n), flush=True)
        sys.stdout.flush()
        got = p.inverse(spec).reshape(n + 3, LB)[:, idx].cpu().numpy().astype(np.longdouble)
        p.close()
        want = _solve(taps, y) / LB
        err = np.sqrt(((got - want) ** 2).sum(0) / (want ** 2).sum(0)).astype(np.float64)
        bar = np.full(len(branches), 2.0 ** -26)
        if not exact:
            bar = np.maximum(bar, 8.0 * 2.0 ** -53 * _condition(taps, n))
        i = (err / (2.0 ** -24 + bar)).argmax()
        print("[pfb] inverse %s n=%d: worst branch %d, %.2e (bar %.2e)" % (kind, n, branches[i], err[i],
                                                                         2.0 ** -24 + bar[i]), flush=True)
        assert (err <= 2.0 ** -24 + bar).all()
