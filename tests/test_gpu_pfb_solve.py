"""GPU: sdbe_pfb_inverse at the edges of its solve (one row to one past a span
of 32, a block of 256 rows and 16 blocks) against scipy's banded FP64 solver on
a sample of branches: x = P^T (P P^T)^-1 yh, yh from the FP64 inverse FFT.  Bar:
SNR >= 90 dB, that of test_gpu_pfb (the FP32 C2R, amplified by the solve's
conditioning).  A prototype with two zeros together on the unit circle takes
the factor-row kernels; its amplification of the FP32 rounding of yh is about
(rows / pi)^2, so its bar is 20 log10(10^6 / rows^2) dB."""
import math
import sys

import numpy as np
import pytest
from scipy.linalg import solveh_banded

from oracle import sdbe_oracle as O

pytestmark = pytest.mark.gpu
LB = 32768
BRANCHES = np.array([0, 1, 4044, 8000, 8001, 12288, 16383, 16384, 16390, 24000, 28724, 32766, 32767])


def _window(kind):
    if kind == "triangle":
        return np.repeat([1.0, 2.0, 1.0, 0.0], LB).astype(np.float32)
    return (O.pfb_window_hann_sinc() if kind == "hann_sinc" else O.pfb_window_hamming()).astype(np.float32)


@pytest.mark.parametrize("kind,n", [(k, n) for k in ("hann_sinc", "hamming")
                                    for n in (1, 2, 3, 31, 32, 33, 255, 256, 257, 289, 511, 4096, 4097)]
                         + [("triangle", 20), ("triangle", 300)])
def test_inverse_edges(kind, n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd.pfb import Pfb
    w = _window(kind)
    g = torch.Generator(device="cuda").manual_seed(n)
    spec = torch.view_as_complex(torch.randn((n, LB // 2 + 1, 2), generator=g, device="cuda"))
    spec.imag[:, 0] = 0.0
    spec.imag[:, -1] = 0.0
    p = Pfb(w, max_spectra=n)
    print("[pfb] inverse %s n=%d" % (kind, n), flush=True)
    sys.stdout.flush()
    got = p.inverse(spec).reshape(n + 3, LB)[:, torch.from_numpy(BRANCHES).cuda()].cpu().numpy().astype(np.float64)
    p.close()
    yh = np.empty((n, BRANCHES.size))
    for s in range(0, n, 256):
        yh[s:s + 256] = np.fft.irfft(spec[s:s + 256].cpu().numpy().astype(np.complex128), n=LB, axis=1)[:, BRANCHES]
    taps = w.reshape(4, LB).astype(np.float64)
    want = np.zeros((n + 3, BRANCHES.size))
    for i, b in enumerate(BRANCHES):
        t = taps[:, b]
        band = np.zeros((min(4, n), n))
        for d in range(min(4, n)):
            band[d, :n - d] = (t[d:] * t[:4 - d]).sum()
        z = solveh_banded(band, yh[:, i], lower=True)
        for k in range(4):
            want[k:k + n, i] += t[k] * z
    snr = 10.0 * math.log10(np.sum(want ** 2) / max(np.sum((got - want) ** 2), 1e-300))
    print("[pfb] inverse %s n=%d: %.1f dB" % (kind, n, snr), flush=True)
    assert snr >= (90.0 if kind != "triangle" else 20.0 * math.log10(1e6 / n ** 2))
