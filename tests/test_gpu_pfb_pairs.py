"""GPU: sdbe_pfb_forward takes spectra two at a time above one per CU (an odd
count leaves a single one): at and around 256, 512 and 513 spectra against the
FP64 oracle, SNR >= 120 dB (FP32 FFT rounding, the bar of test_gpu_pfb); and the
persistent inverse FFT's rows at the same counts, through forward(inverse) >=
100 dB on spectra that are a PFB's own."""
import math
import sys

import numpy as np
import pytest

from oracle import sdbe_oracle as O

pytestmark = pytest.mark.gpu
LB = 32768


def _snr(ref, got):
    return 10.0 * math.log10(np.sum(np.abs(ref) ** 2) / max(np.sum(np.abs(got - ref) ** 2), 1e-300))


@pytest.mark.parametrize("n", [255, 256, 257, 258, 511, 513])
def test_forward_pairs(n):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd.pfb import Pfb
    w = O.pfb_window_hann_sinc().astype(np.float32)
    x = np.random.default_rng(n).normal(size=(n + 3) * LB).astype(np.float32)
    p = Pfb(w, max_spectra=n)
    spec = p.forward(torch.from_numpy(x).cuda())
    got = spec.cpu().numpy().astype(np.complex128)
    taps, seg = w.reshape(4, LB).astype(np.float64), x.reshape(n + 3, LB).astype(np.float64)
    worst = min(_snr(np.fft.rfft(sum(taps[k] * seg[i + k] for k in range(4))), got[i]) for i in range(n))
    back = p.forward(p.inverse(spec)).cpu().numpy().astype(np.complex128)
    again = _snr(got, back)
    p.close()
    print("[pfb] n=%d: worst spectrum %.1f dB, forward(inverse) %.1f dB" % (n, worst, again), flush=True)
    sys.stdout.flush()
    assert worst >= 120.0 and again >= 100.0
