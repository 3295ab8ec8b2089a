"""GPU: the cross-power tiles of sdbe_xcorr_search at their edges (4-wide tiles
below 36 offsets, 12-wide ones with a 4-wide rest from there on; averages below,
at and past a multiple of the tile width) against the FP64 oracle: lag functions
within 2e-5, peaks and standard deviations within 1e-4 relative (the bars of
test_gpu_xcorr: FP32 transforms of normalised values)."""
import sys

import numpy as np
import pytest

from oracle import sdbe_oracle as O

pytestmark = pytest.mark.gpu
LW = 32768


@pytest.mark.parametrize("n_off,avg", [(1, 1), (4, 3), (5, 4), (63, 5), (64, 16), (65, 17), (79, 15)])
def test_cross_tiles(n_off, avg):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd.qa import XCorr
    nw = n_off + avg + 1
    rng = np.random.default_rng(1000 * n_off + avg)
    common = rng.normal(size=(nw + 1) * LW)
    x0 = (common[LW:] + 0.5 * rng.normal(size=nw * LW)).astype(np.float32)
    x1 = (common[LW - 37:-37] + 0.5 * rng.normal(size=nw * LW)).astype(np.float32)
    first = -(n_off // 2)
    xc = XCorr(max_windows=n_off + avg - 1, max_offsets=n_off)
    print("[xcorr] %d offsets of %d windows" % (n_off, avg), flush=True)
    sys.stdout.flush()
    s, peak, std = (v.cpu().numpy() for v in xc.search(torch.from_numpy(x0).cuda(), torch.from_numpy(x1).cuda(),
                                                       first, n_off, avg))
    so, _, po = O.corr_Xt_search(O.corr_spectra(x0.astype(np.float64)), O.corr_spectra(x1.astype(np.float64)),
                                 range(first, first + n_off), search_avg=avg)
    assert np.abs(s - so).max() <= 2e-5
    assert np.allclose(peak, po, rtol=1e-4) and np.allclose(std, so.std(axis=1), rtol=1e-4)
    xc.close()


@pytest.mark.parametrize("n_off,avg", [(35, 12), (36, 1), (36, 11), (37, 12), (41, 13), (47, 25)])
def test_cross_tiles_first_wide(n_off, avg):
    test_cross_tiles(n_off, avg)
