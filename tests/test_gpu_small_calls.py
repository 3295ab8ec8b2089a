"""GPU: the launch shapes of small calls (stage C2's rows one by one, fewer
stage-C1 tiles per workgroup) give the bytes of the large call's shapes, in
every FFT mode: each block-pol of a call of n equals the same block-pol of a
call of 33, which runs its rows in pairs, payload and headers (PER_BLOCK
thresholds; no tolerance, the arithmetic per block-pol is the same)."""
import sys

import pytest

from sdbe_amd import synth as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,sizes", [(0, (1, 2, 3, 4, 5, 8, 9, 12, 20, 23, 24, 25)), (1, (1, 9)), (2, (1,)),
                                             (3, (1, 9))])
def test_small_call_equals_large_call(precision, sizes):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd import _lib as L
    from sdbe_amd.stage import SdbeStage
    n = 33
    x = torch.from_numpy(S.codes_to_beng_int8(S.gaussian_codes(S.rng_for(12), 39 * n))).cuda().reshape(n, 39, 16384, 2)

    def run(k):
        st = SdbeStage(policy=L.THRESH_PER_BLOCK, out_mode=L.OUT_FRAMES, chunk=k + (k & 1), max_spectra=k,
                       fft_precision=precision)
        st.set_state(secs=5, df=124000, ref_epoch=30, psn=7)
        out = st.process_spectra(x[:k].contiguous())
        torch.cuda.synchronize()
        st.close()
        return out

    want = run(n)
    for k in sizes:
        print("[small] precision %d, %d block-pols" % (precision, k), flush=True)
        sys.stdout.flush()
        assert torch.equal(run(k), want[:k])
