"""GPU: the band-trimmed codes stored by the segment kernel itself, where a
block's threshold is known before its samples (FIXED, and REFERENCE once its slot
has latched), and those packed afterwards (PER_BLOCK, REFERENCE not yet latched),
over calls of two chunks, in every preset.

Expected: resample_f32 gives the same float samples, so every code is that of
v = x - offset in FP32, (|v| >= th | 2) ^ 3 (v < 0), with the threshold that the
policy defines from the block statistics.  No tolerance: the samples, the
difference and the comparison are the same FP32 operations."""
import sys

import numpy as np
import pytest

from sdbe_amd import synth as S

pytestmark = pytest.mark.gpu
SKIP = {6: 150, 8: 150, 10: 16, 11: 150}
NCH = 16384


def _codes(x, th, off):
    v = x - np.float32(off)
    c = ((np.abs(v) >= np.float32(th)) | np.uint32(2)) ^ np.where(v < 0, np.uint32(3), np.uint32(0))
    w = c.astype(np.uint32).reshape(-1, 16) << (2 * np.arange(16, dtype=np.uint32))
    return np.bitwise_or.reduce(w, axis=1)


@pytest.mark.parametrize("frac", [6, 8, 10, 11])
def test_codes_of_every_policy(frac):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd import _lib as L
    from sdbe_amd.stage import SdbeStage
    D = L.TRIM_PRESETS[frac][0]
    n = 3
    beng = torch.from_numpy(S.codes_to_beng_int8(S.gaussian_codes(S.rng_for(40 + frac), D * n))).cuda()
    blocks = beng.reshape(n, D, NCH, 2)

    def stage(policy, fixed=(1.0, 0.0)):
        return SdbeStage(rate_frac=frac, skip_mhz=SKIP[frac], policy=policy, out_mode=L.OUT_FRAMES, chunk=2,
                         max_spectra=n, fixed=fixed)

    st = stage(L.THRESH_PER_BLOCK)
    x, stats = st.resample_f32(blocks)
    x, stats = x.cpu().numpy(), stats.cpu().numpy()
    st.close()
    sig = float(stats[0, 1])
    for policy, fixed in ((L.THRESH_PER_BLOCK, (1.0, 0.0)), (L.THRESH_FIXED, (0.8 * sig, 0.25 * sig)),
                          (L.THRESH_FIXED, (0.0, 0.0)), (L.THRESH_REFERENCE, (1.0, 0.0))):
        st = stage(policy, fixed)
        # REFERENCE: block 0 latches in the first call (its second chunk finds it
        # latched, as the whole second call does); after a reset block 1 comes first
        for call, order in enumerate(([0, 1, 2], [2, 0, 1], [1, 2, 0])):
            if call == 2:
                st.reset_latch(0)
            print("[trim codes] %d/11 policy %d call %d" % (frac, policy, call), flush=True)
            sys.stdout.flush()
            out = st.process_spectra(blocks[order].contiguous()).cpu().numpy()
            pay = out[:, :, 32:].copy().view(np.uint32).reshape(n, -1)
            for i, b in enumerate(order):
                t, o = fixed if policy == L.THRESH_FIXED else (stats[b, 1], stats[b, 0])
                if policy == L.THRESH_REFERENCE:
                    t, o = stats[1 if call == 2 else 0, ::-1]
                assert np.array_equal(pay[i], _codes(x[b], np.float32(t), np.float32(o))), (frac, policy, call, i)
        st.close()
