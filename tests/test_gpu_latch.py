"""GPU: the REFERENCE latch over a ragged batch with empty leading blocks
(software/aphids/vdif_inout_gpu_thread.cu:954-1005) equals the block-by-block
walk: each block-pol's payload is byte-identical to the same spectra under the
FIXED threshold the walk gives it, whatever the chunking, and the slots keep
what the walk leaves in them for the next call."""
import sys

import numpy as np
import pytest

from sdbe_amd import synth as S

pytestmark = pytest.mark.gpu
# (latch slot, empty blocks per polarisation 0 and 1): slot 5 is shared by two
# streams, whose first non-empty polarisation-0 block is in the second
STREAMS = [(5, (0, 1, 2), (0,)), (2, (), (0,)), (5, (), ()), (7, (0, 1), (0, 1))]
BLOCKS = [3, 1, 2, 2]


@pytest.mark.parametrize("chunk", [2, 6, 256])
def test_latch_equals_the_walk(chunk):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd import _lib as L
    from sdbe_amd.stage import BatchStream, SdbeStage, process_blocks
    rng = S.rng_for(91)
    data = []
    for nb, (_, e0, e1) in zip(BLOCKS, STREAMS):
        pols = []
        for empty in (e0, e1):
            x = S.codes_to_beng_int8(S.gaussian_codes(rng, 39 * nb, sigma=float(rng.uniform(0.5, 2.0)), quant_sigma=1.0))
            for b in empty:
                x[39 * b:39 * (b + 1)] = 0
            pols.append(torch.from_numpy(x).cuda())
        data.append(pols)
    flat = [(s, b, p) for s, nb in enumerate(BLOCKS) for b in range(nb) for p in (0, 1)]
    rows = [data[s][p][39 * b:39 * (b + 1)] for s, b, p in flat]
    st = SdbeStage(out_mode=L.OUT_PAYLOAD, chunk=2, max_spectra=len(flat))
    _, stats = st.resample_f32(torch.stack(rows))
    stats = stats.cpu().numpy()
    st.close()
    st = SdbeStage(out_mode=L.OUT_PAYLOAD, chunk=chunk, max_spectra=1)
    slots = {}
    for call in range(2):
        outs = [torch.zeros((2, 64 * nb, 8192), dtype=torch.uint8, device="cuda") for nb in BLOCKS]
        process_blocks(st, [BatchStream(d[0], d[1], o, policy=L.THRESH_REFERENCE, latch_slot=v[0])
                            for d, o, v in zip(data, outs, STREAMS)])
        for i, (s, b, p) in enumerate(flat):
            slot = STREAMS[s][0]
            cur = slots.get(slot, (np.float32(0), np.float32(0)))
            if cur[0] == 0 and p == 0:
                cur = slots[slot] = (np.float32(stats[i][1]), np.float32(stats[i][0]))
            one = SdbeStage(policy=L.THRESH_FIXED, fixed=(float(cur[0]), float(cur[1])), out_mode=L.OUT_PAYLOAD,
                            chunk=2, max_spectra=1)
            want = one.process_spectra(rows[i].reshape(1, 39, 16384, 2))
            print("[latch] chunk %d call %d stream %d block %d pol %d th %g" % (chunk, call, s, b, p, cur[0]), flush=True)
            sys.stdout.flush()
            assert torch.equal(outs[s][p, 64 * b:64 * (b + 1)], want[0])
            one.close()
    st.close()
