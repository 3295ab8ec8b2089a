"""GPU: sdbe_unpack_group_int8 writes the caller's rows directly when they are
16-byte aligned and overlap nothing, and through the handle's rows otherwise.
Both routes, and packets at an offset of 4 bytes (word loads in place of
16-byte ones), give the oracle's rows, bitmap and unique count (bit-exact), in
either packet geometry."""
import ctypes as C
import sys

import numpy as np
import pytest

from oracle import sdbe_oracle as O
from sdbe_amd import synth as S

pytestmark = pytest.mark.gpu
FRAMES = 13


@pytest.mark.parametrize("geometry", [0, 1])
def test_unpack_rows_routes(geometry):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from sdbe_amd import _lib as L
    from sdbe_amd.stage import SdbeStage
    groups, _ = S.make_group_packets(77 + geometry, n_groups=1, drop_frac=0.01, frames=FRAMES, geometry=geometry)
    pk, b0 = groups[0]
    want = (O.vdif_to_beng_8x1024 if geometry else O.vdif_to_beng)(pk, b0, FRAMES)
    rows = [np.ascontiguousarray(x).reshape(-1).view(np.uint8) for x in want.beng]
    n_bytes = rows[0].size
    st = SdbeStage(rate_frac=8, skip_mhz=150, chunk=2, max_spectra=1, packet_geometry=geometry)
    raw = torch.from_numpy(pk.view(np.uint8).reshape(-1)).cuda()

    def call(p_pk, p0, p1):
        L.check(st.lib.sdbe_unpack_group_int8(st.h, C.c_void_p(p_pk), pk.shape[0], b0, C.c_void_p(p0),
                                              C.c_void_p(p1), None, None), "unpack", st.h)
        assert st.stats()["n_unique"] == pk.shape[0]

    def check(name, a, b):
        print("[unpack] geometry %d %s" % (geometry, name), flush=True)
        sys.stdout.flush()
        assert np.array_equal(a.cpu().numpy(), rows[0]) and np.array_equal(b.cpu().numpy(), rows[1]), name

    buf = torch.zeros(2 * n_bytes + 64, dtype=torch.uint8, device="cuda")
    for off in (0, 4, 8):       # 4, 8: the rows are not 16-byte aligned
        buf.zero_()
        call(raw.data_ptr(), buf.data_ptr() + off, buf.data_ptr() + off + n_bytes)
        check("rows at +%d" % off, buf[off:off + n_bytes], buf[off + n_bytes:off + 2 * n_bytes])
    shifted = torch.zeros(raw.numel() + 16, dtype=torch.uint8, device="cuda")
    shifted[4:4 + raw.numel()] = raw
    buf.zero_()
    call(shifted.data_ptr() + 4, buf.data_ptr(), buf.data_ptr() + n_bytes)
    check("packets at +4", buf[:n_bytes], buf[n_bytes:2 * n_bytes])
    # the packets lie where the rows of polarisation 0 go
    buf.zero_()
    buf[:raw.numel()] = raw
    call(buf.data_ptr(), buf.data_ptr() + 32, buf.data_ptr() + 32 + n_bytes)
    check("rows over the packets", buf[32:32 + n_bytes], buf[32 + n_bytes:32 + 2 * n_bytes])
    st.close()
