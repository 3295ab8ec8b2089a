"""CPU: the PFB inverse's constant-coefficient solve
(sdbe_amd/csrc/sdbe_pfb_solve.hpp), built for the host one branch at a time
(pfb_solve_host.cpp), over the prototypes it can be asked to solve: which of them a
plan admits to it, the minimum-phase factor, and the error of the solve against 80
bits where it is admitted.  Bar for the error: 2^-26, a quarter of the FP32 rounding
of a sample (2^-24), or the error of FP64 banded Cholesky on the same rows."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import sdbe_oracle as O

LB = 32768
ROWS = (1, 2, 3, 20, 31, 32, 33, 64, 128, 225, 255, 256, 257, 300, 511, 512, 1000, 4097)
BLOCKS = 17                                           # of 256 rows: plans of up to 4352


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    so = tmp_path_factory.mktemp("pfb") / "pfb_solve_host.so"
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-o", str(so),
                    str(Path(__file__).with_name("pfb_solve_host.cpp"))], check=True, capture_output=True)
    lib = C.CDLL(str(so))
    lib.factor_error.restype = C.c_double
    return lib


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _admitted(host, taps, blocks=BLOCKS):
    taps = np.ascontiguousarray(taps, dtype=np.float32)
    out = np.zeros(len(taps), dtype=np.int32)
    host.admit(len(taps), _p(taps), blocks, _p(out))
    return out.astype(bool)


def _check_errors(host, taps, rows, what):
    taps = np.ascontiguousarray(taps, dtype=np.float32)
    for n in rows:
        y = np.random.default_rng(n).normal(size=n).astype(np.float32)
        e = np.zeros(2)
        host.errors(_p(taps), n, _p(y), BLOCKS, _p(e))
        assert e[0] <= max(2.0 ** -26, e[1]), (what, n, e)


def _window(kind):
    m = 4 * LB - 1
    k = np.arange(4 * LB, dtype=np.float64)
    u = 2.0 * k / m - 1.0
    name, _, par = kind.partition(" ")
    if name == "hann_sinc":
        w = O.pfb_window_hann_sinc()
    elif name == "hamming":
        a = float(par or 0.54)
        w = O.pfb_window_hamming() if not par else a - (1.0 - a) * np.cos(2.0 * np.pi * k / m)
    elif name == "gauss":
        w = np.exp(-0.5 * ((k - m / 2.0) / (float(par) * LB)) ** 2)
    elif name == "kaiser":
        w = np.i0(float(par) * np.sqrt(1.0 - u * u)) / np.i0(float(par))
    elif name == "triangle":
        w = float(par) + (1.0 - float(par)) * (1.0 - np.abs(u))
    else:
        w = np.repeat([float(t) for t in par.split()], LB)
    return np.asarray(w, dtype=np.float32).reshape(4, LB).T


@pytest.mark.parametrize("kind,whole", [("hann_sinc", True), ("hamming", True), ("hamming 0.53", True), ("kaiser 5", True),
                                        ("gauss 0.8", True), ("flat 1 1 1 0.5", True), ("hamming 0.585", False),
                                        ("gauss 0.953", False), ("gauss 0.954", False), ("gauss 0.955", False),
                                        ("kaiser 4.27", False), ("triangle 0", False), ("triangle 0.001", False),
                                        ("flat 0.3334 1 1 0.3334", False), ("flat 1 2 1 0", False),
                                        ("flat 1 3 3 1", False), ("flat 0 0 0 0", False)])
def test_windows(host, kind, whole):
    """A plan is admitted if all of its branches are; in those that are, whatever the
    window, the error is within the bar."""
    taps = _window(kind)
    adm = _admitted(host, taps if not kind.startswith("flat") else taps[:1])
    assert adm.all() == whole
    branches = [0] if kind.startswith("flat") else list(range(0, LB, 1237)) + [4036, 16383, 16384, 28731]
    for b in branches:
        if _admitted(host, taps[b:b + 1])[0]:
            _check_errors(host, taps[b], ROWS if b % 2 else ROWS[::3], (kind, b))


def test_hamming_within_one_block(host):
    """The reference's Hamming window in calls of at most 256 rows, whose corner is sought
    in the block itself: the solve adds nothing visible to the FP32 rounding of
    its samples (2^-30, a 64th of it), or no more than FP64 banded Cholesky."""
    taps = _window("hamming")
    for b in list(range(3900, 4301, 25)) + list(range(28500, 29001, 25)) + [28905]:
        t = np.ascontiguousarray(taps[b])
        for n in (64, 128, 225, 255, 256):
            y = np.random.default_rng(b).normal(size=n).astype(np.float32)
            e = np.zeros(2)
            host.errors(_p(t), n, _p(y), 1, _p(e))
            assert e[0] <= max(2.0 ** -30, e[1]), (b, n, e)


def _zero_sets():
    """Taps by their zeros: one to three together at moduli 0.9 to 1, gaps 0 to 0.1, at
    -1, 1 and in conjugate pairs, each zero inside or mirrored outside the circle."""
    for mod in (0.9, 0.95, 0.957, 0.97, 0.98, 0.99, 0.995, 0.999, 1.0):
        for gap in (0.0, 0.001, 0.01, 0.02, 0.05, 0.1):
            for sign in (-1.0, 1.0):
                for third in (None, 0.5, -0.99 * sign):
                    z = [sign * mod, sign * (mod - gap), sign * (mod - 2 * gap) if third is None else third]
                    for mirror in (0, 1, 2, 5, 7):
                        yield [1.0 / x if mirror >> i & 1 and x else x for i, x in enumerate(z)]
            z = mod * np.exp(1j * (np.pi - gap))
            for third in (-mod, 0.3):
                yield [z, np.conj(z), third]
                yield [1.0 / z, 1.0 / np.conj(z), third]


def test_zeros(host):
    """Factor: the taps' autocorrelation to 80-bit rounding (2^-60 of its lag 0).
    Solve: the bar wherever admitted."""
    sets = list(_zero_sets())
    taps = np.array([np.poly(z).real / np.abs(np.poly(z).real).max() for z in sets], dtype=np.float32)
    adm = _admitted(host, taps)
    assert 400 < adm.sum() < len(sets) - 400          # the grid lies on both sides of the rule
    for i, t in enumerate(taps):
        t = np.ascontiguousarray(t)
        assert host.factor_error(_p(t)) <= 2.0 ** -60, sets[i]
        if adm[i]:
            _check_errors(host, t, (ROWS[i % len(ROWS)], 300), sets[i])


def test_odd_taps(host):
    """Taps that leave no cubic, or none of moderate coefficients; what is not finite is not admitted."""
    for t in ([1, 0, 0, 0], [0, 0, 0, 1], [0, 1, 0.5, 0], [0, 0.5, 1, 0], [1e-30, 1, 0.5, 0], [1, 0.5, 0.2, 1e-38],
              [0, 1, 0, 0.5], [3e38, 1e38, 1e37, 0], [-1, 0.2, 0, 0.3], [1, 0, 0, -0.9]):
        t = np.array(t, dtype=np.float32)
        assert _admitted(host, t[None])[0] and host.factor_error(_p(t)) <= 2.0 ** -60, t
        if np.abs(t).max() < 1e30:
            _check_errors(host, t, ROWS, t)
    bad = np.array([[0, 0, 0, 0], [np.nan, 1, 0, 0], [1, np.inf, 0, 0], [0, 0, np.nan, 0]], dtype=np.float32)
    assert not _admitted(host, bad).any()
