"""The plans of the passes compiled at run time, from the library's own planner
(lp_debug_rtc_names; no device needed): what a block declares fits the 160 KB of
LDS at every grid, so that none of them fails to compile, and a selection
compiles for gfx950 with hipRTC (register and matrix-core radices, two
matrix-core stages, rows whose LDS is close to the limit)."""
import ctypes
import ctypes.util
import os
import re

import pytest

from lprec_amd import _lib

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lprec_amd", "csrc")
LDS = 160 * 1024


def planned(N, P0, Ns, filt=1, cols_threads=0):
    buf = ctypes.create_string_buffer(4096)
    n = _lib.load().lp_debug_rtc_names(N, P0, Ns, filt, cols_threads, LDS, buf, len(buf))
    assert 0 < n <= len(buf)
    return [s for s in buf.value.decode().split("\n") if s]


def declared_lds(name):
    """Bytes of the arrays that the kernel declares (rtc_kernels.hpp), padded to 16 each, and the 256 bytes that
    __syncthreads_or takes in the inverse row pass."""
    kernel, args = re.match(r"lpct::(\w+)<(.*)>", name).groups()
    a = [int(v) for v in args.split(",")]
    up = lambda n, m: (n + m - 1) // m * m
    if kernel.startswith("k_rows"):
        H, R, LS = a[0], a[1], a[2]
        slots = H if a[6] & 1 else H + H // 16 + 1
        return (up(8 * R * max(LS, slots), 16) + up(8 * R, 16) + up(8 * (H // 2 + 1), 16)
                + (256 if kernel == "k_rows_inv_ct" else 0))
    M, first = (a[0], a[4]) if kernel == "k_cols_ct" else (2 * a[0], a[3])
    slots = M if first & 1 else M + M // 16 + 1
    return 8 * (up(slots, 128) if kernel == "k_cols_ct" else slots)


def test_planned_blocks_fit_lds():
    over = []
    for N in range(16, 10240, 16):
        for Ns in (1, 4, 32):
            over += [(N, Ns, n, declared_lds(n)) for n in planned(N, max(1, 3 * N // 4), Ns) if declared_lds(n) > LDS]
    assert not over, over[:5]


def _hiprtc():
    for name in ("/opt/rocm/lib/libhiprtc.so", ctypes.util.find_library("hiprtc")):
        if name:
            try:
                return ctypes.CDLL(name)
            except OSError:
                pass
    pytest.skip("libhiprtc not available")


def _compile(names):
    """None, or the log of the failed compile."""
    rtc = _hiprtc()
    prog = ctypes.c_void_p()
    assert rtc.hiprtcCreateProgram(ctypes.byref(prog), b'#include "rtc_kernels.hpp"\n', b"plans.hip", 0, None, None) == 0
    for n in names:
        assert rtc.hiprtcAddNameExpression(prog, n.encode()) == 0
    opts = [b"--offload-arch=gfx950", b"-O3", b"-std=c++17", ("-I" + CSRC).encode(),
            b"-Xclang", b"-target-feature", b"-Xclang", b"-packed-fp32-ops"]
    log = None
    if rtc.hiprtcCompileProgram(prog, len(opts), (ctypes.c_char_p * len(opts))(*opts)) != 0:
        n = ctypes.c_size_t()
        rtc.hiprtcGetProgramLogSize(prog, ctypes.byref(n))
        buf = ctypes.create_string_buffer(n.value + 1)
        rtc.hiprtcGetProgramLog(prog, buf)
        log = buf.value.decode(errors="replace")[:3000]
    rtc.hiprtcDestroyProgram(ctypes.byref(prog))
    return log


@pytest.mark.parametrize("N,Ns", [
    (64, 1),                # the smallest grid in use
    (528, 8), (1056, 7),    # composite register radices
    (2064, 1), (2064, 32),  # 43
    (2096, 8),              # 131
    (4608, 1), (4608, 16),  # rows of 2304 points: 8 of them and the R2C twiddles do not fit
    (4624, 1),              # 17 x 17
    (8640, 1), (9216, 1), (9552, 1),
])
def test_planned_passes_compile_for_gfx950(N, Ns):
    names = planned(N, 3 * N // 4, Ns)
    assert len(names) == 4, names   # rows there and back, columns, filtered pair
    log = _compile(names)
    assert log is None, log


def test_a_pass_that_does_not_compile_leaves_the_others():
    """Rows whose LDS is over the limit, beside columns and filter rows that compile."""
    _hiprtc()
    names = ["lpct::k_rows_fwd_ct<2304, 8, 2468, 768, 2, 1, 24, 12, 8>", "lpct::k_cols_ct<528, 64, 4, 2, 11, 12, 4>",
             "lpct::k_sino_rows_pair_ct<264, 64, 4, 11, 12, 4>"]
    assert _compile(names[:1]) is not None and _compile(names[1:]) is None
    got = ctypes.c_uint()
    assert _lib.load().lp_debug_rtc_compile("\n".join(names).encode(), ctypes.byref(got)) == 0
    assert got.value == 0b110


def test_threads_asked_for_keep_the_column_pass():
    """Tuning key 11 at every length where it is accepted (32 points a thread): the columns have a plan, with that
    many threads unless a thread would hold more than 16 points (a prime radix may not divide among them so)."""
    for N in range(16, 4944, 16):
        for threads in (256, 512, 1024):
            if threads * 32 < 2 * N:
                continue
            names = [n for n in planned(N, N, 8, 0, threads) if "k_cols_ct" in n]
            if not names:
                assert N & (N - 1) == 0 and N >= 128, N   # the register kernels' lengths
                continue
            used = int(names[0].split(",")[1])
            assert used == threads or 2 * N > 16 * threads, names
