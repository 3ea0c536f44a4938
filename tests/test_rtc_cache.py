"""Handles of the same lengths share the passes compiled at run time, also where another batch changes some of their
plans: each pass is compiled once per process (lp_debug_rtc_compile takes a handle's way; no device needed)."""
import ctypes

from lprec_amd import _lib


def planned(N, P0, Ns):
    buf = ctypes.create_string_buffer(4096)
    assert _lib.load().lp_debug_rtc_names(N, P0, Ns, 1, 0, 160 * 1024, buf, len(buf)) > 0
    return [n for n in buf.value.decode().split("\n") if n]


def compiled(names):
    """Passes compiled for a handle that asks for these."""
    lib, got = _lib.load(), ctypes.c_uint()
    before = lib.lp_debug_rtc_passes()
    assert lib.lp_debug_rtc_compile("\n".join(names).encode(), ctypes.byref(got)) == 0
    assert got.value == (1 << len(names)) - 1
    return lib.lp_debug_rtc_passes() - before


def test_a_pass_is_compiled_once():
    lines = {Ns: planned(336, 252, Ns) for Ns in (1, 8, 32)}
    seen = set()
    for Ns in (1, 8, 32, 8):
        new = set(lines[Ns]) - seen
        assert compiled(lines[Ns]) == len(new), Ns
        seen |= new
    assert len(seen) < 12   # some are shared

