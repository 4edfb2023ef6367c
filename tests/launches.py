"""Which kernels a call launched, from the library's launch report: a comparison of two paths has to know that it took both."""
import ctypes
import json

from lact_amd import _lib


def launches(fn):
    """What fn returns, and the launch report: kernel, site, stream (in the order of their first launch), count, times."""
    lib, buf = _lib.lib(), ctypes.create_string_buffer(1 << 16)
    _lib.check(lib.lact_profile_enable(1))
    try:
        res = fn()
        _lib.check(lib.lact_profile_report(buf, len(buf)))
    finally:
        _lib.check(lib.lact_profile_enable(0))
    return res, json.loads(buf.value)


def kernels(fn):
    """What fn returns, and the names of the kernels that it launched."""
    res, report = launches(fn)
    return res, {r["kernel"] for r in report}


def streams(fn):
    """What fn returns, and the number of streams that its kernels were launched on."""
    res, report = launches(fn)
    return res, 1 + max(r["stream"] for r in report)
