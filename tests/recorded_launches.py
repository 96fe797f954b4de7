"""Runs in a process of its own: the built library's host code on the recorder of tests/hip_recorder.cpp.  A test imports
`Recorder` there and calls the C entry points with made-up device addresses; what would have been launched comes back."""

import ctypes
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT))

from lighthouse_amd import _lib  # noqa: E402


class PadCopy(ctypes.Structure):
    _fields_ = [("dst", ctypes.c_uint64), ("src", ctypes.c_uint64), ("ld_dst", ctypes.c_int64), ("ld_src", ctypes.c_int64),
                ("rows_dst", ctypes.c_int32), ("cols_dst", ctypes.c_int32), ("rows_src", ctypes.c_int32), ("cols_src", ctypes.c_int32)]


class GemmArgs(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint64) for n in ("out", "c", "a", "b", "bias")] + \
               [(n, ctypes.c_int32) for n in ("M", "N", "K")] + [(n, ctypes.c_int64) for n in ("lda", "ldb", "ldc")] + \
               [(n, ctypes.c_int32) for n in ("flags", "out_dt", "bias_dt")] + [("alpha", ctypes.c_float), ("splits", ctypes.c_int32)] + \
               [("ws", ctypes.c_uint64), ("touch_b", ctypes.c_int32)]


class Touch(ctypes.Structure):
    _fields_ = [("p", ctypes.c_uint64 * 3), ("lines", ctypes.c_uint32 * 3)]


class Launch(ctypes.Structure):
    _fields_ = [("mangled", ctypes.c_char_p), ("grid", ctypes.c_uint32), ("block", ctypes.c_uint32),
                ("arg0", ctypes.c_ubyte * 120), ("arg1", ctypes.c_ubyte * 48)]

    @property
    def name(self):
        return self.mangled.decode()

    @property
    def gemm(self):
        return GemmArgs.from_buffer_copy(self.arg0)

    @property
    def touched(self):
        """(first byte, lines of 128 bytes) of each range that the launch touches for later ones."""
        t = Touch.from_buffer_copy(self.arg1) if "5Touch" in self.name or "gemm_normed" in self.name else Touch()
        return [(p, n) for p, n in zip(t.p, t.lines) if n]

    @property
    def copies(self):
        """(destination, source) of each matrix a padding copy writes, as (first byte, one past the last)."""
        if "pad_copy_kernel" not in self.name:
            return []
        es = {"t": 2, "j": 4, "h": 1}[self.name.split("pad_copy_kernelI")[1][0]]
        found = {}
        for raw in (self.arg0, self.arg1):
            c = PadCopy.from_buffer_copy(raw)
            span = lambda p, ld, rows, cols: (p, p + es * ((rows - 1) * ld + cols)) if rows and cols else (p, p)  # noqa: E731
            found[c.dst] = (span(c.dst, c.ld_dst, c.rows_dst, c.cols_dst), span(c.src, c.ld_src, c.rows_src, c.cols_src))
        return list(found.values())


class Recorder:
    def __init__(self, so):
        self.recorder = ctypes.CDLL(so, ctypes.RTLD_GLOBAL)  # (in front of the runtime that the library is linked to)
        self.recorder.recorder_launch.restype = ctypes.POINTER(Launch)
        self.lib = _lib.load()

    def calls(self, entry, *args):
        """Status of the call and its launches."""
        self.recorder.recorder_reset()
        rc = getattr(self.lib, entry)(*args)
        return rc, [Launch.from_buffer_copy(self.recorder.recorder_launch(i).contents) for i in range(self.recorder.recorder_count())]


def build(folder):
    so = Path(folder) / "libhip_recorder.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(ROOT / "tests" / "hip_recorder.cpp"), "-o", str(so)], check=True)
    return str(so)
