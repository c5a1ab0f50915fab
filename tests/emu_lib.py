"""The CPU builds of the batched aligner (tests/wave_emu) as libraries."""

from __future__ import annotations

import ctypes as C
import fcntl
import os
import subprocess
from contextlib import contextmanager

from marvel_amd import align
from marvel_amd.lib import MiAlignParams, MiLaResult, MiLaTask

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "wave_emu")


def build():
    with open(os.path.join(HERE, ".lock"), "w") as f:   # one builder at a time (pytest -n)
        fcntl.flock(f, fcntl.LOCK_EX)
        subprocess.check_call(["make", "-s", "-j2", "-C", HERE, "libs"])


class Lib:
    def __init__(self, garbage: bool = False):
        self.h = C.CDLL(os.path.join(HERE, "_build", "libemu_la_garbage.so" if garbage else "libemu_la.so"))
        p, ll = C.c_void_p, C.c_longlong
        self.h.mi_la_batch_host.argtypes = [C.POINTER(MiAlignParams), p, ll, C.POINTER(MiLaTask), C.c_int,
                                            C.POINTER(MiLaResult), p, ll]
        self.h.mi_la_batch_device_noalloc.argtypes = [C.POINTER(MiAlignParams), p, ll, p, C.c_int, p, p, ll, p]
        self.h.mi_set_tuning.argtypes = [p]
        self.h.mi_last_error.restype = C.c_char_p

    def __getattr__(self, name):
        return getattr(self.h, name)

    def last_error(self) -> str:
        return self.h.mi_last_error().decode()


@contextmanager
def in_place_of_gpu(lib: Lib):
    """marvel_amd.align's batches run on `lib`."""
    saved, align.lib = align.lib, lib
    try:
        yield
    finally:
        align.lib = saved
