"""The threaded copy of large logits into the caller's buffer (no GPU)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from strasgpt_amd import _paths

pytestmark = pytest.mark.skipif(not os.path.exists(_paths.hip_lib()), reason="library not built")

KIB = 1024


@pytest.mark.parametrize("n", [1, 512 * KIB - 1, 1024 * KIB - 1, 1024 * KIB, 1024 * KIB + 1, 3000 * KIB + 5,
                               4096 * KIB, 4096 * KIB - 4097, 12345677])
def test_copy_whole_and_no_more(n):
    """Sizes around one, two and eight pieces of 512 KiB and around whole pages,
    into unaligned destinations: every byte arrives, none beside them changes."""
    from strasgpt_amd import runtime as rt
    copy = rt.lib().st_host_copy
    copy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    copy.restype = None
    src = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    for offset in (0, 4, 4095):
        dst = np.full(n + 8192, 0xA5, np.uint8)
        copy(dst.ctypes.data + offset, src.ctypes.data, n)
        np.testing.assert_array_equal(dst[offset:offset + n], src)
        assert (dst[:offset] == 0xA5).all() and (dst[offset + n:] == 0xA5).all()


def test_exported_names_are_the_library_s_own():
    """Every exported C function carries one of the library's prefixes: a
    program's own function of a common name is not taken in its place."""
    out = subprocess.run(["nm", "-D", "--defined-only", _paths.hip_lib()], capture_output=True, text=True, check=True)
    names = [line.split()[2] for line in out.stdout.splitlines() if line.split()[1] == "T"]
    prefixes = ("transformer_", "safetensors_", "tokenizer_", "sampler_", "strasgpt_", "sg_", "st_",
                "_Z", "_init", "_fini",
                "json_scanner_lex_destroy")  # (a driver of the reference calls it)
    assert names and not [n for n in names if not n.startswith(prefixes)]
