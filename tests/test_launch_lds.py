"""Dynamic LDS beyond 64 KiB has to be asked for, per kernel, before a launch that wants it.  Checked on the host: a stand-in for
the runtime calls in question notes what is asked for and launched, and the library's entry points run on addresses
that nobody looks at."""
import os
import subprocess
import sys

import pytest

from bitnet_amd import _lib

STAND_IN = r"""
#include <stddef.h>
#include <stdio.h>
typedef struct { unsigned x, y, z; } dim3;
static size_t pending;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) { pending = lds; return 0; }
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) { *lds = pending; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int what, int value) {
    if (what == 8) printf("asked %p %d\n", f, value), fflush(stdout); /* the largest dynamic LDS */
    return 0;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, void* stream) {
    printf("launched %p %zu\n", f, lds), fflush(stdout);
    return 0;
}
"""
CALLS = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
p = ctypes.c_void_p(0x100000)
what = sys.argv[3]
if what == "attention":
    for heads, kv in ((32, 32), (32, 16), (20, 5), (64, 8)):
        for tokens in (17, 4096):
            assert lib.bitnet_attn_prefill(p, p, p, p, 1, tokens, 4096, 0, heads, kv, 128, None) == 0
elif what == "gemm":
    for tile in range(16):
        for split in (0, 1, 2, 4):
            assert lib.bitlinear_set_tuning(5, tile, 0, split) == 0
            lib.bitlinear_int8xint2(p, p, p, p, p, 100, 2560, 2560, None)
            assert lib.bitlinear_last_status() == 0
"""


@pytest.mark.parametrize("what", ["attention", "gemm"])
def test_every_launch_with_more_than_64_kib_of_lds_has_asked_for_it(what, tmp_path):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    source, stand_in = tmp_path / "runtime.c", tmp_path / "runtime.so"
    source.write_text(STAND_IN)
    subprocess.run(["gcc", "-shared", "-fPIC", str(source), "-o", str(stand_in)], check=True)
    out = subprocess.run([sys.executable, "-c", CALLS, str(stand_in), _lib.LIB_PATH, what], check=True, capture_output=True, text=True).stdout
    asked, large = {}, set()
    for line in out.splitlines():
        did, kernel, size = line.split()
        if did == "asked":
            asked[kernel] = max(asked.get(kernel, 0), int(size))
        else:
            assert int(size) <= max(65536, asked.get(kernel, 0)), (kernel, size)
            large |= {kernel} if int(size) > 65536 else set()
    assert len(large) >= 3, out  # (the attention's three instances; the ring kernel's)
