"""Which blocks a layer is packed by: 64 columns and 256 threads where blocks of 128 columns would be at most 128, or more than one and up
to one and a half per CU, or more than one where columns are loaded one by one; else 128 columns and 512 threads.  The launch goes to a stand-in that prints it."""
import os
import subprocess
import sys

HIP_CALLS = r"""
#include <stddef.h>
#include <stdio.h>
typedef struct { unsigned x, y, z; } dim3_;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* s) { (void)lds; (void)s; printf("%u %u\n", g.x, b.x); fflush(stdout); return 1; }
int hipGetLastError(void) { return 0; }
"""

# (nbits, K, N, address of the weights) -> blocks, threads
CASES = [((4, 1024, 1024, 16), (16 * 4, 256)), ((2, 4096, 64, 16), (8, 256)), ((2, 4096, 2048, 16), (32 * 8, 256)), ((3, 4096, 2052, 16), (17 * 8, 512)),
         ((4, 4096, 1024, 16), (16 * 16, 256)), ((4, 4128, 1024, 16), (8 * 17, 512)), ((8, 4096, 896, 16), (7 * 32, 512)), ((4, 4096, 22016, 16), (172 * 16, 512)),
         ((8, 4096, 1024, 16), (16 * 32, 256)), ((4, 4096, 2048, 16), (32 * 16, 256)), ((2, 4096, 4096, 16), (32 * 8, 512)), ((3, 4096, 4096, 16), (32 * 8, 512)),
         ((2, 4096, 4100, 16), (65 * 8, 256)), ((3, 4096, 4224, 16), (66 * 8, 256)), ((4, 4096, 3072, 16), (48 * 16, 256)), ((8, 4096, 1536, 16), (24 * 32, 256)),
         ((4, 4096, 3076, 16), (25 * 16, 512)), ((8, 4128, 1536, 16), (12 * 33, 512)), ((2, 4096, 6148, 16), (49 * 8, 512)),
         # columns no multiple of four, or an address no multiple of 16 bytes
         ((3, 4096, 2049, 16), (17 * 8, 512)), ((2, 4096, 4095, 16), (32 * 8, 512)), ((2, 4096, 8190, 16), (128 * 8, 256)), ((4, 4096, 22016, 20), (344 * 16, 256)), ((8, 4096, 4093, 16), (64 * 32, 256))]


def test_small_layers_are_packed_by_narrow_blocks(tmp_path):
    from qfactory import native
    native.build()
    (tmp_path / "calls.c").write_text(HIP_CALLS)
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "calls.c"), "-o", str(tmp_path / "calls.so")], check=True)
    probe = ("import ctypes; from ctypes import c_int64 as I, c_void_p as P; lib = ctypes.CDLL(%r)\n"
             "for nbits, K, N, at in %r:\n assert lib.qf_pack_weight(P(at), P(16), I(K), I(N), nbits, None) == 0\n")
    out = subprocess.run([sys.executable, "-c", probe % (native.LIBRARY, [case for case, _ in CASES])],
                         env=dict(os.environ, LD_PRELOAD=str(tmp_path / "calls.so")), check=True, capture_output=True, text=True,
                         timeout=120).stdout.splitlines()
    assert out == [f"{blocks} {threads}" for _, (blocks, threads) in CASES]
