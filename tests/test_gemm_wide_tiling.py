"""The rule that picks a tiling of the pipelined GEMM kernel: host logic, no GPU."""
import pytest


def test_the_rule_gives_a_tiling_the_kernel_takes():
    """Every problem the rule accepts passes the host-side mirror of the kernel's own checks."""
    from qfactory.core import tiling
    for M in (17, 32, 33, 64, 100, 128, 256, 512, 1024, 4096):
        for N in (1, 64, 1000, 4096, 22016, 57344):
            for K in (256, 512, 896, 1024, 4096, 11008, 28672):
                for nbits, gs in ((4, 128), (4, 32), (8, 128), (8, 32), (2, 64), (3, 128)):
                    t = tiling.gemm_wide_tiling(M, N, K, nbits, gs)
                    if t is not None:
                        assert tiling.gemm_wide_valid(t, K, nbits, gs) and t["BM"] < 2 * M
                        assert tiling.gemm_wide_lds_bytes(t, nbits) <= 160 * 1024
                    if nbits == 3 or K % (1024 // nbits):
                        assert t is None


def test_where_the_rule_takes_over():
    """From 17 rows on, at 2, 4 and 8 bits, on rows of whole 128-byte windows and five iterations: never None there, always None
    elsewhere; the specialisation of such a problem is built on it."""
    from qfactory.core import tiling
    for N, K in ((12288, 4096), (4096, 11264), (8192, 28672), (77, 2560), (1, 5120)):
        for nbits in (2, 4, 8):
            assert tiling.gemm_wide_tiling(16, N, K, nbits, 128) is None
            for M in (17, 32, 33, 64, 256, 4096):
                assert tiling.gemm_wide_tiling(M, N, K, nbits, 128) is not None, (M, N, K, nbits)
        assert tiling.gemm_wide_tiling(64, N, K, 3, 128) is None
    for K, nbits, gs in ((11008, 2, 128), (4224, 4, 128), (8256, 8, 64), (768, 2, 128), (4096, 4, 16)):
        assert tiling.gemm_wide_tiling(64, 4096, K, nbits, gs) is None, (K, nbits)
    # at 17 .. 32 rows: one round of blocks, or more than two and a half
    for N, takes in ((16384, True), (16385, False), (19008, False), (40960, False), (40961, True)):
        assert (tiling.gemm_wide_tiling(32, N, 4352, 4, 128) is not None) == takes, N
        assert tiling.gemm_wide_tiling(33, N, 4352, 4, 128) is not None
    assert _qfunc(32, 19008, 14592, 4, 128).tiling_configs == tiling.gemm_tiling(32, 19008, 14592, 4, 128)
    # 8 bits, where the table's form does not fit in LDS: two steps per iteration in half the groups
    assert [tiling.gemm_wide_tiling(M, N, 4096, 8, 128)[k] for M, N in ((32, 12288), (128, 12288)) for k in ("WN", "MT", "KI", "WK")] == \
        [2, 1, 2, 2, 4, 2, 2, 1]
    for M, N, K, nbits in ((32, 9280, 4608, 2), (64, 22016, 4096, 4), (1024, 8192, 8192, 8)):
        q = _qfunc(M, N, K, nbits, 128)
        assert q.regime == "gemm" and q.tiling_configs == tiling.gemm_wide_tiling(M, N, K, nbits, 128)
        assert "qf::GemmWideCfg<" in q.emit()


@pytest.mark.parametrize("K", [4608, 5120, 8192, 14336])
@pytest.mark.parametrize("nbits", [2, 4, 8])
def test_at_32_rows_only_two_rounds_of_blocks_stay_on_the_other_kernel(nbits, K):
    """More than two rounds of 32 x 64 blocks are one round of 32 x 224 at 2 and 4 bits: nothing there waits for a first round to end."""
    from qfactory.core import tiling
    for N in (16385, 24576, 32768):
        assert tiling.gemm_wide_tiling(32, N, K, nbits, 128) is None
    for N in (16384, 32769, 33280, 36864, 40960):
        t = tiling.gemm_wide_tiling(32, N, K, nbits, 128)
        assert t is not None and 32 * t["NT"] * t["WN"] == (64 if nbits == 8 or N == 16384 else 224), (N, t)


def _qfunc(M, N, K, nbits, gs):
    import torch
    from qfactory.core.qfunc import QMatmulQFunc
    from qfactory.core.qtile import AsymQTile, QTile
    return QMatmulQFunc(QTile((M, K), torch.float16, 16), AsymQTile((N, K), torch.int8, nbits, (1, gs)), "nt")


@pytest.mark.parametrize("M,N,K,nbits,gs", [(32, 9280, 4608, 2, 128), (64, 22016, 4096, 4, 128), (256, 12288, 4096, 4, 128),
                                           (512, 8192, 8192, 8, 128), (64, 4096, 1024, 4, 32)])
def test_search_space_is_the_pipelined_kernels_where_it_serves(M, N, K, nbits, gs):
    """``lower`` offers the default first, the tiles of the rule's table in their forms, and one tiling of the other GEMM
    kernel to measure against; the schedule has nothing to add (the kernel has one load path)."""
    from qfactory.core import tiling
    q = _qfunc(M, N, K, nbits, gs)
    cands = [c.tiling_configs for c in q.lower()]
    wide = [t for t in cands if "WM" in t]
    assert cands[0] == tiling.gemm_wide_tiling(M, N, K, nbits, gs) and len(wide) == len(cands) - 1 >= 8
    assert cands[-1] == tiling.gemm_tiling(M, N, K, nbits, gs)
    assert all(tiling.gemm_wide_valid(t, K, nbits, gs) and t["BM"] < 2 * M for t in wide)
    assert len({tuple(sorted(t.items())) for t in cands}) == len(cands)
    tiles = {tuple(t[k] for k in ("WM", "WN", "MT", "NT")) for t in wide}
    assert tiles == {key[:4] for key in tiling.GEMM_WIDE_COST if 32 * key[0] * key[2] < 2 * M
                     and any(tiling.gemm_wide_valid(dict(zip(("WM", "WN", "MT", "NT", "KI", "WK"), key[:4] + (ki, 1))), K, nbits, gs) for ki in (1, 2))}
    assert [s.l2cache_b for s in q.schedule()] == [False]


def test_search_space_of_the_other_gemm_kernel_is_as_it_was():
    from qfactory.core import tiling
    for shape in ((64, 4096, 4096, 3, 128), (64, 4096, 4224, 4, 32)):
        q = _qfunc(*shape)
        assert [c.tiling_configs for c in q.lower()] == tiling.gemm_candidates(*shape)
        assert [s.l2cache_b for s in q.schedule()] == [False, True]


HIP_CALLS = r"""
#include <stddef.h>
#include <stdio.h>
typedef struct { unsigned x, y, z; } dim3_;
int hipFuncSetAttribute(const void* f, int attr, int value) { (void)f; printf("attribute %d %d\n", attr, value); fflush(stdout); return 0; }
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* s) { (void)g; (void)b; (void)s; printf("launch %zu\n", lds); fflush(stdout); return 1; }
int hipGetLastError(void) { return 0; }
"""


def test_the_first_launch_of_a_two_tiling_object_raises_both_lds_limits(tmp_path):
    """Whichever tiling the first launch takes, no later launch (which may come under graph capture) has an attribute
    left to set.  The object's HIP calls go to stand-ins that print what they are asked for."""
    import os
    import subprocess
    import sys
    import prebuild
    from qfactory.core import tiling
    from qfactory.jit import jit
    (qfunc,) = prebuild.qfuncs_of(prebuild._case(256, 12288, 1024))
    sizes = [tiling.gemm_wide_lds_bytes(t, 4) for t in (tiling.gemm_wide_low_tiling(256, 12288, 1024, 4, 128), qfunc.tiling_configs)]
    assert sizes[0] != sizes[1] and min(sizes) > 64 * 1024
    (tmp_path / "calls.c").write_text(HIP_CALLS)
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "calls.c"), "-o", str(tmp_path / "calls.so")], check=True)
    obj = os.path.join(jit.compile(qfunc).path, "kernel.so")
    probe = ("import ctypes; launch = ctypes.CDLL(%r).launch_m; rc = ctypes.c_int(-1)\n"
             "for m in %r:\n launch(m, None, None, None, None, None, None, ctypes.byref(rc))\n assert rc.value == 0, rc.value\n")
    for rows in ((1, 256, 192, 193), (256, 1, 193, 192)):
        out = subprocess.run([sys.executable, "-c", probe % (obj, rows)], env=dict(os.environ, LD_PRELOAD=str(tmp_path / "calls.so")),
                             check=True, capture_output=True, text=True, timeout=120).stdout.splitlines()
        assert sorted(int(line.split()[2]) for line in out[:2] if line.startswith("attribute")) == sorted(sizes), out
        assert out[2:] == [f"launch {sizes[0] if m <= 192 else sizes[1]}" for m in rows], out
