"""The rule that picks a tiling of the pipelined GEMM kernel: host logic, no GPU."""


def test_the_rule_gives_a_tiling_the_kernel_takes():
    """Every problem the rule accepts passes the host-side mirror of the kernel's own checks."""
    from qfactory.core import tiling
    for M in (33, 64, 100, 128, 256, 512, 1024, 4096):
        for N in (1, 64, 1000, 4096, 22016, 57344):
            for K in (256, 512, 896, 1024, 4096, 11008, 28672):
                for nbits, gs in ((4, 128), (4, 32), (8, 128), (8, 32), (2, 64), (3, 128)):
                    t = tiling.gemm_wide_tiling(M, N, K, nbits, gs)
                    if t is not None:
                        assert tiling.gemm_wide_valid(t, K, nbits, gs) and t["BM"] < 2 * M
                        assert tiling.gemm_wide_lds_bytes(t, nbits) <= 160 * 1024
                    if nbits == 3 or K % (1024 // nbits):
                        assert t is None
