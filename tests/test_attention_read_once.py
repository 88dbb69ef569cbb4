"""From which length on the decode attention loads its cache rows past the Infinity Cache: where a step's rows, those of every
layer together, are more than its 256 MB.  The limit is the kernel's last argument; here the launch goes to a stand-in that prints it."""
import os
import subprocess
import sys

import pytest

HIP_CALLS = r"""
#include <stddef.h>
#include <stdio.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3_;
static dim3_ grid, block;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void* s) { (void)lds; (void)s; grid = g; block = b; return 0; }
int __hipPopCallConfiguration(dim3_* g, dim3_* b, size_t* lds, void** s) { *g = grid; *b = block; *lds = 0; *s = NULL; return 0; }
int hipLaunchKernel(const void* f, dim3_ g, dim3_ b, void** args, size_t lds, void* s) {
    (void)f; (void)b; (void)lds; (void)s;
    printf("%u %u %d\n", g.x, g.y, *(int*)args[10]); fflush(stdout);
    return 0;
}
int hipGetLastError(void) { return 0; }
"""

# (batch, heads, head_dim, layers) -> shortest sequence whose rows are loaded past the cache
CASES = [((16, 32, 128, 8), 128), ((16, 32, 128, 0), 128), ((1, 32, 128, 32), 512), ((4, 32, 128, 32), 128), ((8, 32, 128, 32), 64),
         ((4, 32, 128, 2), 2048), ((32, 32, 128, 2), 256), ((32, 32, 128, 1), 512), ((32, 32, 64, 1), 1024), ((32, 32, 256, 1), 256),
         ((64, 32, 128, 2), 32), ((64, 32, 128, 1), 32), ((33, 32, 128, 1), 63), ((64, 32, 128, 16), 16),
         ((5, 32, 32, 1), 13108), ((2, 3, 128, 1 << 20), 1), ((65535, 64, 256, 1), 1), ((1, 1, 32, 1), 2097152)]


def test_the_limit_is_what_the_cache_holds_over_all_layers(tmp_path):
    from qfactory import native
    native.build()
    (tmp_path / "calls.c").write_text(HIP_CALLS)
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "calls.c"), "-o", str(tmp_path / "calls.so")], check=True)
    # no device: the addresses are never read, the caches' length is not part of the rule
    probe = ("import ctypes; from ctypes import c_int64 as I, c_void_p as P; lib = ctypes.CDLL(%r)\n"
             "at = [P(16)] * 8\n"
             "for B, H, hd, layers in %r:\n"
             " assert lib.qf_decode_attention_layers(*at[:5], I(B), I(H), I(hd), I(4096), I(layers), None) == 0\n"
             " assert lib.qf_rope_decode_attention_layers(*at[:7], I(B), I(H), I(hd), I(4096), I(layers), None) == 0\n"
             " if layers == 0:\n"
             "  assert lib.qf_decode_attention(*at[:5], I(B), I(H), I(hd), I(4096), None) == 0\n"
             "  assert lib.qf_rope_decode_attention(*at[:7], I(B), I(H), I(hd), I(4096), None) == 0\n"
             "for layers in (-1, (1 << 20) + 1):\n"
             " assert lib.qf_decode_attention_layers(*at[:5], I(1), I(1), I(128), I(16), I(layers), None) == 1\n")
    out = subprocess.run([sys.executable, "-c", probe % (native.LIBRARY, [case for case, _ in CASES])],
                         env=dict(os.environ, LD_PRELOAD=str(tmp_path / "calls.so")), check=True, capture_output=True, text=True,
                         timeout=120).stdout.splitlines()
    want = [f"{heads} {batch} {limit}" for (batch, heads, _, layers), limit in CASES for _ in range(2 if layers else 4)]
    assert out == want


def _caches(B, H, hd, max_len, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    k, v = (torch.randn(B, H, max_len, hd, device="cuda", generator=g).to(torch.float16) for _ in range(2))
    qkv = torch.randn(B, 3 * H * hd, device="cuda", generator=g).to(torch.float16)
    ang = torch.arange(max_len, device="cuda", dtype=torch.float32)[:, None] * torch.rand(hd // 2, device="cuda", generator=g)[None, :]
    return k, v, qkv, ang.cos(), ang.sin()


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [32, 64, 128, 256])
def test_rows_read_once_give_the_same_bits(hd):
    """Every number of stages, their ends and sequences longer than all of them, in both modes of both entry points; the cached mode
    is what the tests of the attention hold against PyTorch's."""
    import torch
    from qfactory import native
    B, H, group = 2, 3, 4096 // hd                                    # positions of a stage: 512 threads, hd / 8 lanes each
    max_len = 10 * group
    k0, v0, qkv, cos, sin = _caches(B, H, hd, max_len, hd)
    for n in sorted({s * group + d for s in range(1, 10) for d in (-1, 0, 1)} | {1, max_len}):
        pos = torch.tensor([n - 1], device="cuda")
        out = []
        for layers in (1, 1 << 20):                                   # 256 MB are never reached, always passed
            k, v, att, rope = k0.clone(), v0.clone(), *(torch.empty(B, H * hd, dtype=torch.float16, device="cuda") for _ in range(2))
            native.decode_attention(qkv[:, :H * hd].contiguous(), k, v, pos, att, layers)
            native.rope_decode_attention(qkv, pos, cos, sin, k, v, rope, layers)
            out.append((att, rope, k, v))
        assert all(torch.equal(a, b) for a, b in zip(*out)), n
        assert torch.isfinite(out[0][0]).all() and torch.isfinite(out[0][1]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("fuse_norm", [True, False])
def test_the_decode_loop_says_how_many_layers_it_has(fuse_norm, monkeypatch):
    """At both forms of the step (norms inside the projections and as launches of their own)."""
    import decode_llama
    import torch
    from qfactory import native
    shape = decode_llama.LlamaShape(layers=3, hidden=256, heads=4, mlp=512, vocab=1000, max_len=32, group_size=64)
    batch = 2
    model = decode_llama.QuantLlama(shape, batch=batch, seed=3)
    model.fuse_norm = fuse_norm
    seen, own = [], native.load().qf_rope_decode_attention_layers

    class Library:
        def __getattr__(self, name):
            return getattr(library, name)

        def qf_rope_decode_attention_layers(self, *args):
            seen.append(args[-2])
            return own(*args)

    library = native.load()
    monkeypatch.setattr(native, "_lib", Library())
    model.decode_step(torch.zeros(batch, 1, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda"))
    torch.cuda.synchronize()
    assert seen == [3, 3, 3]
