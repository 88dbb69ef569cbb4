"""Causal attention of a prompt over the KV cache (libqfactory_hip.so) against softmax in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, pos):
    q, k, v = (t.double().cpu() for t in (q, k, v))
    scores = q.transpose(1, 2) @ k.transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5        # (B, H, T, max_len)
    hidden = torch.arange(k.shape[2])[None, :] > pos.cpu()[:, None]
    return (scores.masked_fill(hidden, float("-inf")).softmax(-1) @ v).transpose(1, 2)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,T,H,max_len,first", [(1, 1, 1, 64, 0), (2, 17, 3, 256, 0), (1, 33, 2, 100, 60), (3, 128, 4, 256, 0),
                                                 (1, 129, 2, 256, 127), (2, 200, 2, 200, 0), (1, 64, 2, 1000, 900)])
def test_prefill_attention(hd, B, T, H, max_len, first):
    """Ragged row blocks, cache lengths that are not whole key tiles, prompts that continue a cache.  What the cache holds
    behind a token's position must not be seen."""
    from qfactory import native
    print(f"[case] B{B} T{T} H{H} hd{hd} max_len{max_len} first{first}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + hd)
    q = (torch.randn(B, T, H, hd, device="cuda", generator=g) * 2).half()
    k, v = ((torch.randn(B, H, max_len, hd, device="cuda", generator=g) * 1.5).half() for _ in range(2))
    pos = torch.arange(first, first + T, device="cuda")
    out = torch.full((B, T, H, hd), float("nan"), dtype=torch.float16, device="cuda")
    ref = _reference(q, k, v, pos)
    native.prefill_attention(q, k, v, pos, out)
    err = (out.double().cpu() - ref).norm() / ref.norm()
    # one rounding of the result to fp16 (2^-11 / sqrt(3) = 2.8e-4); probabilities enter with 22 bits, sums are fp32
    assert err <= 4e-4, err
    again = torch.empty_like(out)
    native.prefill_attention(q, k, v, pos, again)
    assert torch.equal(out, again)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("T,max_len,first", [(70, 256, 0), (129, 200, 3), (33, 100, 60)])
def test_rows_behind_a_position_never_reach_it(hd, T, max_len, first):
    """Unwritten cache rows (NaN and infinities behind the last position, in the prompt's last key tile and past it) leave
    no trace; an infinite or NaN V inside the prompt reaches the tokens from its position on, as it should, and none before."""
    from qfactory import native
    print(f"[case] hd{hd} T{T} max_len{max_len} first{first}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    B, H = 2, 2
    q = torch.randn(B, T, H, hd, device="cuda", generator=g).half()
    k, v = (torch.randn(B, H, max_len, hd, device="cuda", generator=g).half() for _ in range(2))
    pos = torch.arange(first, first + T, device="cuda")
    ref = _reference(q, k, v, pos)
    for cache in (k, v):
        cache[:, :, first + T:] = float("nan")
        cache[:, :, first + T::3] = float("inf")
    out = native.prefill_attention(q, k, v, pos, torch.empty_like(q))
    assert (out.double().cpu() - ref).norm() / ref.norm() <= 4e-4
    dims = {0: float("inf"), 5: float("-inf"), hd - 1: float("nan")}
    at = first + T // 2
    for d, value in dims.items():
        v[1, 0, at, d] = value
    odd = native.prefill_attention(q, k, v, pos, torch.empty_like(q)).double().cpu()
    want = ref.clone()
    for d, value in dims.items():
        want[1, T // 2:, 0, d] = value
        assert torch.equal(odd[..., d][~want[..., d].isfinite()].nan_to_num(nan=-1.0),
                           want[..., d][~want[..., d].isfinite()].nan_to_num(nan=-1.0))
    seen = want.isfinite()
    assert odd[seen].isfinite().all()
    assert (odd[seen] - ref[seen]).norm() / ref[seen].norm() <= 4e-4


def test_positions_in_any_order():
    from qfactory import native
    g = torch.Generator(device="cuda").manual_seed(5)
    B, T, H, hd, max_len = 2, 140, 2, 128, 192
    q = torch.randn(B, T, H, hd, device="cuda", generator=g).half()
    k, v = (torch.randn(B, H, max_len, hd, device="cuda", generator=g).half() for _ in range(2))
    pos = torch.randperm(max_len, device="cuda", generator=g)[:T].contiguous()
    out = torch.empty_like(q)
    native.prefill_attention(q, k, v, pos, out)
    ref = _reference(q, k, v, pos)
    assert (out.double().cpu() - ref).norm() / ref.norm() <= 4e-4


def test_bad_arguments_are_rejected_without_launching():
    from qfactory import native
    buf = torch.zeros(4096, dtype=torch.float16, device="cuda")
    pos = torch.zeros(1, dtype=torch.int64, device="cuda")
    call = lambda hd, q=buf.data_ptr(), tokens=1: native.load().qf_prefill_attention(
        q, buf.data_ptr(), buf.data_ptr(), pos.data_ptr(), buf.data_ptr(), 1, tokens, 1, hd, 1, None)
    assert call(32) == 1 and call(96) == 1
    assert call(64, q=buf.data_ptr() + 2) == 1 and call(64, q=None) == 1 and call(64, tokens=0) == 1
