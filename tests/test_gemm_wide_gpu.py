"""The pipelined GEMM kernel (include/qf_gemm_wide.hip.h) at the edges of its tilings against the CPU oracle."""
import pytest
import torch

import prebuild
from helpers import assert_close, make_problem, reference_output

pytestmark = pytest.mark.gpu

NO_SEARCH = {"enable_transform": False, "enable_schedule": False, "enable_lower": False}


def _id(c):
    t = dict(c["tiling"])
    return (f"M{c['M']}-N{c['N']}-K{c['K']}-b{c['NBITS']}-g{c['GS']}-{'sym' if c['sym'] else 'asym'}-"
            + "x".join(str(t[k]) for k in ("WM", "WN", "MT", "NT", "KI", "WK")))


def _launch(runtime, x, layer, out):
    z = layer.z if layer.z is not None else torch.empty(1, dtype=torch.int8, device="cuda")
    rc = runtime.run_raw(x.shape[0], (x.data_ptr(), layer.w.data_ptr(), out.data_ptr(), layer.s.data_ptr(), z.data_ptr()),
                         torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0


@pytest.mark.parametrize("case", [c for c in prebuild.wide_cases() if "tiling" in c], ids=_id)
def test_tilings_at_their_edges(oracle, case):
    from qfactory import QLinear
    from qfactory.jit import jit
    M, N, K, nbits, GS, sym = (case[k] for k in ("M", "N", "K", "NBITS", "GS", "sym"))
    print(f"[case] {_id(case)}", flush=True)
    A, weight, scale, zero = make_problem(77 + N + K + M, M, N, K, nbits, GS, sym)
    layer = QLinear.init(1, K, N, nbits, weight.cuda(), GS, scale.cuda(), None if zero is None else zero.cuda(),
                         compile_flags=NO_SEARCH)
    (qfunc,) = prebuild.qfuncs_of(case)
    assert qfunc.regime == "gemm" and qfunc.tiling_configs == dict(case["tiling"])
    runtime = jit.compile(qfunc)
    assert runtime.description.endswith("waits=counted")
    x = A.cuda()
    # a row of its own behind the output: nothing may be written there
    store = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device="cuda")
    _launch(runtime, x, layer, store[:M])
    assert store[M].isnan().all()
    first = store[:M].clone()
    assert_close(oracle, first.cpu().numpy(), reference_output(oracle, A, layer.w, layer.s, layer.z, nbits, GS), _id(case))
    _launch(runtime, x, layer, store[:M])
    assert torch.equal(first, store[:M])
    # an activation that starts off a 16-byte boundary, a single row, rows of one tile only
    shifted = torch.empty(M * K + 8, dtype=torch.float16, device="cuda")[1:1 + M * K].view(M, K)
    shifted.copy_(x)
    for rows in (M, min(M, 32), 1):
        store.fill_(float("nan"))
        _launch(runtime, shifted[:rows], layer, store[:rows])
        assert torch.equal(first[:rows], store[:rows]) and store[rows:].isnan().all()


def test_the_widest_layers_of_17_to_32_rows(oracle):
    """More columns than two rounds of 32 x 64 blocks, the last of 149 tiles 129 columns wide: the layer's own launch, against the
    oracle at the ends of the first and the last tiles."""
    from qfactory import QLinear
    from qfactory.core import tiling
    N, K = 33281, 4608
    assert tiling.gemm_wide_tiling(32, N, K, 4, 128)["WN"] == 7
    A, weight, scale, zero = make_problem(7, 32, N, K, 4, 128)
    layer = QLinear.init(32, K, N, 4, weight.cuda(), 128, scale.cuda(), zero.cuda(), compile_flags=NO_SEARCH)
    rows = [*range(230), *range(N - 360, N)]
    want = reference_output(oracle, A, layer.w, layer.s, layer.z, 4, 128, rows=rows)
    whole = layer(A.cuda())
    assert_close(oracle, whole.cpu().numpy()[:, rows], want, "32 rows")
    assert torch.equal(layer(A[:17].cuda()), whole[:17])


def test_every_tiling_of_a_search(oracle):
    """All candidates of a search on a ragged problem (windows of K that do not deal evenly over the groups among them)
    against the oracle: a search may pick any."""
    from qfactory import QLinear
    from qfactory.jit import jit
    case = prebuild.search_cases()[1]
    M, N, K, nbits, GS = (case[k] for k in ("M", "N", "K", "NBITS", "GS"))
    rows = M - 3
    A, weight, scale, zero = make_problem(91, rows, N, K, nbits, GS)
    layer = QLinear.init(1, K, N, nbits, weight.cuda(), GS, scale.cuda(), zero.cuda(), compile_flags=NO_SEARCH)
    ref = reference_output(oracle, A, layer.w, layer.s, layer.z, nbits, GS)
    x = A.cuda()
    (qfunc,) = prebuild.qfuncs_of(case)
    for cand in qfunc.lower():
        print(f"[case] {cand.tiling_configs}", flush=True)
        out = torch.full((rows, N), float("nan"), dtype=torch.float16, device="cuda")
        _launch(jit.compile(cand), x, layer, out)
        assert_close(oracle, out.cpu().numpy(), ref, str(cand.tiling_configs))


@pytest.mark.parametrize("rows", [129, 192, 193, 256])
def test_both_tilings_of_a_row_count_bucket(oracle, rows):
    """The object of the 256-row bucket holds a tiling for launches of at most 192 rows and one for the others."""
    from qfactory import QLinear
    from qfactory.core import tiling
    N, K = 12288, 1024
    assert tiling.gemm_wide_low_tiling(256, N, K, 4, 128) not in (None, tiling.gemm_wide_tiling(256, N, K, 4, 128))
    A, weight, scale, zero = make_problem(rows, rows, N, K, 4, 128)
    layer = QLinear.init(256, K, N, 4, weight.cuda(), 128, scale.cuda(), zero.cuda(), compile_flags=NO_SEARCH)
    out = layer(A.cuda())
    columns = list(range(0, N, 97))
    ref = reference_output(oracle, A, layer.w, layer.s, layer.z, 4, 128, rows=columns)
    assert_close(oracle, out[:, columns].cpu().numpy(), ref, f"{rows} rows")
