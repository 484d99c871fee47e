"""Activations that ``gsq_qmm`` stages as fp16 (fp32, bf16, fp16 not 16-byte aligned): the result is
that of the product on the same values as aligned fp16, bit for bit, over both fp16 kernels'
ranges, and in pieces when the rows exceed the staging area."""
import pytest
import torch

from mlx_gsq_amd import synth, tables

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)


def _call(qtype, packed, x, m, n, k, code):
    from mlx_gsq_amd import _lib
    from mlx_gsq_amd.formats import TYPE_IDS
    y = torch.full((m, n), float("nan"), device="cuda")
    rc = _lib.lib().gsq_qmm(TYPE_IDS[qtype], packed.data_ptr(), x.data_ptr(), code, y.data_ptr(), 0, m, n, k,
                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib().gsq_last_error()
    return y


@pytest.mark.parametrize("m", [1, 16, 17, 65, 300])
@pytest.mark.parametrize("form", ["bf16", "fp32", "bf16+1", "fp32+1", "fp16+1"])
@pytest.mark.parametrize("qtype,n,k", [("Q4_K", 515, 768), ("IQ3_S", 64, 256)])
def test_staged_matches_fp16(qtype, n, k, form, m):
    from mlx_gsq_amd import _lib
    tables.set_tables(tables.synthetic_tables(0))
    _lib.ensure_tables(qtype, torch.device("cuda:0"))
    packed = torch.from_numpy(synth.make_packed(qtype, n, k, seed=1)).cuda()
    dtype = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp16": torch.float16}[form[:4]]
    off = 1 if form.endswith("+1") else 0  # one element past an aligned address
    x = torch.randn(m * k + 1, generator=torch.Generator().manual_seed(m)).to(dtype).cuda()[off:off + m * k]
    assert (x.data_ptr() % 16 != 0) == bool(off)
    want = _call(qtype, packed, x.half().clone(), m, n, k, 1)
    got = _call(qtype, packed, x, m, n, k, _lib.DTYPE_CODES[dtype])
    assert torch.isfinite(got).all() and torch.equal(got, want)


def test_rows_beyond_the_staging_area():
    """128 MB of fp16 staging hold 3855 rows of K = 17408: 4000 rows go in two pieces of 2048 and 1952."""
    m, n, k = 4000, 40, 17408
    packed = torch.from_numpy(synth.make_packed("Q4_K", n, k, seed=2)).cuda()
    x = torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(3)).bfloat16()
    got = _call("Q4_K", packed, x, m, n, k, 2)
    h = x.half()
    want = torch.cat([_call("Q4_K", packed, h[a:b], b - a, n, k, 1) for a, b in ((0, 2048), (2048, 4000))])
    assert torch.isfinite(got).all() and torch.equal(got, want)


@pytest.mark.parametrize("m", [20, 130])
def test_captured_on_a_prepared_stream(m):
    """bf16 rows captured on a stream prepared with a staging area: every replay, between eager calls on
    that stream with other rows, gives the eager result of the aligned fp16 rows."""
    from mlx_gsq_amd import _lib
    from mlx_gsq_amd.formats import TYPE_IDS
    n, k = 520, 1024
    packed = torch.from_numpy(synth.make_packed("Q4_K", n, k, seed=4)).cuda()
    x = torch.empty(m, k, dtype=torch.bfloat16, device="cuda")
    y = torch.empty(m, n, device="cuda")
    other = torch.randn(m + 30, k, device="cuda")
    cap = torch.cuda.Stream()
    _lib.prepare(stream=cap, staging=True)
    cap.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        rc = _lib.lib().gsq_qmm(TYPE_IDS["Q4_K"], packed.data_ptr(), x.data_ptr(), 2, y.data_ptr(), 0, m, n, k,
                                cap.cuda_stream)
    assert rc == 0, _lib.lib().gsq_last_error()
    torch.cuda.synchronize()
    for rep in range(3):
        x.copy_(torch.randn(m, k, generator=torch.Generator().manual_seed(rep)))
        y.fill_(float("nan"))
        want = _call("Q4_K", packed, x.half(), m, n, k, 1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {rep}"
        with torch.cuda.stream(cap):
            _call("Q4_K", packed, other, m + 30, n, k, 0)
        torch.cuda.synchronize()


@pytest.mark.parametrize("m", [12, 90, 200])  # small-batch kernel, one and six blocks; tiled kernel
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("qtype", ["Q4_K", "IQ2_S"])
def test_rows_not_finite(qtype, dtype, m):
    """NaN, infinities and values past fp16's range stay in their rows, where the outputs are those of
    the kernel that stages nothing (up to the sign of NaN)."""
    from mlx_gsq_amd import _lib
    from mlx_gsq_amd.formats import TYPE_IDS
    tables.set_tables(tables.synthetic_tables(0))
    _lib.ensure_tables(qtype, torch.device("cuda:0"))
    _lib.prepare()
    n, k = 300, 512
    packed = torch.from_numpy(synth.make_packed(qtype, n, k, seed=5)).cuda()
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dtype).cuda()
    clean = _call(qtype, packed, x, m, n, k, _lib.DTYPE_CODES[dtype])
    rows = [1, 2, m - 1] if dtype == torch.float16 else [1, 2, 5, m - 1]
    x[1, 300], x[2, 7], x[m - 1, 511] = float("nan"), float("inf"), float("-inf")
    if dtype != torch.float16:
        x[5, 100] = 1e5
    got = _call(qtype, packed, x, m, n, k, _lib.DTYPE_CODES[dtype])
    ref, xf = torch.full((m, n), 0.5, device="cuda"), x.float()
    rc = _lib.lib().gsq_qmm_noalloc(TYPE_IDS[qtype], packed.data_ptr(), xf.data_ptr(), 0, ref.data_ptr(), 0, m, n, k,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib().gsq_last_error()
    fine = torch.ones(m, dtype=torch.bool)
    fine[rows] = False
    assert torch.isfinite(clean).all() and torch.equal(got[fine.cuda()], clean[fine.cuda()])
    assert not torch.isfinite(got[rows]).any()
    torch.testing.assert_close(got[rows], ref[rows], rtol=0, atol=0, equal_nan=True)
