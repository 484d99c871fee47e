"""Products at the edges of their tiles and plans: the small-batch kernel (16, 32, 48, 64 and 96 rows;
128 weight rows) and the tiled one (64, 128, 192 and 256 rows; 256 weight rows; whole tiles first, then
tiles split over workgroups and summed by a second launch).

Against the oracle's float32 weights in float64, elementwise. A weight is rounded to fp16 at most
twice (group scale times value, then superblock scale): 2 * 2^-11 of sum |w x|, or 2^-24 |x| where it
is subnormal. K products are summed in fp32: K * 2^-24 of sum |w x|. Then one rounding to the output."""
import pytest
import torch

from mlx_gsq_amd import synth, tables
from oracle import gsq_oracle as O

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

SHAPES = [
    (17, 257, 256),     # one column per tile: nothing to split
    (32, 129, 512),
    (33, 128, 2560),    # one row group over ten workgroups
    (48, 1, 256),
    (49, 127, 768),
    (64, 255, 512),
    (65, 515, 1280),    # six blocks (128-row tiles for Q6_K, IQ1_S), weight rows of odd length
    (96, 40001, 512),   # several columns and parts of two groups per workgroup
    (97, 130, 1280),    # 128-row tiles
    (128, 256, 768),
    (129, 771, 768),    # 192-row tiles
    (192, 64, 2560),
    (193, 1, 512),      # 256-row tiles; a single weight row
    (257, 130, 1024),
    (550, 300, 1280),   # three tiles of 192 rows
    (3100, 5121, 512),  # 273 tiles: a round of whole tiles, then whole ones
    (3100, 5121, 768),  # a round of whole tiles, then 17 tiles over 26 workgroups
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("qtype,out", [("Q4_K", "float32"), ("IQ3_S", "float16"), ("Q6_K", "bfloat16"),
                                       ("IQ2_S", "float32"), ("IQ1_S", "bfloat16")])
def test_tiled_product(qtype, out, shape):
    from mlx_gsq_amd import _lib
    from mlx_gsq_amd.formats import TYPE_IDS
    m, n, k = shape
    T = tables.synthetic_tables(0)
    tables.set_tables(T)
    _lib.ensure_tables(qtype, torch.device("cuda:0"))
    packed = synth.make_packed(qtype, n, k, seed=3)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).half().cuda()
    dt = getattr(torch, out)
    pd = torch.from_numpy(packed).cuda()
    guard = 32  # elements around the result that must stay
    buf = torch.full((m * n + 2 * guard,), 7.0, device="cuda", dtype=dt)
    y = buf[guard:guard + m * n].view(m, n)
    rc = _lib.lib().gsq_qmm(TYPE_IDS[qtype], pd.data_ptr(), x.data_ptr(), 1, y.data_ptr(), _lib.DTYPE_CODES[dt],
                            m, n, k, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib().gsq_last_error()
    w = torch.from_numpy(O.dequantize_reference(packed, qtype, T.get(qtype))).double().reshape(n, k).cuda()
    xd = x.double()
    want, mag = xd @ w.t(), xd.abs() @ w.abs().t()
    tol = (2 * 2.0**-11 + k * 2.0**-24) * mag + 2.0**-24 * xd.abs().sum(1, keepdim=True)
    eps = {"float32": 2.0**-24, "float16": 2.0**-11, "bfloat16": 2.0**-9}[out]
    tol = tol + 2 * eps * want.abs() + (2.0**-25 if out == "float16" else 0)
    err = (y.double() - want).abs()
    assert torch.isfinite(y).all() and (err <= tol).all(), float((err / tol).max())
    assert (buf[:guard] == 7).all() and (buf[guard + m * n:] == 7).all()
