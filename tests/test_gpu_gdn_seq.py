"""GatedDeltaNet over a sequence (``gdn_seq``) against a float64 recurrence: lengths around the
staged chunk of 16 tokens, and of the convolution's runs of 8, every key head dim the column-split
kernels take (and one they do not), odd row strides, each activation dtype."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

# (batch, tokens, key heads, value heads, key dim, value dim, convolution kernel, row padding, dtype)
CASES = [(1, 1, 2, 2, 128, 64, 4, 0, torch.float16), (2, 2, 2, 6, 128, 128, 4, 0, torch.float16),
         (1, 15, 3, 3, 64, 64, 2, 0, torch.float16), (1, 16, 1, 2, 32, 192, 4, 0, torch.bfloat16),
         (2, 17, 2, 4, 128, 128, 8, 2, torch.float16), (1, 33, 3, 3, 32, 256, 3, 1, torch.float16),
         (1, 40, 8, 16, 64, 128, 4, 3, torch.float32), (1, 129, 2, 6, 128, 128, 4, 0, torch.float16),
         (1, 9, 2, 4, 96, 64, 4, 0, torch.float16)]


def _reference(qkv, z, ab, conv, cw, ssm_a, dt, rec, nw, hk, hv, dk, dv, eps):
    """The recurrence in float64; conv and rec are the states before the sequence."""
    B, S, C = qkv.shape
    K = cw.shape[1]
    x = torch.cat([conv, qkv], 1)
    y = sum(x[:, j:j + S] * cw[:, j] for j in range(K))
    y = y * torch.sigmoid(y)
    q, k, v = y.split([hk * dk, hk * dk, hv * dv], -1)

    def norm(t, n, e):
        t = t.reshape(B, S, -1, n)
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + e)
    q = (norm(q, dk, 1e-6) / dk).repeat(1, 1, hv // hk, 1)
    k = (norm(k, dk, 1e-6) * dk ** -0.5).repeat(1, 1, hv // hk, 1)
    v = v.reshape(B, S, hv, dv)
    beta = torch.sigmoid(ab[..., hv:])
    decay = torch.exp(ssm_a * torch.nn.functional.softplus(ab[..., :hv] + dt))
    outs = []
    for t in range(S):
        rec = rec * decay[:, t, :, None, None]
        delta = (v[:, t] - (rec * k[:, t, :, :, None]).sum(-2)) * beta[:, t, :, None]
        rec = rec + k[:, t, :, :, None] * delta[:, :, None, :]
        outs.append((rec * q[:, t, :, :, None]).sum(-2))
    out = norm(torch.stack(outs, 1).reshape(B, S, -1), dv, eps) * nw
    zz = z.reshape(B, S, hv, dv)
    return (out * zz * torch.sigmoid(zz)).reshape(B, S, -1), x[:, S:], rec


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)).replace("torch.", ""))
def test_gdn_seq_matches_float64(case):
    from mlx_gsq_amd.runtime.kernels import model_ops
    B, S, hk, hv, dk, dv, K, pad, dtype = case
    g = torch.Generator().manual_seed(S + dk)
    C = 2 * hk * dk + hv * dv

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(dtype)
    rows = rnd(B, S, C + hv * dv + pad)
    qkv, z = rows[..., :C], rows[..., C:C + hv * dv]
    ab, conv, cw, nw = rnd(B, S, 2 * hv), rnd(B, K - 1, C), 0.5 * rnd(C, K), 1 + 0.1 * rnd(dv)
    ssm_a, dt = -torch.exp(2 * torch.rand(hv, generator=g)), torch.randn(hv, generator=g) - 2
    rec = torch.randn(B, hv, dk, dv, generator=g)
    want, wconv, wrec = _reference(*(t.double() for t in (qkv, z, ab, conv, cw, ssm_a, dt, rec, nw)), hk, hv, dk, dv, 1e-6)
    d = rows.cuda()
    gconv, grec = conv.cuda(), rec.cuda()
    got = model_ops.gdn_seq(d[..., :C], d[..., C:C + hv * dv], ab.cuda(), gconv, cw.cuda(), ssm_a.cuda(), dt.cuda(), grec,
                            nw.cuda(), key_heads=hk, value_heads=hv, head_k_dim=dk, head_v_dim=dv, eps=1e-6)

    def err(a, b):
        return float((a.double().cpu() - b).norm() / b.norm())
    # one rounding to the output dtype (relative 2^-11, 2^-8, 2^-24 at most per value), and fp32
    # sums of up to 128 terms carried over the tokens: a few ulp (6e-8) each
    half_ulp = {torch.float16: 2 ** -11, torch.bfloat16: 2 ** -8, torch.float32: 2 ** -24}[dtype]
    assert err(got, want) <= half_ulp + 2e-6
    assert err(grec, wrec) <= 2e-6
    assert torch.equal(gconv.cpu().double(), wconv)


@pytest.mark.parametrize("dk", [128, 96])  # column-split kernels; the whole-head one
def test_gdn_seq_not_finite(dk):
    """A NaN in one token's value reaches that head's outputs from there on and its state's column, and
    nothing else; a NaN or infinity in a state likewise."""
    from mlx_gsq_amd.runtime.kernels import model_ops
    B, S, hk, hv, dv, K = 1, 50, 2, 4, 64, 4
    g = torch.Generator().manual_seed(dk)
    C = 2 * hk * dk + hv * dv

    def rnd(*shape):
        return torch.randn(*shape, generator=g).half()
    qkv, z, ab, conv, cw, nw = rnd(B, S, C), rnd(B, S, hv * dv), rnd(B, S, 2 * hv), rnd(B, K - 1, C), rnd(C, K), rnd(dv)
    ssm_a, dt = -torch.rand(hv, generator=g), torch.randn(hv, generator=g)
    rec = torch.randn(B, hv, dk, dv, generator=g)

    def run(qkv=qkv, rec=rec):
        gconv, grec = conv.cuda(), rec.cuda()
        out = model_ops.gdn_seq(qkv.cuda(), z.cuda(), ab.cuda(), gconv, cw.cuda(), ssm_a.cuda(), dt.cuda(), grec, nw.cuda(),
                                key_heads=hk, value_heads=hv, head_k_dim=dk, head_v_dim=dv, eps=1e-6)
        return out.cpu().view(S, hv, dv), grec.cpu()
    out0, rec0 = run()
    assert torch.isfinite(out0).all() and torch.isfinite(rec0).all()
    t, h, j = 21, 2, 37
    x = qkv.clone()
    x[0, t, 2 * hk * dk + h * dv + j] = float("nan")
    out, r = run(qkv=x)
    bad = torch.zeros(S, hv, dtype=torch.bool)
    bad[t:, h] = True
    assert torch.isnan(out[bad]).all() and torch.equal(out[~bad], out0[~bad])
    col = torch.zeros(hv, dv, dtype=torch.bool)
    col[h, j] = True
    assert torch.isnan(r[0].transpose(1, 2)[col]).all()
    assert torch.equal(r[0].transpose(1, 2)[~col], rec0[0].transpose(1, 2)[~col])
    for bad_value in (float("nan"), float("inf")):
        y = rec.clone()
        y[0, h, 3, j] = bad_value
        out, r = run(rec=y)
        assert torch.isnan(out[:, h, j]).all() and torch.equal(out[:, [0, 1, 3]], out0[:, [0, 1, 3]])
        assert torch.equal(r[0].transpose(1, 2)[~col], rec0[0].transpose(1, 2)[~col])
