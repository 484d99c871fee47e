"""Gated attention of a prompt (``attn_seq``) against float64: token counts around the 16-row waves
and 64-row tiles, contexts before the prompt that shift the diagonal through the key tiles, every
head dim, both dtypes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

# (batch, tokens, position of the first, cache length, heads, kv heads, head dim, rotary dim, dtype)
CASES = [(1, 2, 0, 2, 2, 1, 64, 16, torch.float16), (2, 15, 3, 40, 4, 2, 128, 128, torch.float16),
         (1, 16, 0, 64, 3, 1, 256, 64, torch.float16), (1, 17, 47, 64, 6, 1, 256, 64, torch.bfloat16),
         (2, 63, 1, 100, 4, 4, 64, 64, torch.bfloat16), (1, 64, 64, 128, 2, 1, 256, 64, torch.float16),
         (1, 65, 63, 512, 6, 2, 256, 64, torch.float16), (1, 130, 333, 463, 2, 1, 128, 32, torch.bfloat16),
         (1, 300, 0, 1024, 24, 4, 256, 64, torch.float16)]


def _reference(qg, k, v, qw, kw, freq, kc, vc, pos, H, G, hd, rd, eps):
    """(out, k cache, v cache) with float64 arithmetic and the kernel's roundings of q and k."""
    B, S, _ = qg.shape
    dt = qg.dtype
    q, gate = qg.double().reshape(B, S, H, 2 * hd).split(hd, -1)

    def norm_rope(t, w):
        t = (t * torch.rsqrt(t.square().mean(-1, keepdim=True) + eps) * w.double()).to(dt).double()
        ang = torch.arange(pos, pos + S).double()[:, None] * freq
        c, s = ang.cos()[None, :, None], ang.sin()[None, :, None]
        lo, hi = t[..., :rd // 2], t[..., rd // 2:rd]
        return torch.cat([lo * c - hi * s, hi * c + lo * s, t[..., rd:]], -1).to(dt)
    q, k = norm_rope(q, qw).double(), norm_rope(k.double().reshape(B, S, G, hd), kw)
    kc, vc = kc.clone(), vc.clone()
    kc[:, :, pos:pos + S] = k.transpose(1, 2)
    vc[:, :, pos:pos + S] = v.reshape(B, S, G, hd).transpose(1, 2)
    K, V = (t[:, :, :pos + S].double().repeat_interleave(H // G, 1) for t in (kc, vc))
    sc = torch.matmul(q.transpose(1, 2), K.transpose(2, 3).contiguous()) * hd ** -0.5
    later = torch.arange(pos + S)[None, :] > torch.arange(pos, pos + S)[:, None]
    att = torch.matmul(torch.softmax(sc.masked_fill(later, float("-inf")), -1), V).transpose(1, 2)
    return (att * torch.sigmoid(gate)).reshape(B, S, H * hd), kc, vc


def _inputs(case, seed=0):
    B, S, pos, L, H, G, hd, rd, dtype = case
    g = torch.Generator().manual_seed(seed + S)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(dtype)
    qk, v = rnd(B, S, H * 2 * hd + G * hd), rnd(B, S, G * hd)
    freq = 1e4 ** (-torch.arange(0, rd, 2).double() / rd)
    return qk, v, 2 + rnd(hd), 2 + rnd(hd), freq, rnd(B, G, L, hd), rnd(B, G, L, hd)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)).replace("torch.", ""))
def test_attn_seq_matches_float64(case):
    from mlx_gsq_amd.runtime.kernels import model_ops
    B, S, pos, L, H, G, hd, rd, dtype = case
    qk, v, qw, kw, freq, kc, vc = _inputs(case)
    n = H * 2 * hd
    want, wk, wv = _reference(qk[..., :n], qk[..., n:], v, qw, kw, freq, kc, vc, pos, H, G, hd, rd, 1e-6)
    d = qk.cuda()
    gk, gv = kc.cuda(), vc.cuda()
    got = model_ops.attn_seq(d[..., :n], d[..., n:], v.cuda(), qw.cuda(), kw.cuda(), freq.cuda(), gk, gv,
                             torch.tensor([pos], device="cuda"), heads=H, kv_heads=G, head_dim=hd, rotary_dim=rd,
                             eps=1e-6)

    def err(a, b):
        return float((a.double().cpu() - b.double()).norm() / b.double().norm())
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)  # spacing of the dtype's values, relative
    # q and k may round differently at ties of the fp32 against the float64 norm (a few in a
    # thousand values, one ulp each); a score of about 5 moves by that share of an ulp
    assert err(gk, wk) <= 0.1 * ulp
    assert torch.equal(gv.cpu(), wv)
    # one rounding of the output (half an ulp at most per value) plus the scores' shift
    assert err(got, want) <= ulp
    assert torch.isfinite(got).all()


def test_attn_seq_precision():
    """Probabilities and their sums stay at fp32 accuracy: with values V in {1, 1 + ulp} times powers
    of two the outputs' float64 error is that of the final rounding alone (fp16 0.29 ulp rms)."""
    from mlx_gsq_amd.runtime.kernels import model_ops
    case = (1, 256, 0, 256, 2, 1, 128, 0, torch.float16)
    B, S, pos, L, H, G, hd, rd, dtype = case
    qk, v, qw, kw, freq, kc, vc = _inputs(case, 5)
    v = (1 + v.sign() * 2.0 ** -10).to(dtype)
    n = H * 2 * hd
    qk[..., :n].view(B, S, H, 2 * hd)[..., hd:] = 20.0  # gates of 1
    want, _, _ = _reference(qk[..., :n], qk[..., n:], v, qw, kw, freq, kc, vc, pos, H, G, hd, rd, 1e-6)
    d = qk.cuda()
    got = model_ops.attn_seq(d[..., :n], d[..., n:], v.cuda(), qw.cuda(), kw.cuda(), freq.cuda(), kc.cuda(), vc.cuda(),
                             torch.tensor([pos], device="cuda"), heads=H, kv_heads=G, head_dim=hd, rotary_dim=rd, eps=1e-6)
    # values near 1 lie 2^-10 (above) or 2^-11 (below) apart: never off by more than half a step,
    # plus 64 fp32 ulps (4e-6) for 256-term sums, scores and exponentials
    assert float((got.double().cpu() - want).abs().max()) <= 2.0 ** -11 + 4e-6


def test_attn_seq_outside_the_cache():
    """Tokens that do not all fit: NaN rows, caches untouched; more tokens than positions: refused."""
    from mlx_gsq_amd.runtime.kernels import model_ops
    case = (1, 20, 0, 32, 2, 1, 64, 16, torch.float16)
    B, S, pos, L, H, G, hd, rd, dtype = case
    qk, v, qw, kw, freq, kc, vc = _inputs(case)
    n = H * 2 * hd
    d = qk.cuda()

    def run(p, kc_, vc_):
        return model_ops.attn_seq(d[..., :n], d[..., n:], v.cuda(), qw.cuda(), kw.cuda(), freq.cuda(), kc_, vc_,
                                  torch.tensor([p], device="cuda"), heads=H, kv_heads=G, head_dim=hd, rotary_dim=rd,
                                  eps=1e-6)
    for p in (13, -1):
        gk, gv = kc.cuda(), vc.cuda()
        assert torch.isnan(run(p, gk, gv)).all()
        assert torch.equal(gk.cpu(), kc) and torch.equal(gv.cpu(), vc)
    assert torch.isfinite(run(12, kc.cuda(), vc.cuda())).all()
    with pytest.raises(ValueError):
        run(0, kc.cuda()[:, :, :16].contiguous(), vc.cuda()[:, :, :16].contiguous())


def _seq(case, qk, v, qw, kw, freq, kc, vc, chunk=None):
    from mlx_gsq_amd.runtime.kernels import model_ops
    B, S, pos, L, H, G, hd, rd, dtype = case
    n, d = H * 2 * hd, qk.cuda()
    gk, gv = kc.cuda(), vc.cuda()
    out = model_ops.attn_seq(d[..., :n], d[..., n:], v.cuda(), qw.cuda(), kw.cuda(), freq.cuda(), gk, gv,
                             torch.tensor([pos], device="cuda"), heads=H, kv_heads=G, head_dim=hd, rotary_dim=rd, eps=1e-6,
                             chunk=chunk)
    return out.cpu(), gk.cpu(), gv.cpu()


# (case, positions per workgroup): chunks that start inside, end at and lie past a query tile's last
# key, a single token of a tile in a chunk, an odd number of key tiles in the last chunk
SPLITS = [((1, 2, 126, 300, 2, 1, 256, 64, torch.float16), 128), ((2, 3, 255, 1000, 4, 2, 128, 128, torch.float16), 256),
          ((1, 70, 100, 700, 3, 1, 64, 16, torch.bfloat16), 128), ((1, 16, 1000, 1100, 6, 2, 256, 64, torch.bfloat16), 384),
          ((1, 130, 0, 900, 2, 1, 128, 32, torch.float16), 128), ((1, 9, 3000, 8192, 24, 4, 256, 64, torch.float16), 1024)]


@pytest.mark.parametrize("case,chunk", SPLITS, ids=lambda c: str(c).replace("torch.", ""))
def test_attn_seq_split(case, chunk):
    """Positions split over workgroups: the float64 result and the unsplit kernel's, whose sums differ
    from the split ones in their last fp32 bits only."""
    B, S, pos, L, H, G, hd, rd, dtype = case
    t = _inputs(case, 1)
    want, wk, wv = _reference(t[0][..., :H * 2 * hd], t[0][..., H * 2 * hd:], *t[1:], pos, H, G, hd, rd, 1e-6)
    got, gk, gv = _seq(case, *t, chunk=chunk)
    whole, hk, hv = _seq(case, *t, chunk=0)

    def err(a, b):
        return float((a.double() - b.double()).norm() / b.double().norm())
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert torch.equal(gk, hk) and torch.equal(gv, hv)
    assert err(got, want) <= ulp
    # a last fp32 bit moves few roundings of the output, one ulp each: a thousandth of the values at most
    # differ by half an ulp of the largest in 2-norm
    assert err(got, whole) <= 0.1 * ulp


def test_attn_seq_split_outside_the_cache():
    case = (1, 20, 0, 512, 2, 1, 64, 16, torch.float16)
    t = _inputs(case, 2)
    for pos in (493, -1):
        out, k, v = _seq(case[:2] + (pos,) + case[3:], *t, chunk=128)
        assert torch.isnan(out).all() and torch.equal(k, t[5]) and torch.equal(v, t[6])
    assert torch.isfinite(_seq(case[:2] + (492,) + case[3:], *t, chunk=128)[0]).all()
    for chunk in (64, 200):
        with pytest.raises(ValueError):
            _seq(case, *t, chunk=chunk)


@pytest.mark.parametrize("chunk", [0, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("order", ["rising", "falling", "even tiles", "odd tiles"])
def test_attn_seq_score_spread(order, dtype, chunk):
    """Scores that rise or fall over hundreds of keys, or lie 45 apart between the even and the odd key
    tiles: the running maximum moves in every tile, or one of the two wave groups holds nothing
    that matters. q and k are +-2 throughout (their norm rounds to exactly that), so only the fp32
    softmax and the output's rounding separate the result from float64."""
    case = (1, 200, 130, 330, 2, 1, 128, 0, dtype)
    B, S, pos, L, H, G, hd, rd, _ = case
    qk, v, qw, kw, freq, kc, vc = _inputs(case, 3)
    key = torch.arange(L)
    match = {"rising": key * hd // L, "falling": hd - key * hd // L,
             "even tiles": (key // 64 % 2 == 0) * 64 + 64 - key % 7, "odd tiles": (key // 64 % 2) * 64 + 64 - key % 7}[order]
    k = torch.where(torch.arange(hd)[None, :] < match[:, None], 1.0, -1.0).to(dtype)  # agrees with q in `match` dims
    n = H * 2 * hd
    qg = qk[..., :n].view(B, S, H, 2 * hd)
    qg[..., :hd] = 1.0
    qg[..., hd:] = 20.0  # gates of 1
    qk[..., n:] = k[pos:]
    qw[:], kw[:] = 2.0, 2.0
    kc[0, 0, :pos] = 2 * k[:pos]
    v, vc = (1 + torch.rand(v.shape, generator=torch.Generator().manual_seed(1))).to(dtype), 1 + vc.abs() % 1
    want, wk, _ = _reference(qk[..., :n], qk[..., n:], v, qw, kw, freq, kc, vc, pos, H, G, hd, rd, 1e-6)
    got, gk, _ = _seq(case, qk, v, qw, kw, freq, kc, vc, chunk)
    assert torch.equal(gk, wk)
    # values in [1, 2]: half a step of the dtype there, plus 1e-5: 2^-24 of exponents up to 80, and
    # sums of 330 terms
    half = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert float((got.double() - want).abs().max()) <= half + 1e-5


@pytest.mark.parametrize("chunk", [0, 128])
def test_attn_seq_not_finite(chunk):
    """A NaN or infinity reaches the outputs it belongs to and no others."""
    case = (1, 150, 20, 300, 4, 2, 64, 16, torch.float16)
    B, S, pos, L, H, G, hd, rd, dtype = case
    qk, v, qw, kw, freq, kc, vc = _inputs(case, 4)
    n, t = H * 2 * hd, 70
    clean, _, _ = _seq(case, qk, v, qw, kw, freq, kc, vc, chunk)
    assert torch.isfinite(clean).all()

    def run(qk=qk, v=v, kc=kc, vc=vc):
        return _seq(case, qk, v, qw, kw, freq, kc, vc, chunk)[0]

    def check(got, bad):
        assert torch.isnan(got[bad]).all() and torch.equal(got[~bad], clean[~bad])
    bad = torch.zeros(B, S, H, hd, dtype=torch.bool)
    x = qk.clone()  # a query: its row and head
    x[0, t, 1 * 2 * hd + 5] = float("nan")
    b = bad.clone()
    b[0, t, 1] = True
    check(run(qk=x), b.view(B, S, -1))
    x = qk.clone()  # a gate: its value
    x[0, t, 2 * 2 * hd + hd + 7] = float("nan")
    b = bad.clone()
    b[0, t, 2, 7] = True
    check(run(qk=x), b.view(B, S, -1))
    for bad_value in (float("nan"), float("inf")):  # a key: rows from its token on, of its query heads
        x = qk.clone()
        x[0, t, n + hd + 9] = bad_value
        b = bad.clone()
        b[0, t:, 2:] = True
        check(run(qk=x), b.view(B, S, -1))
    # a value: its dim, from its token on (and, masked by a weight of 0, before it in its key tile)
    y = v.clone()
    y[0, t, hd + 11] = float("inf")
    got = run(v=y).view(B, S, H, hd)
    c = clean.view(B, S, H, hd)
    assert not torch.isfinite(got[0, t:, 2:, 11]).any()
    other = torch.ones(H, hd, dtype=torch.bool)
    other[2:, 11] = False
    assert torch.equal(got[:, :, other], c[:, :, other])
    # positions past the new tokens hold anything
    kc2, vc2 = kc.clone(), vc.clone()
    kc2[:, :, pos + S:], vc2[:, :, pos + S:] = float("nan"), float("inf")
    assert torch.equal(run(kc=kc2, vc=vc2), clean)
