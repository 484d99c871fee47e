"""Which calls of the gated attention layer with several tokens go to the prompt kernel, and that those
it does not take get the torch formulation's result (values, cache and gradients) on a GPU as well."""
import copy

import pytest
import torch

from mlx_gsq_amd.models import Qwen35Args
from mlx_gsq_amd.models.qwen35 import FullAttention, Qwen35Cache

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def _args(hd):
    return Qwen35Args(hidden_size=64, num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2, head_dim=hd)


def _layer(hd=64, dtype=F16, seed=0):
    a, g = _args(hd), torch.Generator().manual_seed(seed)

    def lin(n, k):
        m = torch.nn.Linear(k, n, bias=False)
        m.weight = torch.nn.Parameter((torch.randn(n, k, generator=g) * k ** -0.5).to(dtype), requires_grad=False)
        return m
    return FullAttention(a, 3, lin(4 * 2 * hd + 2 * hd, 64), lin(2 * hd, 64), lin(64, 4 * hd),
                         (1 + torch.rand(hd, generator=g)).to(dtype), (1 + torch.rand(hd, generator=g)).to(dtype))


def _x(S=9, dtype=F16, B=1, seed=1):
    return torch.randn(B, S, 64, generator=torch.Generator().manual_seed(seed)).to(dtype)


def _cache(layer, L=32, dtype=F16, B=1):
    return Qwen35Cache(layer.args, B, L, "cpu", dtype)


def _strided(t):
    out = torch.empty(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device=t.device)[..., ::2]
    return out.copy_(t)


def _shifted(t):  # contiguous, one value past an aligned address
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


def _taken(layer, x, cache, qk=None, v=None):
    qk = layer.qk_proj(x) if qk is None else qk
    return layer._seq_kernel(x, qk, layer.v_proj(x) if v is None else v, cache)


def test_kernel_takes_16_bit_prompts():
    for hd in (64, 128, 256):
        for dtype in (F16, BF16):
            layer = _layer(hd, dtype)
            assert _taken(layer, _x(dtype=dtype), _cache(layer, dtype=dtype))
    layer = _layer()
    assert _taken(layer, _x(S=32), _cache(layer, L=32))
    with torch.no_grad():
        assert _taken(layer, _x().requires_grad_(), _cache(layer))


def test_kernel_refuses():
    layer, x = _layer(), _x()
    cache = _cache(layer)
    assert _taken(layer, x, cache)
    # dtypes
    assert not _taken(_layer(dtype=F32), _x(dtype=F32), _cache(layer, dtype=F32))
    assert not _taken(layer, x, _cache(layer, dtype=F32))
    assert not _taken(layer, x.float(), cache, qk=layer.qk_proj(x), v=layer.v_proj(x))
    for name in ("q_norm_w", "k_norm_w"):
        other = _layer()
        setattr(other, name, getattr(other, name).float())
        assert not _taken(other, x, cache)
        other = _layer()
        setattr(other, name, _strided(getattr(other, name)))
        assert not _taken(other, x, cache)
    other = _layer()
    other.inv_freq = other.inv_freq.float()
    assert not _taken(other, x, cache)
    # head dims without a kernel, more tokens than positions, more sequences than a launch has
    assert not _taken(_layer(96), x, _cache(_layer(96)))
    assert not _taken(layer, _x(S=33), _cache(layer, L=32))
    for B, taken in ((65535, True), (65536, False)):
        assert layer._seq_kernel(x, torch.empty(B, 2, 640, dtype=F16), torch.empty(B, 2, 128, dtype=F16), cache) == taken
    # layouts and alignments
    qk, v = layer.qk_proj(x), layer.v_proj(x)
    for f in (_strided, _shifted):
        assert not _taken(layer, x, cache, qk=f(qk))
        assert not _taken(layer, x, cache, v=f(v))
        c = _cache(layer)
        c.k[3] = f(c.k[3])
        assert not _taken(layer, x, c)


def test_kernel_refuses_derivatives():
    layer = _layer()
    assert not _taken(layer, _x().requires_grad_(), _cache(layer))
    other = _layer()
    other.v_proj.weight.requires_grad_()
    assert not _taken(other, _x(), _cache(other))
    other = _layer()
    other.k_norm_w.requires_grad_()
    assert not _taken(other, _x(), _cache(other))
    with torch.autograd.forward_ad.dual_level():
        x = torch.autograd.forward_ad.make_dual(_x(), _x(seed=2))
        assert not _taken(layer, x, _cache(layer))


def test_positions_per_workgroup():
    """Long caches are split over the CUs that a few query tiles leave idle, into whole pairs of key tiles."""
    from mlx_gsq_amd.runtime.kernels.model_ops import ATTN_SEQ_MIN_CHUNK, attn_seq_chunk
    for wgs in (1, 24, 48, 127, 128, 129, 256, 4000):
        for L in (8192, 8193, 16384, 32768, 100000, 131072, 1 << 20):
            c = attn_seq_chunk(wgs, L, 256)
            if wgs > 128:
                assert c == 0
                continue
            n = -(-L // c)
            assert c % 128 == 0 and c >= ATTN_SEQ_MIN_CHUNK and 1 < n and n * wgs <= 256
    assert attn_seq_chunk(24, 8191, 256) == 0 and attn_seq_chunk(24, 32768, 256) == 4096


def _run(layer, x, cache, device):
    layer, cache, x = copy.deepcopy(layer).to(device), copy.deepcopy(cache), x.to(device)
    cache.pos = cache.pos.to(device)
    for c in (cache.k, cache.v):
        for i in c:
            c[i] = c[i].to(device)
    with torch.no_grad():
        y = layer(x, cache)
    return y, cache.k[3], cache.v[3]


# (head dim, layer dtype, cache dtype, tokens, taken)
ROUTES = [(64, F16, F16, 70, True), (128, BF16, BF16, 9, True), (96, F16, F16, 9, False), (64, F16, F32, 9, False),
          (64, F32, F32, 9, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("hd,dtype,cdtype,S,taken", ROUTES)
def test_layer_on_gpu_matches_cpu(hd, dtype, cdtype, S, taken):
    """The layer on a GPU, by either route, against its torch formulation on the CPU."""
    layer, x = _layer(hd, dtype), _x(S, dtype, B=2)
    cache = _cache(layer, 80, cdtype, B=2)
    for c in (cache.k, cache.v):
        c[3].copy_(_x(seed=3, S=c[3].numel() // 64).view(c[3].shape))
    cache.pos.fill_(5)
    cache.length = 5
    assert _taken(layer, x, cache) == taken
    for got, want in zip(_run(layer, x, cache, "cuda"), _run(layer, x, cache, "cpu")):
        assert got.dtype == want.dtype
        # the projections' sums differ in their last fp32 bits, which flips some of the roundings to
        # `dtype` after them (one ulp each); their sums through the layer stay below half an ulp
        # (2-norm over 2-norm), against fp32's 4e-5 for the fp32 layer
        tol = {F16: 2.0 ** -11, BF16: 2.0 ** -8, F32: 4e-5}[dtype]
        assert float((got.double().cpu() - want.double()).norm() / want.double().norm()) <= tol


@pytest.mark.gpu
def test_gradients_on_gpu():
    """A layer of differentiable projections: gradients reach x through the torch formulation."""
    layer, x = _layer(64, F32), _x(9, F32)
    grads = []
    for device in ("cpu", "cuda"):
        m, xi = copy.deepcopy(layer).to(device), x.detach().to(device).requires_grad_()
        y = m(xi, Qwen35Cache(layer.args, 1, 16, device, F32))
        (y * torch.arange(y.numel(), device=device).view(y.shape)).sum().backward()
        grads.append(xi.grad.double().cpu())
    assert float((grads[0] - grads[1]).norm() / grads[0].norm()) <= 4e-5
    m, xi = copy.deepcopy(_layer()).cuda(), _x().cuda().requires_grad_()
    y = m(xi, Qwen35Cache(layer.args, 1, 16, "cuda", F16))
    y.sum().backward()
    assert xi.grad is not None and bool(torch.isfinite(xi.grad).all()) and float(xi.grad.abs().max()) > 0
