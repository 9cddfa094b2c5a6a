"""GPU tests of the few-token dense kernels (``csrc/ffn_small.hip``) at the edges of their tiles, against the persistent
kernels that large batches take (a capped grid selects those) and, through them, the oracle-tested entry points."""

from __future__ import annotations

import pytest
import torch

from taac_2026_amd.api import norm_linear, norm_linear_heads, qkv_projection, valid_rows

pytestmark = pytest.mark.gpu


def _bf16(g, *shape, scale=1.0):
    return (scale * torch.randn(*shape, generator=g)).to(torch.bfloat16)


def _both(test_hooks, call):
    """The call through the few-token kernels and through the persistent ones."""
    small = call()
    test_hooks(max_workgroups=256)
    large = call()
    test_hooks(max_workgroups=0)
    return small, large


@pytest.mark.parametrize("m,k,n", [(1, 256, 768), (31, 128, 384), (33, 256, 64), (64, 256, 320), (130, 128, 192), (10240, 256, 256)])
def test_projection_equals_the_persistent_kernel(device, test_hooks, m, k, n):
    """Same products in the same order: bit for bit, with and without norm, bias and (aliased) residual; output feature
    counts that leave wavefronts of the last workgroup idle."""
    g = torch.Generator().manual_seed(m + n)
    x, w, b = _bf16(g, m, k).to(device), _bf16(g, n, k, scale=k ** -0.5).to(device), _bf16(g, n).to(device)
    nw, res = (1 + _bf16(g, k, scale=0.1)).to(device), _bf16(g, m, n).to(device)
    with torch.no_grad():
        for kw in (dict(), dict(norm_weight=nw), dict(residual=res), dict(norm_weight=nw, residual=res)):
            for bias in (b, None):
                small, large = _both(test_hooks, lambda: norm_linear(x, w, bias, **kw))
                assert torch.equal(small, large)
        held = res.clone()
        norm_linear(x, w, b, residual=held, out=held)
        assert torch.equal(held, norm_linear(x, w, b, residual=res))


@pytest.mark.parametrize("d_model,heads", [(256, 8), (256, 4), (128, 4)])
@pytest.mark.parametrize("norm,rope", [(True, None), (True, 10000.0), (False, 10000.0)])
def test_query_key_epilogue_equals_the_persistent_kernel(device, test_hooks, d_model, heads, norm, rope):
    """Projection, norm factors and rotation over a ragged set of valid rows."""
    g = torch.Generator().manual_seed(d_model + heads)
    batch, tokens = 5, 45
    x, w = _bf16(g, batch, tokens, d_model).to(device), _bf16(g, 3 * d_model, d_model, scale=d_model ** -0.5).to(device)
    b, nw = _bf16(g, 3 * d_model).to(device), (1 + _bf16(g, d_model, scale=0.1)).to(device)
    qw, kw = ((1 + _bf16(g, d_model, scale=0.1)).to(device) for _ in range(2))
    rows = valid_rows(torch.tensor([45, 0, 1, 33, 17], dtype=torch.int32, device=device), tokens)
    with torch.no_grad():
        for index in (None, rows):
            def call():
                out = torch.zeros(batch * tokens, 3 * d_model, dtype=torch.bfloat16, device=device)
                return [t for t in qkv_projection(x, w, b, num_heads=heads, norm_weight=nw, query_weight=qw if norm else None,
                                                  key_weight=kw if norm else None, rope_base=rope, token_rows=index, out=out)
                        if t is not None]
            for small, large in zip(*_both(test_hooks, call)):
                assert torch.equal(small, large)
            if norm and rope is None:
                small, large = _both(test_hooks, lambda: norm_linear_heads(x, w, b, head_dim=d_model // heads, norm_weight=nw,
                                                                           token_rows=index))
                assert torch.equal(small, large)
