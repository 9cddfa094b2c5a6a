"""GPU tests of the few-token dense kernels (``csrc/ffn_small.hip``) at the edges of their tiles, against the persistent
kernels that large batches take (a capped grid selects those) and, through them, the oracle-tested entry points."""

from __future__ import annotations

import copy
import threading

import pytest
import torch

from taac_2026_amd import workloads
from taac_2026_amd.api import (PCVRBackbone, attention_out_ffn, attention_out_ffn_heads, norm_linear, norm_linear_heads, qkv_projection,
                               swiglu_ffn, valid_rows)

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


def _near_but_for_roundings(small, large):
    """At most a step of bf16 apart, at few values (one token may be a test's only one)."""
    torch.testing.assert_close(small.float(), large.float(), rtol=2 ** -7, atol=2 ** -6)
    assert (small != large).float().mean() <= 2 ** -5 + 1 / small.shape[0]


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


@pytest.mark.parametrize("m,k,heads,valid", [(5475, 256, 8, 1.0), (12001, 256, 4, 0.7), (16417, 128, 4, 1.0), (32768, 256, 8, 0.3)])
def test_projection_of_several_tiles_per_workgroup(device, test_hooks, m, k, heads, valid):
    """More tiles than columns of workgroups (two workgroups per compute unit and part at K = 256, six at 128), or columns beyond
    the valid tokens: bit for bit the persistent kernel's rows, and no others written."""
    g = torch.Generator().manual_seed(m)
    x, w, b = _bf16(g, 1, m, k).to(device), _bf16(g, 3 * k, k, scale=k ** -0.5).to(device), _bf16(g, 3 * k).to(device)
    nw, res = (1 + _bf16(g, k, scale=0.1)).to(device), _bf16(g, m, 3 * k).to(device)
    rows = valid_rows(torch.tensor([int(m * valid)], dtype=torch.int32, device=device), m)
    with torch.no_grad():
        def call():
            blank = torch.full((m, 3 * k), 7.0, dtype=torch.bfloat16, device=device)
            qk = qkv_projection(x, w, b, num_heads=heads, norm_weight=nw, query_weight=nw, key_weight=nw, rope_base=1e4, token_rows=rows,
                                out=blank.clone())
            return [norm_linear(x[0], w, b, norm_weight=nw, token_rows=rows, out=blank.clone()),
                    norm_linear(x[0], w, b, residual=res, token_rows=rows, out=blank.clone()), *(t for t in qk if t is not None)]
        small, large = _both(test_hooks, call)
        for a, c in zip(small, large):
            assert torch.equal(a, c)
        assert (small[0][int(m * valid):] == 7.0).all()


@pytest.mark.parametrize("m,d,f", [(1, 256, 32), (33, 128, 32), (31, 256, 96), (64, 128, 512), (100, 256, 1024), (8192, 256, 64)])
@pytest.mark.parametrize("gate_first", [True, False])
def test_feed_forward_matches_the_persistent_kernel(device, test_hooks, m, d, f, gate_first):
    """Both add the hidden units up in one order: without a norm and a projection in front the same bits. The norm's sum of squares
    meets from other partial sums and the projection's bias joins at another place, which moves a normalised value or x1 by about
    2**-20 of its terms. Bound: that flips a rounding to bf16 where the value lies that near to one, at one value in 2**12: of the
    layer output before the residual joins (magnitude below 4 here, one step = 2**-6 at most, whole when the residual cancels the
    value) and of the result (one step, 2**-7 relative). Few tokens have such a value in front of their products (a flipped
    normalised input or hidden unit is worth less than 2**-9 in a sum), and few of their outputs then lie near a rounding."""
    g = torch.Generator().manual_seed(m + f)
    x, res, nw = _bf16(g, m, d).to(device), _bf16(g, m, d).to(device), (1 + _bf16(g, d, scale=0.1)).to(device)
    wo, bo = _bf16(g, d, d, scale=d ** -0.5).to(device), _bf16(g, d, scale=0.1).to(device)
    wu, bu = _bf16(g, 2 * f, d, scale=d ** -0.5).to(device), _bf16(g, 2 * f, scale=0.1).to(device)
    wd, bd = _bf16(g, d, f, scale=f ** -0.5).to(device), _bf16(g, d, scale=0.1).to(device)

    def check(call):
        _near_but_for_roundings(*_both(test_hooks, call))

    with torch.no_grad():
        for fold in (True, False):
            check(lambda: swiglu_ffn(x, wu, bu, wd, bd, residual=res, gate_first=gate_first, norm_weight=nw, fold_activation=fold))
            for bias in ((bu, bd), (None, None)):
                small, large = _both(test_hooks, lambda: swiglu_ffn(x, wu, bias[0], wd, bias[1], gate_first=gate_first, fold_activation=fold))
                assert torch.equal(small, large)
            if gate_first:
                check(lambda: attention_out_ffn(x, wo, bo, res, wu, bu, wd, bd, norm_weight=nw, fold_activation=fold))
                planes = x.view(m, -1, 32).permute(1, 0, 2).contiguous()
                assert torch.equal(attention_out_ffn_heads(planes, wo, bo, res, wu, bu, wd, bd, norm_weight=nw, fold_activation=fold),
                                   attention_out_ffn(x, wo, bo, res, wu, bu, wd, bd, norm_weight=nw, fold_activation=fold))
        held = res.clone()
        attention_out_ffn(x, wo, bo, held, wu, bu, wd, bd, norm_weight=nw, out=held)
        assert torch.equal(held, attention_out_ffn(x, wo, bo, res, wu, bu, wd, bd, norm_weight=nw))


@pytest.mark.parametrize("d,f,rows_over,valid", [(256, 64, 1, 1.0), (256, 1024, 33, 1.0), (256, 96, 1, 0.5), (256, 64, 33, 0.99), (128, 32, 1, 1.0),
                                                 (128, 512, 65, 0.8), (128, 32, 1, 0.4), (256, 1056, None, 1.0), (128, 2080, None, 0.7),
                                                 (128, 640, -40, 1.0), (128, 1024, 33, 1.0), (128, 1056, 1, 0.3), (128, 2080, 65, 0.6),
                                                 (256, 1056, 33, 1.0), (256, 1056, 1, 0.4), (256, 2080, 65, 0.7)])
def test_forms_of_the_few_token_feed_forward(device, test_hooks, d, f, rows_over, valid):
    """Rows just over the places that the chip has for one-tile workgroups (one per compute unit at D = 256, three at 128), with so many
    valid that workgroups take two tiles, the last of them a remainder, or one; hidden sizes over one slab of 1024 units (512 where two
    tiles or several workgroups share the LDS), with a remainder (rows_over None: 70 rows). Bound: as in the test above. Rows that are not listed stay as they are."""
    places = torch.cuda.get_device_properties(device).multi_processor_count * (1 if d == 256 else 3)
    m = 70 if rows_over is None else 32 * places + rows_over
    g = torch.Generator().manual_seed(m + f)
    x, res, nw = _bf16(g, m, d).to(device), _bf16(g, m, d).to(device), (1 + _bf16(g, d, scale=0.1)).to(device)
    wo, bo = _bf16(g, d, d, scale=d ** -0.5).to(device), _bf16(g, d, scale=0.1).to(device)
    wu, bu = _bf16(g, 2 * f, d, scale=d ** -0.5).to(device), _bf16(g, 2 * f, scale=0.1).to(device)
    wd, bd = _bf16(g, d, f, scale=f ** -0.5).to(device), _bf16(g, d, scale=0.1).to(device)
    listed = valid_rows(torch.tensor([int(m * valid)], dtype=torch.int32, device=device), m)
    with torch.no_grad():
        for fused in (True, False):
            def call():
                out = torch.full_like(res, 7.0)
                if fused:
                    return attention_out_ffn(x, wo, bo, res, wu, bu, wd, bd, norm_weight=nw, token_rows=listed, out=out)
                return swiglu_ffn(x, wu, bu, wd, bd, residual=res, norm_weight=nw, token_rows=listed, out=out)
            small, large = _both(test_hooks, call)
            _near_but_for_roundings(small, large)
            assert (small[int(m * valid):] == 7.0).all()
            small, large = _both(test_hooks, lambda: swiglu_ffn(x, wu, bu, wd, bd, token_rows=listed, out=torch.full_like(res, 7.0)))
            assert torch.equal(small, large)


@pytest.mark.parametrize("batch,sequence,d_model,heads,d_ff", [(1, 20, 256, 8, 1024), (1, 480, 256, 8, 1024), (5, 90, 256, 4, 64),
                                                               (16, 120, 256, 8, 512), (3, 61, 128, 4, 256),
                                                               (32, 120, 256, 8, 512), (20, 120, 128, 4, 256), (7, 61, 256, 8, 128),
                                                               (2, 300, 256, 8, 512), (7, 61, 256, 8, 384), (1, 20, 128, 4, 1024)])
def test_backbone_with_hidden_units_divided_over_workgroups(device, test_hooks, batch, sequence, d_model, heads, d_ff):
    """Batches small enough for 2 or 4 workgroups per token tile, against the persistent kernels and from run to run (the
    partial sums are added in a fixed order, whoever arrives last). Bound of the hidden state: roundings of the blocks'
    outputs flip by one bf16 step (2**-8 relative) and travel through the following blocks."""
    inputs = workloads.backbone_inputs(batch=batch, n_feature_tokens=8, n_sequence_tokens=sequence, d_model=d_model,
                                       num_heads=heads, d_ff=d_ff, n_blocks=2, min_sequence_len=1, seed=batch)
    model = PCVRBackbone(d_model=d_model, num_heads=heads, d_ff=d_ff, n_blocks=2)
    workloads.load_backbone_state(model, inputs)
    model = model.to(device=device, dtype=torch.bfloat16).eval()
    emb, lengths = 50 * inputs.emb.to(device), inputs.key_lengths.to(device)
    with torch.no_grad():
        (p, h), (p_large, h_large) = _both(test_hooks, lambda: model(emb, lengths, return_hidden=True))
        torch.testing.assert_close(p, p_large, rtol=0, atol=2e-3)
        torch.testing.assert_close(h.float(), h_large.float(), rtol=2 ** -5, atol=2 ** -4)
        for _ in range(3):
            again, h_again = model(emb, lengths, return_hidden=True)
            assert torch.equal(again, p) and torch.equal(h_again, h)


def test_calls_in_flight_on_several_streams_do_not_share_memory(device):
    """One module, two threads with a stream each: every call has the arrival counters, partial sums and activations of its own
    workspace, so that the results are those of the calls one after the other, bit for bit."""
    model = PCVRBackbone(d_model=256, num_heads=8, d_ff=1024, n_blocks=2).to(device=device, dtype=torch.bfloat16).eval()
    g = torch.Generator().manual_seed(9)
    requests = [(_bf16(g, 1 + i % 3, 100, 256).to(device),
                 torch.randint(1, 101, (1 + i % 3,), generator=g, dtype=torch.int32).to(device)) for i in range(24)]
    with torch.no_grad():
        want = [model(emb, lengths, return_hidden=True) for emb, lengths in requests]
    torch.cuda.synchronize()
    got: list = [None] * len(requests)

    def serve(first: int) -> None:
        with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream(device)):
            for i in range(first, len(requests), 2):
                got[i] = model(*requests[i], return_hidden=True)
            torch.cuda.current_stream(device).synchronize()

    threads = [threading.Thread(target=serve, args=(first,)) for first in range(2)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    for (p, hidden), (want_p, want_hidden) in zip(got, want):
        assert torch.equal(p, want_p) and torch.equal(hidden, want_hidden)
    assert len(model._workspaces) == 3 and len(copy.deepcopy(model)._workspaces) == 0
    # two calls on one stream, the first of which has not run yet, and one on another stream in between
    busy, other = torch.cuda.Stream(device), torch.cuda.Stream(device)
    torch.cuda.synchronize()
    with torch.no_grad():
        with torch.cuda.stream(busy):
            torch.cuda._sleep(20_000_000)
            first = model(*requests[0])
        with torch.cuda.stream(other):
            second = model(*requests[1])
        with torch.cuda.stream(busy):
            third = model(*requests[2])
    torch.cuda.synchronize()
    assert all(torch.equal(p, want[i][0]) for i, p in enumerate((first, second, third)))


def test_a_captured_call_has_its_own_memory(device):
    """A forward recorded into a graph, replayed between eager calls of the same module on other inputs and streams: every result is
    that of the eager call on the same input."""
    model = PCVRBackbone(d_model=256, num_heads=8, d_ff=1024, n_blocks=2).to(device=device, dtype=torch.bfloat16).eval()
    g = torch.Generator().manual_seed(10)
    lengths = torch.tensor([100, 37], dtype=torch.int32, device=device)
    inputs = [_bf16(g, 2, 100, 256).to(device) for _ in range(4)]
    other = torch.cuda.Stream(device)
    with torch.no_grad():
        want = [model(emb, lengths) for emb in inputs]
        static = inputs[0].clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            p = model(static, lengths)
        for i, emb in enumerate(inputs):
            static.copy_(emb)
            torch.cuda.synchronize()
            with torch.cuda.stream(other):
                eager = model(inputs[i - 1], lengths)
            graph.replay()
            again = model(inputs[i - 2], lengths)
            torch.cuda.synchronize()
            assert torch.equal(p, want[i]) and torch.equal(eager, want[i - 1]) and torch.equal(again, want[i - 2])
