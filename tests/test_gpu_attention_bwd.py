"""GPU parity: attention training forward (log-sum-exp) and backward (through the C ABI) against torch autograd of the
CPU oracle's closed form evaluated in float64."""

from __future__ import annotations

import pytest
import torch

from oracle import reference as oracle
from taac_2026_amd.api import flash_attention, scaled_dot_product_attention

pytestmark = pytest.mark.gpu

# Gradient tolerance of the reference's GPU tests for 16-bit attention (tests/gpu/infrastructure/accelerators/
# test_tilelang_ops_cuda.py:98-141): 3e-2.
TOL = dict(rtol=3e-2, atol=3e-2)


def _reference(q, k, v, lengths, grad_out, *, causal, zero_pad):
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    out = oracle.attention(qr, kr, vr, lengths, is_causal=causal, zero_padded_queries=zero_pad)
    out.backward(grad_out.double())
    return out.detach(), qr.grad, kr.grad, vr.grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,dim", [(50, 32), (130, 64), (300, 32), (64, 16), (257, 64), (33, 8), (150, 48)])
@pytest.mark.parametrize("causal,zero_pad", [(False, False), (False, True), (True, False)])
def test_backward_matches_autograd_of_the_oracle(device, dtype, tokens, dim, causal, zero_pad):
    batch, heads = 4, 2
    g = torch.Generator().manual_seed(tokens * 7 + dim)
    q, k, v = (torch.randn(batch, heads, tokens, dim, generator=g).to(dtype) for _ in range(3))
    grad_out = torch.randn(batch, heads, tokens, dim, generator=g).to(dtype)
    lengths = torch.tensor([tokens, 1, max(1, tokens // 2), max(1, tokens - 3)], dtype=torch.int32)
    ref_out, ref_dq, ref_dk, ref_dv = _reference(q, k, v, lengths, grad_out, causal=causal, zero_pad=zero_pad)
    qd, kd, vd = (t.to(device).requires_grad_(True) for t in (q, k, v))
    out = flash_attention(qd, kd, vd, key_lengths=lengths.to(device), is_causal=causal, zero_padded_queries=zero_pad)
    out.backward(grad_out.to(device))
    torch.testing.assert_close(out.detach().cpu().double(), ref_out, rtol=2e-2, atol=2e-2)
    for got, ref, name in ((qd.grad, ref_dq, "dq"), (kd.grad, ref_dk, "dk"), (vd.grad, ref_dv, "dv")):
        assert got.dtype == dtype and got.shape == ref.shape
        torch.testing.assert_close(got.cpu().double(), ref, msg=lambda m, n=name: f"{n}: {m}", **TOL)
    # keys in the padding receive exactly zero gradient
    for b in range(batch):
        if lengths[b] < tokens:
            assert kd.grad[b, :, int(lengths[b]):].abs().max().item() == 0.0
            assert vd.grad[b, :, int(lengths[b]):].abs().max().item() == 0.0
            if zero_pad:
                assert qd.grad[b, :, int(lengths[b]):].abs().max().item() == 0.0


def test_backward_is_reproducible_and_reads_the_projection_layout(device):
    """(B, T, D) projections that are chunk views of one packed tensor, as the model packages produce them; two runs
    give bit-identical gradients (one writer per element, fixed summation order)."""
    batch, tokens, heads, dim = 3, 200, 4, 32
    g = torch.Generator().manual_seed(0)
    packed = torch.randn(batch, tokens, 3 * heads * dim, generator=g).to(torch.bfloat16)
    lengths = torch.tensor([200, 77, 130], dtype=torch.int32)
    grad_out = torch.randn(batch, tokens, heads * dim, generator=g).to(torch.bfloat16)
    grads = []
    for _ in range(2):
        pd = packed.to(device).requires_grad_(True)
        q, k, v = pd.chunk(3, dim=-1)
        out = scaled_dot_product_attention(q, k, v, num_heads=heads, attn_mask=None, dropout_p=0.0, training=True,
                                           key_lengths=lengths.to(device), zero_padded_queries=True)
        out.backward(grad_out.to(device))
        grads.append(pd.grad.clone())
    assert torch.equal(grads[0], grads[1])
    pr = packed.double().requires_grad_(True)
    q, k, v = pr.chunk(3, dim=-1)
    ref = oracle.scaled_dot_product_attention(q, k, v, num_heads=heads, key_lengths=lengths, zero_padded_queries=True)
    ref.backward(grad_out.double())
    torch.testing.assert_close(grads[0].cpu().double(), pr.grad, **TOL)


@pytest.mark.parametrize("dim,causal", [(32, False), (64, False), (64, True)])
def test_direct_transfer_backward_equals_register_staged_backward(device, dim, causal):
    """Full head dims stream their chunks from global memory straight into LDS, where rows beyond the valid length repeat
    the last valid row instead of zeros; their products are cancelled by zero probabilities, so both backward routes give
    the same bits from the same saved forward (taac_flash_attn_bwd through the C ABI with and without
    TAAC_ATTN_REGISTER_STAGING; the two forwards differ by roundings, see test_gpu_attention.py, so one forward feeds
    both)."""
    from taac_2026_amd import _native

    batch, heads, tokens = 5, 2, 333
    g = torch.Generator().manual_seed(dim + causal)
    q, k, v, grad_out = (torch.randn(batch, heads, tokens, dim, generator=g).to(torch.bfloat16).to(device) for _ in range(4))
    lengths = torch.tensor([333, 1, 64, 65, 200], dtype=torch.int32, device=device)
    library = _native.load_library()
    stream = _native.current_stream(q.device)
    out = torch.empty_like(q)
    lse = torch.empty(batch, heads, tokens, dtype=torch.float32, device=device)
    strides = lambda *ts: [_native.Int64x4(*t.stride()) for t in ts]  # noqa: E731
    flags = _native.ATTN_CAUSAL if causal else 0
    zero_pad = int(not causal)
    _native.check(library.taac_flash_attn_train_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), lengths.data_ptr(), out.data_ptr(), lse.data_ptr(), batch, heads, tokens,
        tokens, dim, *strides(q, k, v, out), flags, zero_pad, _native.dtype_code(q.dtype), stream), "train_fwd")
    grads = {}
    for name, route in (("direct", 0), ("registers", _native.ATTN_REGISTER_STAGING)):
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        delta = torch.empty_like(lse)
        _native.check(library.taac_flash_attn_bwd(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), grad_out.data_ptr(), lse.data_ptr(),
            lengths.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), delta.data_ptr(), batch, heads, tokens, tokens,
            dim, *strides(q, k, v, out, grad_out, dq, dk, dv), flags | route, zero_pad, _native.dtype_code(q.dtype), stream),
            "bwd")
        grads[name] = (dq, dk, dv)
    for direct, staged in zip(grads["direct"], grads["registers"]):
        assert torch.isfinite(direct.float()).all()
        assert torch.equal(direct, staged)
    # and the module-level route switch reaches both kernels: gradients of the two routes agree to rounding
    for staging in ("direct", "registers"):
        qd, kd, vd = (t.clone().requires_grad_(True) for t in (q, k, v))
        flash_attention(qd, kd, vd, key_lengths=lengths, is_causal=causal, zero_padded_queries=not causal,
                        kv_staging=staging).backward(grad_out)
        for got, want in zip((qd.grad, kd.grad, vd.grad), grads["direct"]):
            # (a step or two of bf16 at the largest gradients: the two forwards round differently)
            torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -5, atol=2 ** -6 * want.float().abs().max().item())


def test_backward_envelope(device):
    q = torch.randn(1, 1, 16, 128, device=device, dtype=torch.bfloat16, requires_grad=True)
    with pytest.raises(RuntimeError, match="head_dim"):
        flash_attention(q, q, q).sum().backward()
    q32 = torch.randn(1, 1, 16, 32, device=device, requires_grad=True)
    with pytest.raises(RuntimeError, match="backward covers"):
        flash_attention(q32, q32, q32)


@pytest.mark.parametrize("dtype,dim,causal,tokens", [(torch.float16, 16, False, 32), (torch.bfloat16, 32, False, 150),
                                                     (torch.bfloat16, 64, True, 200), (torch.float16, 64, False, 77)])
def test_training_dropout_with_a_fixed_keep_mask(device, dtype, dim, causal, tokens):
    """Dropout on the attention probabilities with the caller's uint8 keep mask, forward and backward, against float64
    autograd of the oracle under the same mask - the check the reference runs on its TileLang kernels
    (tests/gpu/infrastructure/accelerators/test_tilelang_ops_cuda.py:103-141: output 2e-2, gradients 3e-2), here also with
    ragged key lengths, a causal triangle and a key count that is no multiple of four (unaligned mask rows)."""
    batch, heads, dropout_p = 3, 4, 0.125
    g = torch.Generator().manual_seed(tokens + dim)
    q, k, v, grad_out = (torch.randn(batch, heads, tokens, dim, generator=g).to(dtype) for _ in range(4))
    lengths = torch.tensor([tokens, max(1, tokens // 3), tokens - 5], dtype=torch.int32)
    mask = (torch.rand(batch, heads, tokens, tokens, generator=g) >= dropout_p).to(torch.uint8)
    qd, kd, vd = (t.to(device).requires_grad_(True) for t in (q, k, v))
    out = flash_attention(qd, kd, vd, key_lengths=lengths.to(device), is_causal=causal, zero_padded_queries=not causal,
                          dropout_p=dropout_p, training=True, dropout_mask=mask.to(device))
    out.backward(grad_out.to(device))
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    want = oracle.attention_dropout(qr, kr, vr, lengths, mask, dropout_p, is_causal=causal, zero_padded_queries=not causal)
    want.backward(grad_out.double())
    torch.testing.assert_close(out.detach().cpu().double(), want.detach(), rtol=2e-2, atol=2e-2)
    for got, ref in ((qd.grad, qr.grad), (kd.grad, kr.grad), (vd.grad, vr.grad)):
        torch.testing.assert_close(got.cpu().double(), ref, rtol=3e-2, atol=3e-2)
    # the mask matters (a run without it differs) and an all-ones mask at p -> 0 is the plain training path
    plain = flash_attention(qd.detach(), kd.detach(), vd.detach(), key_lengths=lengths.to(device), is_causal=causal,
                            zero_padded_queries=not causal)
    assert (plain.float() - out.detach().float()).abs().max().item() > 5e-2
    ones = torch.ones_like(mask).to(device)
    q1 = qd.detach().clone().requires_grad_(True)
    same = flash_attention(q1, kd.detach(), vd.detach(), key_lengths=lengths.to(device), is_causal=causal,
                           zero_padded_queries=not causal, dropout_p=1e-9, training=True, dropout_mask=ones)
    torch.testing.assert_close(same.detach().float(), plain.float(), rtol=2e-2, atol=2e-2)


def test_dropout_draws_its_own_mask_and_rejects_what_it_does_not_cover(device):
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(2, 2, 64, 32, generator=g).to(torch.bfloat16).to(device) for _ in range(3))
    torch.manual_seed(0)
    a = flash_attention(q, k, v, dropout_p=0.5, training=True)
    torch.manual_seed(0)
    b = flash_attention(q, k, v, dropout_p=0.5, training=True)
    c = flash_attention(q, k, v, dropout_p=0.5, training=True)
    assert torch.equal(a, b) and not torch.equal(a, c)
    with pytest.raises(RuntimeError, match="only supports dropout during training"):
        flash_attention(q, k, v, dropout_p=0.5, training=False)
    with pytest.raises(ValueError, match="dropout_mask must be uint8"):
        flash_attention(q, k, v, dropout_p=0.5, training=True, dropout_mask=torch.ones(2, 2, 64, 63, dtype=torch.uint8, device=device))


def _native_backward(q, k, v, out, grad_out, lse, lengths, causal, zero_pad, *, staged=False, words=None, visible=None, key_valid=None):
    """dq, dk, dv through the C ABI (poisoned with NaN before the call); ``staged``: the register-staged kernels; ``words``:
    mask bits with optional validity words; ``visible``: the same mask as bytes."""
    from taac_2026_amd import _native

    library = _native.load_library()
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    delta = torch.empty_like(lse)
    (batch, heads, rows, dim), keys = q.shape, k.shape[2]
    strides = [_native.Int64x4(*t.stride()) for t in (q, k, v, out, grad_out, *grads)]
    head = [t.data_ptr() for t in (q, k, v, out, grad_out, lse)] + [_native.ptr(lengths)]
    outs = [t.data_ptr() for t in (*grads, delta)]
    tail = [_native.dtype_code(q.dtype), _native.current_stream(q.device)]
    if words is not None:
        status = library.taac_flash_attn_bits_bwd(*head, words.data_ptr(), words.stride(0), _native.ptr(key_valid), None, 1.0, *outs,
                                                  batch, heads, rows, keys, dim, *strides, int(zero_pad), *tail)
    elif visible is not None:
        status = library.taac_flash_attn_mask_bwd(*head, visible.data_ptr(), rows * keys, 0, None, *outs, batch, heads, rows, keys, dim,
                                                  *strides, int(zero_pad), *tail)
    else:
        status = library.taac_flash_attn_bwd(*head, *outs, batch, heads, rows, keys, dim, *strides, int(causal) | (2 if staged else 0),
                                             int(zero_pad), *tail)
    _native.check(status, "backward")
    return grads


def _log_sum_exp(q, k, visible):
    """out-independent statistics in float64: log-sum-exp of the visible scaled scores and the probabilities."""
    scores = (q.double() @ k.double().transpose(-1, -2)) / q.shape[-1] ** 0.5
    scores = scores.masked_fill(~visible, float("-inf"))
    return torch.logsumexp(scores, dim=-1), torch.nan_to_num(torch.softmax(scores, dim=-1), nan=0.0)


def _exact_gradients(q, k, v, out, grad_out, probabilities):
    """The closed form in float64, with D from the saved output as the kernels take it, and the same sums over the terms'
    absolute values."""
    def gradients(q, k, v, out, g, sign):
        d = (g * out).sum(-1, keepdim=True)
        ds = probabilities * (g @ v.transpose(-1, -2) - sign * d) * q.shape[-1] ** -0.5
        return ds @ k, ds.transpose(-1, -2) @ q, probabilities.transpose(-1, -2) @ g

    tensors = [t.double() for t in (q, k, v, out, grad_out)]
    return list(zip(gradients(*tensors, 1.0), gradients(*(t.abs() for t in tensors), -1.0)))


def _check_gradients(got, other, exact, dtype):
    # a term's probability or dS is rounded to 16 bits and so is the sum: 2^-8 of it (bf16: 8 bits) or 2^-11 (fp16: 11 bits) each
    unit = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    for name, a, s, (e, size) in zip(("dq", "dk", "dv"), got, other, exact):
        assert not torch.isnan(a).any(), name
        assert (a[size == 0] == 0).all(), name  # padding and samples without a key
        error, error_other = (a.double() - e), (s.double() - e)
        assert (error.abs() <= unit * size + 1e-6).all(), name
        assert error.norm() <= 1.05 * error_other.norm() + 1e-6 * size.norm(), (name, error.norm(), error_other.norm())


# One workgroup per (sample, head): one to four key tiles per wavefront, their last ones partly filled, sizes and pairs on both sides of
# what such a workgroup holds and of what the dispatch asks for.
@pytest.mark.parametrize("rows,keys,dim,batch,heads", [
    (1, 1, 32, 3, 2), (31, 31, 64, 3, 2), (33, 33, 32, 3, 2), (128, 128, 64, 5, 2), (100, 37, 32, 3, 2), (20, 128, 64, 3, 2),
    (129, 129, 32, 64, 8), (256, 256, 32, 64, 8), (257, 257, 32, 128, 8), (490, 490, 32, 128, 8), (512, 512, 32, 128, 8),
    (129, 129, 64, 128, 4), (256, 256, 64, 128, 4), (257, 257, 64, 128, 4), (257, 257, 32, 448, 8), (384, 384, 32, 448, 8),
    (385, 385, 32, 128, 8), (512, 512, 32, 192, 8)])
@pytest.mark.parametrize("dtype,causal,zero_pad", [(torch.bfloat16, False, True), (torch.float16, True, False), (torch.bfloat16, True, True)])
def test_backward_with_all_keys_in_one_workgroup(device, rows, keys, dim, batch, heads, dtype, causal, zero_pad):
    if rows != keys and zero_pad:
        pytest.skip("zero_padded_queries needs as many queries as keys")
    g = torch.Generator(device=device).manual_seed(rows * 3 + dim)
    # the projection layout: heads next to each other in a row
    draw = lambda n: torch.randn(batch, n, heads, dim, generator=g, device=device).to(dtype).transpose(1, 2)  # noqa: E731
    q, k, v, grad_out = draw(rows), draw(keys), draw(keys), draw(rows)
    lengths = torch.randint(0, keys + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    lengths[0], lengths[1], lengths[2] = keys, 0, max(1, keys - 1)
    index = torch.arange(keys, device=device)
    visible = (index < lengths[:, None])[:, None, None, :].expand(batch, 1, rows, keys)
    if causal:
        visible = visible & (index <= torch.arange(rows, device=device)[:, None])
    if zero_pad:
        visible = visible & (torch.arange(rows, device=device) < lengths[:, None])[:, None, :, None]
    lse, p = _log_sum_exp(q, k, visible)
    out = (p @ v.double()).to(dtype)
    exact = _exact_gradients(q, k, v, out, grad_out, p)
    args = (q, k, v, out, grad_out, lse.float().contiguous(), lengths, causal, zero_pad)
    got, staged = _native_backward(*args), _native_backward(*args, staged=True)
    _check_gradients(got, staged, exact, dtype)
    assert all(torch.equal(a, b) for a, b in zip(got, _native_backward(*args)))


@pytest.mark.parametrize("rows,dim,batch,heads,valid", [(40, 32, 3, 2, True), (128, 64, 3, 2, False), (250, 32, 64, 8, True),
                                                        (300, 32, 128, 8, False), (129, 64, 128, 4, False), (255, 64, 128, 4, True)])
def test_mask_bits_backward_with_all_keys_in_one_workgroup(device, rows, dim, batch, heads, valid):
    g = torch.Generator(device=device).manual_seed(rows + dim)
    draw = lambda: torch.randn(batch, heads, rows, dim, generator=g, device=device).to(torch.bfloat16)  # noqa: E731
    q, k, v, grad_out = draw(), draw(), draw(), draw()
    lengths = torch.randint(1, rows + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    words_per_row = (rows + 31) // 32
    bits = torch.rand(batch, rows, words_per_row * 32, generator=g, device=device) < 0.4
    weights = (1 << torch.arange(32, device=device, dtype=torch.int64))
    pack = lambda t: (t.reshape(*t.shape[:-1], words_per_row, 32) * weights).sum(-1).to(torch.int32).contiguous()  # noqa: E731
    words = pack(bits)
    key_valid = torch.rand(batch, words_per_row * 32, generator=g, device=device) < 0.8
    index = torch.arange(rows, device=device)
    visible = bits[:, :, :rows] & (index < lengths[:, None])[:, None, :]
    if valid:
        visible = visible & key_valid[:, None, :rows]
    alive = visible & (index < lengths[:, None])[:, :, None]
    lse, p = _log_sum_exp(q, k, alive[:, None])
    out = (p @ v.double()).to(torch.bfloat16)
    exact = _exact_gradients(q, k, v, out, grad_out, p)
    args = (q, k, v, out, grad_out, lse.float().contiguous(), lengths, False, True)
    got = _native_backward(*args, words=words, key_valid=pack(key_valid) if valid else None)
    dense = _native_backward(*args, visible=visible.to(torch.uint8).contiguous())
    _check_gradients(got, dense, exact, torch.bfloat16)


@pytest.mark.parametrize("rows,dim,batch,heads", [(128, 32, 8, 4), (200, 32, 64, 8), (400, 32, 128, 8), (250, 64, 128, 4), (77, 64, 8, 4)])
def test_one_workgroup_rounds_as_the_two_kernels_do(device, rows, dim, batch, heads):
    """Every sum has the order and every value the rounding of the two kernels: the same bits, so that a gradient does not depend on how
    many samples a batch has."""
    g = torch.Generator(device=device).manual_seed(rows)
    q, k, v, grad_out = (torch.randn(batch, heads, rows, dim, generator=g, device=device).to(torch.bfloat16) for _ in range(4))
    lengths = torch.randint(1, rows + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    index = torch.arange(rows, device=device)
    inside = index < lengths[:, None]
    lse, p = _log_sum_exp(q, k, (inside[:, None, :] & inside[:, :, None])[:, None])
    args = (q, k, v, (p @ v.double()).to(torch.bfloat16), grad_out, lse.float().contiguous(), lengths, False, True)
    for name, a, b in zip(("dq", "dk", "dv"), _native_backward(*args), _native_backward(*args, staged=True)):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("rows,dim,batch,heads", [(512, 32, 192, 8), (256, 32, 64, 8), (256, 64, 128, 4), (128, 64, 8, 4)])
@pytest.mark.parametrize("causal", [False, True])
def test_one_workgroup_with_every_number_of_key_tiles(device, rows, dim, batch, heads, causal):
    """Lengths over the whole range, on both sides of every key tile's edge: groups of tiles that are whole, half or not there."""
    g = torch.Generator(device=device).manual_seed(rows + causal)
    q, k, v, grad_out = (torch.randn(batch, heads, rows, dim, generator=g, device=device).to(torch.bfloat16) for _ in range(4))
    edges = torch.arange(32, rows + 1, 32, device=device)
    edges = torch.cat([edges, edges - 31, (edges + 1).clamp_max(rows), edges - 1])
    lengths = edges[torch.arange(batch, device=device) % edges.numel()].to(torch.int32)
    index = torch.arange(rows, device=device)
    inside = index < lengths[:, None]
    seen = inside[:, None, :] & inside[:, :, None] & ((index[None, :] <= index[:, None]) | (not causal))
    lse, p = _log_sum_exp(q, k, seen[:, None])
    args = (q, k, v, (p @ v.double()).to(torch.bfloat16), grad_out, lse.float().contiguous(), lengths, causal, True)
    for name, a, b in zip(("dq", "dk", "dv"), _native_backward(*args), _native_backward(*args, staged=True)):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype,rows,dim,batch,heads,part", [
    (torch.bfloat16, 129, 32, 64, 8, 63), (torch.float16, 256, 32, 64, 8, 21), (torch.bfloat16, 250, 64, 130, 4, 65),
    (torch.float16, 160, 64, 130, 4, 65), (torch.bfloat16, 64, 32, 388, 4, 194), (torch.bfloat16, 97, 32, 260, 8, 52)])
@pytest.mark.parametrize("valid", [False, True])
def test_mask_bits_backward_of_a_batch_and_of_its_parts(device, dtype, rows, dim, batch, heads, part, valid):
    """On one side of the dispatch's lines a batch, on the other its parts: a sample's gradients have the same bits."""
    g = torch.Generator(device=device).manual_seed(rows)
    q, k, v, grad_out = (torch.randn(batch, heads, rows, dim, generator=g, device=device).to(dtype) for _ in range(4))
    lengths = torch.randint(1, rows + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    n_words = (rows + 31) // 32
    words, key_valid = (torch.randint(-2 ** 31, 2 ** 31, (batch, n, n_words), generator=g, device=device).to(torch.int32) for n in (rows, 1))
    on = lambda t: ((t.unsqueeze(-1) >> torch.arange(32, device=device)) & 1).flatten(-2)[..., :rows] != 0  # noqa: E731
    inside = torch.arange(rows, device=device) < lengths[:, None]
    visible = on(words) & inside[:, None, :] & inside[:, :, None]
    if valid:
        visible = visible & on(key_valid)
    lse, p = _log_sum_exp(q, k, visible[:, None])
    out, lse = (p @ v.double()).to(dtype), lse.float().contiguous()

    def gradients(s):
        return _native_backward(q[s], k[s], v[s], out[s], grad_out[s], lse[s], lengths[s], False, True, words=words[s],
                                key_valid=key_valid[s] if valid else None)

    whole = gradients(slice(0, batch))
    parts = [gradients(slice(i, i + part)) for i in range(0, batch, part)]
    for name, a, *pieces in zip(("dq", "dk", "dv"), whole, *parts):
        assert torch.equal(a, torch.cat(pieces)), name


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("rows,dim,batch,heads,bits", [(40, 32, 4, 2, False), (100, 64, 4, 2, True), (250, 32, 64, 8, True),
                                                       (400, 32, 128, 8, False), (200, 64, 128, 4, False), (400, 32, 4, 2, True)])
def test_padding_keys_receive_zeros_whatever_the_gradient(device, rows, dim, batch, heads, bits, value):
    """A gradient that is not finite reaches the keys its query sees, not the padding in the same tile; other samples are untouched."""
    g = torch.Generator(device=device).manual_seed(rows)
    q, k, v, grad_out = (torch.randn(batch, heads, rows, dim, generator=g, device=device).to(torch.bfloat16) for _ in range(4))
    lengths = torch.randint(rows // 4, rows + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    lengths[0] = rows - 5
    grad_out[0, :, 3, 1] = value
    index = torch.arange(rows, device=device)
    inside = index < lengths[:, None]
    lse, p = _log_sum_exp(q, k, (inside[:, None, :] & inside[:, :, None])[:, None])
    words = torch.full((batch, rows, (rows + 31) // 32), -1, dtype=torch.int32, device=device) if bits else None
    got = _native_backward(q, k, v, (p @ v.double()).to(torch.bfloat16), grad_out, lse.float().contiguous(), lengths, False, True, words=words)
    for name, t in zip(("dq", "dk", "dv"), got):
        assert (t.transpose(1, 2)[~inside] == 0).all(), name
        assert torch.isfinite(t[1:]).all(), name
    assert not torch.isfinite(got[2][0, :, :rows - 5]).all()
