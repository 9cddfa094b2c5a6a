"""GPU parity: the fused readout (token norm -> cls | candidate | masked mean -> RMSNorm -> classifier, through the C
ABI) against the CPU oracle."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from oracle import reference as oracle
from taac_2026_amd.api import CandidateClsPooler, CandidateReadoutHead, candidate_readout

pytestmark = pytest.mark.gpu

TOL = dict(rtol=2e-2, atol=2e-2)  # the benchmark configuration's bf16 tolerance


def _draw(batch, tokens, d, hidden, actions, seed):
    g = torch.Generator().manual_seed(seed)
    bf = lambda t: t.to(torch.bfloat16)
    x = bf(torch.randn(batch, tokens, d, generator=g))
    wt, wp = bf(1 + 0.1 * torch.randn(d, generator=g)), bf(1 + 0.1 * torch.randn(3 * d, generator=g))
    w1, b1 = bf(torch.randn(hidden, 3 * d, generator=g) * (3 * d) ** -0.5), bf(0.1 * torch.randn(hidden, generator=g))
    w2, b2 = bf(torch.randn(actions, hidden, generator=g) * hidden ** -0.5), bf(0.1 * torch.randn(actions, generator=g))
    pad = torch.rand(batch, tokens, generator=g) < 0.3
    pad[0] = True          # a sample of padding only
    if batch > 1:
        pad[1] = False     # a sample without padding
    return x, wt, wp, w1, b1, w2, b2, pad


@pytest.mark.parametrize("batch,tokens,d,hidden,actions", [(5, 37, 256, 256, 1), (3, 100, 128, 64, 3), (2, 9, 64, 40, 2),
                                                           (4, 70, 1024, 1024, 1), (3, 33, 320, 96, 4), (1, 1, 8, 8, 1)])
@pytest.mark.parametrize("candidate", [True, False])
def test_matches_oracle(device, batch, tokens, d, hidden, actions, candidate):
    x, wt, wp, w1, b1, w2, b2, pad = _draw(batch, tokens, d, hidden, actions, seed=tokens + d)
    cls_index, cand_index = tokens // 3, (tokens - 1 if candidate else None)
    want_emb, want_logits = oracle.candidate_readout(x, pad, cls_index=cls_index, candidate_index=cand_index,
                                                     token_norm_weight=wt, pool_norm_weight=wp, eps=1e-6,
                                                     classifier=(w1, b1, w2, b2))
    to = lambda t: t.to(device)
    with torch.no_grad():
        logits, emb = candidate_readout(to(x), cls_index=cls_index, candidate_index=cand_index, padding_mask=to(pad),
                                        token_norm_weight=to(wt), pool_norm_weight=to(wp), fc1_weight=to(w1),
                                        fc1_bias=to(b1), fc2_weight=to(w2), fc2_bias=to(b2), return_embedding=True)
        probs = candidate_readout(to(x), cls_index=cls_index, candidate_index=cand_index, padding_mask=to(pad),
                                  token_norm_weight=to(wt), pool_norm_weight=to(wp), fc1_weight=to(w1), fc1_bias=to(b1),
                                  fc2_weight=to(w2), fc2_bias=to(b2), sigmoid=True)
    assert emb.shape == (batch, 3 * d) and emb.dtype == torch.bfloat16
    assert logits.shape == (batch, actions) and logits.dtype == torch.float32
    torch.testing.assert_close(emb.cpu().float(), want_emb, **TOL)
    torch.testing.assert_close(logits.cpu(), want_logits, **TOL)
    torch.testing.assert_close(probs.cpu(), torch.sigmoid(want_logits), **TOL)
    if not candidate:
        assert emb[:, d:2 * d].abs().max().item() == 0.0
    # the reference's own bf16 evaluation of the same modules stays within twice the tolerance
    ref_emb, ref_logits = oracle.candidate_readout(x, pad, cls_index=cls_index, candidate_index=cand_index,
                                                   token_norm_weight=wt, pool_norm_weight=wp, eps=1e-6,
                                                   classifier=(w1, b1, w2, b2), fp32=False)
    torch.testing.assert_close(emb.cpu().float(), ref_emb.float(), rtol=4e-2, atol=4e-2)
    torch.testing.assert_close(logits.cpu(), ref_logits.float(), rtol=6e-2, atol=6e-2)


def test_valid_token_forms_agree_and_optional_parts(device):
    """key_lengths, the matching prefix padding mask and (for full lengths) no mask at all give identical results;
    without norms and classifier the three thirds are the picked tokens and the plain masked mean."""
    x, wt, wp, w1, b1, w2, b2, _ = _draw(6, 50, 256, 256, 1, seed=3)
    lengths = torch.tensor([50, 0, 1, 17, 32, 49], dtype=torch.int32)
    pad = torch.arange(50)[None, :] >= lengths[:, None]
    to = lambda t: t.to(device)
    kw = dict(cls_index=0, candidate_index=7, token_norm_weight=to(wt), pool_norm_weight=to(wp), fc1_weight=to(w1),
              fc1_bias=to(b1), fc2_weight=to(w2), fc2_bias=to(b2), return_embedding=True)
    with torch.no_grad():
        by_len = candidate_readout(to(x), key_lengths=to(lengths), **kw)
        by_mask = candidate_readout(to(x), padding_mask=to(pad), **kw)
        full_a = candidate_readout(to(x), key_lengths=torch.full((6,), 50, dtype=torch.int32, device=device), **kw)
        full_b = candidate_readout(to(x), **kw)
        bare = candidate_readout(to(x), cls_index=4, candidate_index=9, padding_mask=to(pad))
    for a, b in ((by_len, by_mask), (full_a, full_b)):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    want, _ = oracle.candidate_readout(x, pad, cls_index=4, candidate_index=9, token_norm_weight=None, pool_norm_weight=None)
    assert torch.equal(bare[:, :256].cpu(), x[:, 4]) and torch.equal(bare[:, 256:512].cpu(), x[:, 9])
    torch.testing.assert_close(bare.cpu().float(), want, rtol=1e-2, atol=1e-3)
    assert bare[1, 512:].abs().max().item() == 0.0  # a sample of padding only


def test_modules_mirror_the_reference_readout(device):
    """CandidateClsPooler takes the reference's batch object; CandidateReadoutHead = final_norm + pooler + classifier,
    forward -> logits, predict -> (logits, embedding)."""
    torch.manual_seed(0)
    d, tokens, batch = 128, 40, 4
    head = CandidateReadoutHead(d, action_num=2, use_candidate_readout=True)
    with torch.no_grad():
        head.final_norm.weight.add_(0.1 * torch.randn(d))
        head.pooler.norm.weight.add_(0.1 * torch.randn(3 * d))
        head.classifier[0].bias.add_(0.1 * torch.randn(d))
    head = head.to(device=device, dtype=torch.bfloat16).eval()
    x = torch.randn(batch, tokens, d).to(torch.bfloat16)
    pad = torch.rand(batch, tokens) < 0.4
    info = SimpleNamespace(cls_index=0, candidate_index=5, padding_mask=pad.to(device))
    with torch.no_grad():
        logits = head(x.to(device), info)
        logits2, emb = head.predict(x.to(device), info)
        pooled = head.pooler(x.to(device), info, token_norm=head.final_norm)
        pooler_only = CandidateClsPooler(d, use_candidate_readout=False).to(device=device, dtype=torch.bfloat16)(x.to(device), info)
    cpu = lambda t: t.detach().cpu()
    fc1, fc2 = head.classifier[0], head.classifier[3]
    want_emb, want_logits = oracle.candidate_readout(
        x, pad, cls_index=0, candidate_index=5, token_norm_weight=cpu(head.final_norm.weight),
        pool_norm_weight=cpu(head.pooler.norm.weight), eps=head.pooler.norm.eps,
        classifier=(cpu(fc1.weight), cpu(fc1.bias), cpu(fc2.weight), cpu(fc2.bias)))
    assert torch.equal(logits, logits2) and torch.equal(emb, pooled)
    torch.testing.assert_close(cpu(logits), want_logits, **TOL)
    torch.testing.assert_close(cpu(emb).float(), want_emb, **TOL)
    want_plain, _ = oracle.candidate_readout(x, pad, cls_index=0, candidate_index=None, token_norm_weight=None,
                                             pool_norm_weight=torch.ones(3 * d, dtype=torch.bfloat16))
    torch.testing.assert_close(cpu(pooler_only).float(), want_plain, **TOL)


@pytest.mark.parametrize("candidate,use_lengths", [(True, False), (False, True)])
def test_readout_takes_a_gradient(device, candidate, use_lengths):
    """Under autograd the readout runs its differentiable route: outputs equal to the one-kernel route, gradients of the
    tokens and of every weight against float64 autograd of the oracle's expression."""
    batch, tokens, d, hidden, actions = 6, 50, 256, 128, 2
    x, wt, wp, w1, b1, w2, b2, pad = _draw(batch, tokens, d, hidden, actions, seed=77)
    lengths = torch.tensor([50, 0, 13, 1, 30, 44], dtype=torch.int32)
    if use_lengths:
        pad = torch.arange(tokens)[None, :] >= lengths[:, None]
    cls_index, cand_index = 2, (tokens - 1 if candidate else None)
    dev = [t.to(device).requires_grad_(True) for t in (x, wt, wp, w1, b1, w2, b2)]
    where = dict(key_lengths=lengths.to(device)) if use_lengths else dict(padding_mask=pad.to(device))
    logits, emb = candidate_readout(dev[0], cls_index=cls_index, candidate_index=cand_index, token_norm_weight=dev[1],
                                    pool_norm_weight=dev[2], fc1_weight=dev[3], fc1_bias=dev[4], fc2_weight=dev[5],
                                    fc2_bias=dev[6], return_embedding=True, **where)
    g = torch.Generator().manual_seed(5)
    grad_logits, grad_emb = torch.randn(batch, actions, generator=g), torch.randn(batch, 3 * d, generator=g).to(torch.bfloat16)
    torch.autograd.backward([logits, emb], [grad_logits.to(device), grad_emb.to(device)])
    ref = [t.double().requires_grad_(True) for t in (x, wt, wp, w1, b1, w2, b2)]
    want_emb, want_logits = oracle.candidate_readout(ref[0], pad, cls_index=cls_index, candidate_index=cand_index,
                                                     token_norm_weight=ref[1], pool_norm_weight=ref[2], eps=1e-6,
                                                     classifier=tuple(ref[3:]), fp32=False)
    torch.autograd.backward([want_logits, want_emb], [grad_logits.double(), grad_emb.double()])
    with torch.no_grad():
        fused_logits, fused_emb = candidate_readout(
            dev[0].detach(), cls_index=cls_index, candidate_index=cand_index, token_norm_weight=dev[1].detach(),
            pool_norm_weight=dev[2].detach(), fc1_weight=dev[3].detach(), fc1_bias=dev[4].detach(),
            fc2_weight=dev[5].detach(), fc2_bias=dev[6].detach(), return_embedding=True, **where)
    torch.testing.assert_close(emb.detach().float(), fused_emb.float(), **TOL)
    torch.testing.assert_close(logits.detach(), fused_logits, rtol=4e-2, atol=4e-2)
    for got, expected in zip(dev, ref):
        scale = expected.grad.abs().max().item()
        error = (got.grad.detach().cpu().double() - expected.grad).abs().max().item()
        assert error <= 3e-2 * max(scale, 1e-6), (error, scale)


def test_errors(device):
    x = torch.randn(2, 8, 64).to(torch.bfloat16).to(device)
    with pytest.raises(ValueError, match="outside the sequence"):
        candidate_readout(x, cls_index=8)
    with pytest.raises(ValueError, match="not both"):
        candidate_readout(x, cls_index=0, key_lengths=torch.ones(2, dtype=torch.int32, device=device),
                          padding_mask=torch.zeros(2, 8, dtype=torch.bool, device=device))
    with pytest.raises(RuntimeError, match="bfloat16"):
        candidate_readout(x.float(), cls_index=0)
    with pytest.raises(RuntimeError, match="multiple of 8"):
        candidate_readout(torch.zeros(1, 4, 12, dtype=torch.bfloat16, device=device), cls_index=0)
    with pytest.raises(RuntimeError, match="CUDA"):
        candidate_readout(x.cpu(), cls_index=0)


@pytest.mark.parametrize("batch,tokens,d,hidden,actions", [(4, 127, 256, 33, 1), (4, 128, 256, 129, 2), (512, 9, 64, 30, 1),
                                                           (513, 9, 64, 30, 1), (600, 40, 256, 65, 3), (3, 257, 256, 256, 1),
                                                           (3, 300, 128, 100, 35), (3, 200, 512, 31, 1), (3, 161, 1000, 260, 1)])
def test_rows_that_do_not_count_leave_no_trace(device, batch, tokens, d, hidden, actions):
    """Both workgroup sizes (few samples or many), hidden layers that end inside a step, and padding rows of NaN and infinity."""
    x, wt, wp, w1, b1, w2, b2, pad = _draw(batch, tokens, d, hidden, actions, seed=tokens + hidden)
    pad[2, 0] = True
    x[pad] = float("nan")
    x[0, ::2] = float("inf")
    cls_index = 1
    pad[1:, cls_index] = False
    x[:, cls_index] = torch.randn(batch, d, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16)
    finite = x.masked_fill(pad[..., None], 0.0)
    finite[:, cls_index] = x[:, cls_index]
    want_emb, want_logits = oracle.candidate_readout(finite, pad, cls_index=cls_index, candidate_index=None,
                                                     token_norm_weight=wt, pool_norm_weight=wp, eps=1e-6,
                                                     classifier=(w1, b1, w2, b2))
    to = lambda t: t.to(device)
    with torch.no_grad():
        logits, emb = candidate_readout(to(x), cls_index=cls_index, padding_mask=to(pad), token_norm_weight=to(wt),
                                        pool_norm_weight=to(wp), fc1_weight=to(w1), fc1_bias=to(b1), fc2_weight=to(w2),
                                        fc2_bias=to(b2), return_embedding=True)
    torch.testing.assert_close(emb.cpu().float(), want_emb, **TOL)
    torch.testing.assert_close(logits.cpu(), want_logits, **TOL)


@pytest.mark.parametrize("tokens,d", [(2, 64), (17, 256), (23, 1000)])
def test_pooling_alone_of_short_samples_does_not_depend_on_the_batch(device, tokens, d):
    """Without the classifier a short sample's rows are added up in the same groups whatever the number of samples: the same bits."""
    batch = 2 * torch.cuda.get_device_properties(device).multi_processor_count + 1
    x, wt, wp, *_ = _draw(batch, tokens, d, 16, 1, seed=tokens)
    kw = dict(cls_index=0, candidate_index=1, token_norm_weight=wt.to(device), pool_norm_weight=wp.to(device))
    with torch.no_grad():
        many = candidate_readout(x.to(device), **kw)
        few = candidate_readout(x[:5].to(device), **kw)
    assert torch.equal(few, many[:5])
