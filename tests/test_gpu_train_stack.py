"""GPU parity: the training stack (``taac_stack_train_fwd`` / ``_bwd``: blocks and readout over the compact valid tokens) at the
edges of its kernels' tiles, against float64 autograd of the CPU oracle. Tolerance: every stored intermediate is rounded to bf16
once (2^-9 relative); a block stores eight in front of its output (normalised rows, q | k | v, probabilities, attention, x1, hidden
state, output; weights) and as many gradients behind it, so the error of a result in the 2-norm stays below 16 * 2^-9 = 2^-5 of its
norm per block it passes."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
import torch.nn.utils.parametrize

from oracle import reference as oracle
from taac_2026_amd.api import MetadataAttentionMask, PCVRBackbone, UnifiedInteractionBlock, run_interaction_blocks

pytestmark = pytest.mark.gpu


def _near(name: str, got: torch.Tensor, want: torch.Tensor, blocks: int) -> None:
    got, want = got.detach().cpu().double(), want.double()
    assert (got - want).norm() <= 2.0 ** -5 * blocks * want.norm() + 1e-9, (name, (got - want).norm() / want.norm())


def _near_rows(name: str, got: torch.Tensor, want: torch.Tensor, lengths: torch.Tensor, blocks: int) -> None:
    """Row by row: a row at a remainder that is missing, stale or another one is off by its whole norm, which the norm over all rows
    does not show. The same bound on the row's norm, with that of a typical row besides (a row that is small because its terms
    cancel has their roundings); padded rows are zeros."""
    got, want = got.detach().cpu().double(), want.double()
    valid = torch.arange(got.shape[1])[None, :] < lengths[:, None]
    assert not got[~valid].any(), name
    size, error = want[valid].norm(dim=-1), (got - want)[valid].norm(dim=-1)
    bound = 2.0 ** -5 * blocks * (size + size.square().mean().sqrt())
    assert (error <= bound).all(), (name, (error / bound).max())


@pytest.mark.parametrize("d_model,heads,d_ff,n_blocks,lengths,tokens,qk_norm,dtype", [
    (256, 8, 1024, 1, [1], 1, False, torch.bfloat16),                     # one token
    (256, 4, 96, 2, [0, 65, 64, 1], 65, True, torch.float32),             # around a 64-token tile; F not a multiple of a gradient tile
    (128, 4, 160, 2, [31, 33, 0], 33, False, torch.float32),
    (128, 2, 256, 1, [257, 3], 257, True, torch.bfloat16),                # rows of a sample over two workgroups of the index
    (256, 4, 96, 1, [(11 * i) % 66 for i in range(40)], 65, False, torch.float32),      # several splits of the small gradient tiles
    (256, 8, 512, 1, [(7 * i) % 33 for i in range(1100)], 32, False, torch.bfloat16),   # 256-token workgroups, some past the count
    (128, 4, 128, 1, [(5 * i) % 41 for i in range(900)], 40, False, torch.float32),
])
def test_training_stack_at_the_edges_of_its_tiles(device, d_model, heads, d_ff, n_blocks, lengths, tokens, qk_norm, dtype):
    batch = len(lengths)
    g = torch.Generator().manual_seed(d_model + tokens)
    model = PCVRBackbone(d_model=d_model, num_heads=heads, d_ff=d_ff, n_blocks=n_blocks, qk_norm=qk_norm)
    with torch.no_grad():
        for parameter in model.parameters():
            if parameter.ndim == 1:
                parameter.copy_((1.0 if parameter.mean() > 0.5 else 0.0) + 0.1 * torch.randn(parameter.shape, generator=g))
            else:
                parameter.copy_(torch.randn(parameter.shape, generator=g) * parameter.shape[1] ** -0.5)
            parameter.copy_(parameter.to(torch.bfloat16))                 # float32 masters hold bf16 values: the same network
    reference = {name: value.detach().double().requires_grad_(True) for name, value in model.named_parameters()}
    model = model.to(dtype).to(device).train()
    emb = torch.randn(batch, tokens, d_model, generator=g).to(torch.bfloat16)
    grad_hidden = torch.randn(batch, tokens, d_model, generator=g).to(torch.bfloat16)
    grad_p = torch.randn(batch, generator=g)
    lengths = torch.tensor(lengths, dtype=torch.int32)

    emb_d = emb.to(device).requires_grad_(True)
    p, hidden = model(emb_d, lengths.to(device), return_hidden=True)
    torch.autograd.backward([p, hidden], [grad_p.to(device), grad_hidden.to(device)])

    emb_r = emb.double().requires_grad_(True)
    padding = torch.arange(tokens)[None, :] >= lengths[:, None]
    mask = (~padding)[:, None, None, :].expand(batch, 1, tokens, tokens)
    x = emb_r
    for i in range(n_blocks):
        block = {name.split(".", 2)[2]: value for name, value in reference.items() if name.startswith(f"blocks.{i}.")}
        x, _ = oracle.interaction_block(x, padding, mask, block, num_heads=heads)
    keep = (~padding).double().unsqueeze(-1)
    pooled = (x * keep).sum(1) / keep.sum(1).clamp_min(1.0)
    want_p = torch.sigmoid(F.linear(pooled, reference["head.weight"], reference["head.bias"]).squeeze(-1))
    torch.autograd.backward([want_p, x * keep], [grad_p.double(), grad_hidden.double()])
    _near("p", p, want_p.detach(), n_blocks)
    _near("hidden", hidden, (x * keep).detach(), n_blocks)
    _near("tokens", emb_d.grad, emb_r.grad, n_blocks)
    _near_rows("hidden", hidden, (x * keep).detach(), lengths, n_blocks)
    _near_rows("tokens", emb_d.grad, emb_r.grad, lengths, n_blocks)
    for name, parameter in model.named_parameters():
        assert parameter.grad.dtype == dtype
        _near(name, parameter.grad, reference[name].grad, n_blocks)


@pytest.mark.parametrize("d_model,heads,d_ff,n_blocks,lengths,tokens,qk_norm,dtype", [
    (256, 8, 1024, 1, [1], 1, False, torch.bfloat16),
    (256, 4, 96, 2, [0, 65, 64, 1], 65, True, torch.float32),
    (128, 4, 160, 2, [31, 33, 0], 33, True, torch.float32),
    (256, 8, 512, 1, [(7 * i) % 33 for i in range(1100)], 32, False, torch.bfloat16),
    (128, 4, 128, 1, [(5 * i) % 41 for i in range(900)], 40, False, torch.float32),
])
def test_training_stack_with_the_persistent_kernels(device, test_hooks, d_model, heads, d_ff, n_blocks, lengths, tokens, qk_norm, dtype):
    """The same at sizes for which the few-token kernels are taken, through the kernels of large batches (a capped grid selects them)."""
    test_hooks(max_workgroups=256)
    test_training_stack_at_the_edges_of_its_tiles(device, d_model, heads, d_ff, n_blocks, lengths, tokens, qk_norm, dtype)


def test_a_stack_is_its_blocks_one_after_the_other(device):
    """``run_interaction_blocks`` under autograd (17 blocks: more than one set-up launch) = the blocks called one by one, bit for
    bit: every kernel is the same, and gathering and scattering the valid rows in between changes no value."""
    g = torch.Generator().manual_seed(3)
    roles = torch.tensor([0, 1] + [2] * 5 + [3] * 3 + [6] * 30 + [7] * 2).to(device)
    batch, tokens, n_blocks = 3, roles.numel(), 17
    blocks = [UnifiedInteractionBlock(128, 4, 1).to(torch.bfloat16).to(device).train() for _ in range(n_blocks)]
    x = torch.randn(batch, tokens, 128, generator=g).to(torch.bfloat16).to(device)
    padding = torch.rand(batch, tokens, generator=g) < 0.4
    padding[:, :2] = False
    padding[1] = True
    padding = padding.to(device)
    grad = torch.randn(batch, tokens, 128, generator=g).to(torch.bfloat16).to(device)

    def run(one_by_one: bool):
        mask = MetadataAttentionMask(enabled=True)(padding, roles)
        xd = x.clone().requires_grad_(True)
        for block in blocks:
            block.zero_grad(set_to_none=True)
        out = xd
        if one_by_one:
            for block in blocks:
                out, _ = block(out, padding, mask, return_attention_tokens=False)
        else:
            out = run_interaction_blocks(blocks, xd, padding, mask)
        out.backward(grad)
        return [out.detach(), xd.grad] + [p.grad for block in blocks for p in block.parameters()]

    for got, want in zip(run(False), run(True)):
        assert torch.equal(got, want)


def test_computed_weights_are_taken_where_a_module_holds_no_parameter(device):
    """A parametrised weight is not in its module's registry: it is computed at each access. The network takes it like the plain
    network with the same value, and its gradient reaches what it is computed from."""
    class Double(torch.nn.Module):
        def forward(self, weight):
            return weight * 2.0

    g = torch.Generator().manual_seed(5)
    plain = PCVRBackbone(d_model=128, num_heads=4, d_ff=128, n_blocks=2).to(torch.bfloat16).to(device)
    computed = PCVRBackbone(d_model=128, num_heads=4, d_ff=128, n_blocks=2).to(torch.bfloat16).to(device)
    computed.load_state_dict(plain.state_dict())
    with torch.no_grad():
        for block, other in zip(plain.blocks, computed.blocks):
            for module, target in ((block.qkv, other.qkv), (block.down, other.down), (block.ffn_norm, other.ffn_norm)):
                module.weight.mul_(2.0)                                   # exact in bf16
                torch.nn.utils.parametrize.register_parametrization(target, "weight", Double(), unsafe=True)
    emb = torch.randn(3, 40, 128, generator=g).to(torch.bfloat16).to(device)
    lengths = torch.tensor([40, 0, 17], dtype=torch.int32, device=device)
    with torch.no_grad():
        assert torch.equal(computed(emb, lengths), plain(emb, lengths))
    got, want = computed(emb, lengths), plain(emb, lengths)
    assert torch.equal(got, want)
    got.sum().backward()
    want.sum().backward()
    for block, other in zip(plain.blocks, computed.blocks):
        assert torch.equal(other.up.weight.grad, block.up.weight.grad)
        for module, target in ((block.qkv, other.qkv), (block.down, other.down), (block.ffn_norm, other.ffn_norm)):
            assert torch.equal(target.parametrizations.weight.original.grad, module.weight.grad * 2.0)


def test_a_head_without_bias_trains(device):
    """No bias = a bias of zero: the same probabilities and gradients, bit for bit."""
    g = torch.Generator().manual_seed(6)
    emb = torch.randn(3, 40, 128, generator=g).to(torch.bfloat16).to(device)
    lengths = torch.tensor([40, 0, 17], dtype=torch.int32, device=device)
    zero, none = (PCVRBackbone(d_model=128, num_heads=4, d_ff=128, n_blocks=1).to(torch.bfloat16).to(device) for _ in range(2))
    none.load_state_dict(zero.state_dict())
    none.head.bias = None
    got, want = none(emb, lengths), zero(emb, lengths)
    assert torch.equal(got, want)
    got.sum().backward()
    want.sum().backward()
    for name, parameter in none.named_parameters():
        assert torch.equal(parameter.grad, zero.get_parameter(name).grad), name


def _network(d_model, heads, d_ff, n_blocks, seed):
    """A network whose parameters are bf16 values, and its parameters as float64 leaves."""
    g = torch.Generator().manual_seed(seed)
    model = PCVRBackbone(d_model=d_model, num_heads=heads, d_ff=d_ff, n_blocks=n_blocks)
    with torch.no_grad():
        for parameter in model.parameters():
            spread = torch.randn(parameter.shape, generator=g)
            center = 1.0 if parameter.ndim == 1 and parameter.mean() > 0.5 else 0.0
            parameter.copy_((center + spread * (0.1 if parameter.ndim == 1 else parameter.shape[1] ** -0.5)).to(torch.bfloat16))
    return model, {name: value.detach().double().requires_grad_(True) for name, value in model.named_parameters()}


def _oracle_hidden(reference, emb, lengths, heads, n_blocks):
    padding = torch.arange(emb.shape[1])[None, :] >= lengths[:, None]
    mask = (~padding)[:, None, None, :].expand(emb.shape[0], 1, emb.shape[1], emb.shape[1])
    x = emb
    for i in range(n_blocks):
        block = {name.split(".", 2)[2]: value for name, value in reference.items() if name.startswith(f"blocks.{i}.")}
        x, _ = oracle.interaction_block(x, padding, mask, block, num_heads=heads)
    return x * (~padding).double().unsqueeze(-1)


def test_samples_beyond_the_offsets_of_the_direct_transfers(device):
    """q | k | v rows of 768 values and 1 398 102 positions: the offsets inside a sample may need more than 31 bits, so the
    attention takes its general kernels. Every sample is still its own (few valid tokens, so that the oracle stays small)."""
    tokens, short, lengths = 1_398_102, 71, torch.tensor([71, 33], dtype=torch.int32)
    if torch.cuda.get_device_properties(device).total_memory < 100 * 2 ** 30:
        pytest.skip("about 30 GB of tensors")
    g = torch.Generator().manual_seed(11)
    model, reference = _network(256, 4, 32, 1, seed=12)
    model = model.to(torch.bfloat16).to(device).train()
    emb = torch.randn(2, short, 256, generator=g).to(torch.bfloat16)
    grad = torch.randn(2, short, 256, generator=g).to(torch.bfloat16)
    emb_d = torch.zeros(2, tokens, 256, dtype=torch.bfloat16, device=device)
    emb_d[:, :short] = emb.to(device)
    emb_d.requires_grad_(True)
    _, hidden = model(emb_d, lengths.to(device), return_hidden=True)
    grad_d = torch.zeros_like(hidden)
    grad_d[:, :short] = grad.to(device)
    hidden.backward(grad_d)
    del grad_d

    emb_r = emb.double().requires_grad_(True)
    want = _oracle_hidden(reference, emb_r, lengths, 4, 1)
    want.backward(grad.double())
    for b in range(2):
        _near(f"hidden of sample {b}", hidden[b, :short], want[b].detach(), 1)
        _near(f"tokens of sample {b}", emb_d.grad[b, :short], emb_r.grad[b], 1)
    assert not hidden[:, short:].any() and not emb_d.grad[:, short:].any()
    for name, parameter in model.named_parameters():
        if not name.startswith("head."):
            _near(name, parameter.grad, reference[name].grad, 1)
    del hidden, emb_d, parameter
    model.zero_grad(set_to_none=True)
    torch.cuda.empty_cache()


def test_a_head_of_several_outputs_trains(device):
    """``Linear(D, 3)`` in the place of the head: probabilities and gradients against the oracle, every row of the head's too."""
    g = torch.Generator().manual_seed(21)
    tokens, lengths = 40, torch.tensor([40, 0, 17, 33], dtype=torch.int32)
    model, reference = _network(128, 4, 128, 2, seed=22)
    model.head = torch.nn.Linear(128, 3)
    with torch.no_grad():
        for parameter in model.head.parameters():
            parameter.copy_((0.3 * torch.randn(parameter.shape, generator=g)).to(torch.bfloat16))
    reference.update({f"head.{name}": value.detach().double().requires_grad_(True) for name, value in model.head.named_parameters()})
    emb, grad = torch.randn(4, tokens, 128, generator=g).to(torch.bfloat16), torch.randn(4, 3, generator=g)
    model = model.to(torch.bfloat16).to(device).train()
    emb_d, emb_r = emb.to(device).requires_grad_(True), emb.double().requires_grad_(True)
    got = model(emb_d, lengths.to(device))
    got.backward(grad.to(device))
    want = _oracle_hidden(reference, emb_r, lengths, 4, 2).sum(1) / lengths.clamp_min(1).double().unsqueeze(-1)
    want = torch.sigmoid(F.linear(want, reference["head.weight"], reference["head.bias"]))
    want.backward(grad.double())
    assert got.shape == (4, 3)
    _near("p", got, want.detach(), 2)
    _near("tokens", emb_d.grad, emb_r.grad, 2)
    for name, parameter in model.named_parameters():
        _near(name, parameter.grad, reference[name].grad, 2)
    for row in range(3):
        _near(f"head.weight[{row}]", model.head.weight.grad[row], reference["head.weight"].grad[row], 2)


def test_blocks_of_different_hidden_sizes_train(device):
    """A network whose middle block was replaced by a narrower one: each block with its own shapes."""
    g = torch.Generator().manual_seed(23)
    tokens, lengths = 45, torch.tensor([45, 0, 17, 33, 1], dtype=torch.int32)
    model, reference = _network(256, 8, 256, 3, seed=24)
    other, _ = _network(256, 8, 96, 1, seed=25)
    model.blocks[1] = other.blocks[0]
    reference = {name: value.detach().double().requires_grad_(True) for name, value in model.named_parameters()}
    emb, grad = torch.randn(5, tokens, 256, generator=g).to(torch.bfloat16), torch.randn(5, generator=g)
    model = model.to(torch.bfloat16).to(device).train()
    emb_d, emb_r = emb.to(device).requires_grad_(True), emb.double().requires_grad_(True)
    got, hidden = model(emb_d, lengths.to(device), return_hidden=True)
    grad_hidden = torch.randn(5, tokens, 256, generator=g).to(torch.bfloat16)
    torch.autograd.backward([got, hidden], [grad.to(device), grad_hidden.to(device)])
    want_hidden = _oracle_hidden(reference, emb_r, lengths, 8, 3)
    pooled = want_hidden.sum(1) / lengths.clamp_min(1).double().unsqueeze(-1)
    want = torch.sigmoid(F.linear(pooled, reference["head.weight"], reference["head.bias"]).squeeze(-1))
    torch.autograd.backward([want, want_hidden], [grad.double(), grad_hidden.double()])
    _near("p", got, want.detach(), 3)
    _near("hidden", hidden, want_hidden.detach(), 3)
    _near("tokens", emb_d.grad, emb_r.grad, 3)
    for name, parameter in model.named_parameters():
        _near(name, parameter.grad, reference[name].grad, 3)


def test_a_layer_of_another_shape_is_refused(device):
    model = PCVRBackbone(d_model=128, num_heads=4, d_ff=128, n_blocks=2)
    model.blocks[1].up = torch.nn.Linear(128, 2 * 96)  # narrower than its down projection
    model = model.to(torch.bfloat16).to(device).train()
    lengths = torch.tensor([5, 0], dtype=torch.int32, device=device)
    with pytest.raises(ValueError, match="does not fit a block"):
        model(torch.zeros(2, 8, 128, dtype=torch.bfloat16, device=device), lengths)
    model.blocks[1].up = torch.nn.Linear(128, 2 * 128).to(torch.bfloat16)  # left on the host
    with pytest.raises(RuntimeError, match="same device"):
        model(torch.zeros(2, 8, 128, dtype=torch.bfloat16, device=device), lengths)


@pytest.mark.parametrize("d_model,dtype", [(256, torch.bfloat16), (128, torch.float32)])
def test_the_feed_forward_backward_rounds_no_product_of_two_weights(device, d_model, dtype):
    """Rows that the norm maps to +-1, a norm weight and up weights whose products all lie 0.3 % above the bf16 value below them: the
    hidden state of the backward is off by that much wherever the two are multiplied and rounded in front of the product, and the
    down projection's gradient, which is linear in it, shrinks. Otherwise normalised rows and products are exact and the hidden
    state is rounded once, 2^-9 of each value at most: no further may the gradient be off along the true one."""
    g = torch.Generator().manual_seed(31)
    batch, tokens, d_ff = 40, 65, 256
    model, _ = _network(d_model, 4, d_ff, 1, seed=32)
    block = model.blocks[0]
    with torch.no_grad():
        for parameter in (block.out.weight, block.out.bias, block.up.bias):
            parameter.zero_()
        block.ffn_norm.weight.fill_(1 + 9 / 128)
        block.up.weight.copy_(torch.where(torch.rand(block.up.weight.shape, generator=g) < 0.5, -1.0, 1.0) * (1 + 7 / 128) / 16)
    reference = {name: value.detach().double().requires_grad_(True) for name, value in model.named_parameters()}
    emb = torch.where(torch.rand(batch, tokens, d_model, generator=g) < 0.5, -1.0, 1.0).to(torch.bfloat16)
    grad = torch.randn(batch, tokens, d_model, generator=g).to(torch.bfloat16)
    lengths = torch.full((batch,), tokens, dtype=torch.int32)
    model = model.to(dtype).to(device).train()
    _, hidden = model(emb.to(device), lengths.to(device), return_hidden=True)
    hidden.backward(grad.to(device))
    _oracle_hidden(reference, emb.double(), lengths, 4, 1).backward(grad.double())
    got, want = model.blocks[0].down.weight.grad.cpu().double(), reference["blocks.0.down.weight"].grad
    along = float((got * want).sum() / (want * want).sum())
    assert abs(along - 1.0) <= 2.0 ** -9, along


def test_hooks_of_all_modules_and_replaced_forwards_see_every_block_of_a_stack(device):
    roles = torch.tensor([0, 1, 2, 3, 6, 6, 6, 7]).to(device)
    blocks = [UnifiedInteractionBlock(128, 4, 1).to(torch.bfloat16).to(device).train() for _ in range(3)]
    padding = torch.zeros(2, roles.numel(), dtype=torch.bool, device=device)
    x = torch.randn(2, roles.numel(), 128, device=device).to(torch.bfloat16).requires_grad_(True)
    mask = MetadataAttentionMask(enabled=True)(padding, roles)
    seen: list = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda module, args, out: seen.append(module))
    try:
        run_interaction_blocks(blocks, x, padding, mask)
    finally:
        handle.remove()
    assert [module for module in seen if module in blocks] == blocks
    blocks[1].forward = lambda tokens, *args, **kwargs: (tokens * 0, None)
    assert not run_interaction_blocks(blocks[:2], x, padding, mask).any()


def test_training_stack_with_the_kernels_of_large_batches(device):
    """More positions than 512 per compute unit: the input gradient of the up projection takes its 256-token workgroups, the last of
    which holds a remainder. The samples are short and the oracle sees their first positions only."""
    batch, tokens, short = 2049, 64, 9
    assert batch * tokens > 512 * torch.cuda.get_device_properties(device).multi_processor_count
    lengths = torch.tensor([(7 * i) % short for i in range(batch)], dtype=torch.int32)
    assert int(lengths.sum()) % 256 not in (0, 255)
    g = torch.Generator().manual_seed(41)
    model, reference = _network(256, 8, 1024, 1, seed=42)
    emb, grad = (torch.randn(batch, tokens, 256, generator=g).to(torch.bfloat16) for _ in range(2))
    model = model.to(torch.bfloat16).to(device).train()
    emb_d = emb.to(device).requires_grad_(True)
    _, hidden = model(emb_d, lengths.to(device), return_hidden=True)
    hidden.backward(grad.to(device))
    emb_r = emb[:, :short].double().requires_grad_(True)
    want = _oracle_hidden(reference, emb_r, lengths, 8, 1)
    want.backward(grad[:, :short].double())
    assert not hidden[:, short:].any() and not emb_d.grad[:, short:].any()
    for name, got, right in (("hidden", hidden[:, :short], want.detach()), ("tokens", emb_d.grad[:, :short], emb_r.grad)):
        _near(name, got, right, 1)
        _near_rows(name, got, right, lengths, 1)
    for name, parameter in model.named_parameters():
        if not name.startswith("head."):
            _near(name, parameter.grad, reference[name].grad, 1)


@pytest.mark.parametrize("d_model,heads,batch,tokens,full,gate_first", [
    (256, 8, 140, 130, False, True), (256, 4, 600, 130, True, True), (128, 4, 300, 130, False, True), (128, 2, 1100, 130, True, True),
    (256, 4, 140, 130, False, False), (128, 4, 300, 130, False, False)])
def test_tokens_between_the_halves_of_a_large_batch(device, test_hooks, d_model, heads, batch, tokens, full, gate_first):
    """The persistent feed-forward kernel of the training forward (a capped grid selects it whatever the number of rows; with the
    activation's constants in the weights, gate first, and without) stores the tokens between a block's halves while it projects: against
    the inference route, which writes them with a kernel of their own, over slices of a few wavefronts and, with enough tokens, over
    whole tiles and a remainder. Both round the projection and the sum once (2^-8 of values below 8: 2^-5 each); on the whole the
    two differ by one rounding. Gate last, the inference route's up weights hold the activation's constants and are rounded with them: a
    gate and a value that are 2^-9 off each, 2^-8 of the update more."""
    test_hooks(max_workgroups=256)
    whole = 2.0 ** -8 if gate_first else 2.0 ** -7
    g = torch.Generator(device=device).manual_seed(batch)
    block = UnifiedInteractionBlock(d_model, heads, 2)
    with torch.no_grad():
        for name, p in block.named_parameters():
            p.copy_(torch.randn(p.shape, generator=torch.Generator().manual_seed(len(name))) * (p.shape[-1] ** -0.5 if p.ndim == 2 else 0.1)
                    + (1.0 if name.endswith("norm.weight") else 0.0))
    block = block.to(torch.bfloat16).to(device)
    block.ffn.gate_first = gate_first
    x = torch.randn(batch, tokens, d_model, generator=g, device=device).to(torch.bfloat16)
    lengths = torch.randint(tokens - 1 if full else 0, tokens + 1, (batch,), generator=g, device=device, dtype=torch.int32)
    padding = torch.arange(tokens, device=device) >= lengths[:, None]
    with torch.no_grad():
        out, between = block.eval()(x, padding, None, key_lengths=lengths)
    got_out, got_between = block.train()(x.clone().requires_grad_(True), padding, None, key_lengths=lengths)
    for got, want in ((got_between, between), (got_out, out)):
        a, b = got[~padding].float(), want[~padding].float()
        assert b.abs().max() < 8 and (a - b).abs().max() <= 2.0 ** -4 and (a - b).norm() <= whole * b.norm()
        assert torch.equal(got[padding], x[padding])


@pytest.mark.parametrize("d_model,heads,batch,tokens", [(256, 8, 900, 25), (128, 4, 1500, 27)])
def test_query_and_key_norms_of_several_steps_a_workgroup(device, d_model, heads, batch, tokens):
    """More rows than the workgroups of the norms' backward take at once: two whole steps and a part of a third."""
    lengths = [(11 * i) % (tokens + 1) for i in range(batch)]
    test_training_stack_at_the_edges_of_its_tiles(device, d_model, heads, 64, 1, lengths, tokens, True, torch.bfloat16)


@pytest.mark.parametrize("width,tokens", [(128, 1), (128, 545), (128, 700), (256, 96), (256, 1056)])
def test_rows_go_back_to_where_scattered_padding_left_them(device, width, tokens):
    """Under a role mask with padding inside the samples: the training stack's output has the rows of the inference kernels' (same values but
    for roundings; a row at another's place is off by its norm), and padded rows carry the gradient that arrives."""
    g = torch.Generator(device=device).manual_seed(tokens)
    blocks = torch.nn.ModuleList([UnifiedInteractionBlock(width, width // 32, 2)]).to(device).to(torch.bfloat16)
    x, grad = (torch.randn(3, tokens, width, generator=g, device=device).to(torch.bfloat16) for _ in range(2))
    padding = torch.rand(3, tokens, generator=g, device=device) < torch.tensor([0.2, 0.8, 0.5], device=device)[:, None]
    padding[:, 0] = False
    mask = MetadataAttentionMask(enabled=True)(padding, torch.randint(0, 8, (tokens,), generator=g, device=device))
    leaf = x.clone().requires_grad_(True)
    out = run_interaction_blocks(blocks, leaf, padding, mask)
    out.backward(grad)
    with torch.no_grad():
        want = run_interaction_blocks(blocks, x, padding, mask).float()
    error = (out.detach().float() - want).norm(dim=-1)
    assert (error <= 2.0 ** -4 * want.norm(dim=-1)).all()
    assert torch.equal(out.detach()[padding], x[padding]) and torch.equal(leaf.grad[padding], grad[padding])
    assert ((leaf.grad - grad)[~padding].float().norm(dim=-1) > 0).all()
