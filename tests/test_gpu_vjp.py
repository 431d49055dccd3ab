"""GPU parity of the audit's margin helpers (code_for_iclr27_amd.vjp, HIP kernels through the C
ABI) against the f64 oracle: head logits for bf16/f16/f32 weights with and without bias, 1..8
rows (several row passes), odd vocabulary sizes and the Llama-3.2-1B / 3.1-8B / Qwen-style hidden
sizes; margins with given and argmax targets; hidden gradients (single target and per-row
targets with due flags); per-layer pre-projection gradients with and without the output gate.

Tolerance (f32 arithmetic, summation order differs from the reference's GEMMs): each result
within 1e-5 of the sum of the absolute values of its terms (plus 1e-6 absolute); margins and
gradients are checked on the GPU's own logits, so each kernel is checked on its own.
"""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from code_for_iclr27_amd import vjp
from oracle import vjp as ovjp

pytestmark = pytest.mark.gpu


def model_with_head(device, vocab, dim, dtype=torch.bfloat16, bias=False, seed=0):
    g = torch.Generator().manual_seed(seed)
    weight = (torch.randn((vocab, dim), generator=g) * 0.05).to(dtype)
    head = SimpleNamespace(weight=weight.to(device),
                           bias=(torch.randn(vocab, generator=g).to(dtype).to(device)
                                 if bias else None))
    return SimpleNamespace(get_output_embeddings=lambda: head), weight.double().numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab,dim,bias", [(1, 32000, 4096, False), (3, 1001, 2048, True),
                                                 (8, 4099, 4096, False), (2, 777, 5120, True)])
def test_head_logits(device, dtype, rows, vocab, dim, bias):
    model, weight = model_with_head(device, vocab, dim, dtype, bias, seed=rows)
    hidden = torch.randn((rows, dim), generator=torch.Generator().manual_seed(9))
    got = vjp.last_token_logits_float32(model, hidden.to(device).to(torch.bfloat16)).cpu().numpy()
    x = hidden.to(torch.bfloat16).double().numpy()
    b = None if not bias else model.get_output_embeddings().bias.double().cpu().numpy()
    expect = ovjp.head_logits(x, weight, b)
    scale = np.abs(x) @ np.abs(weight).T + (0 if b is None else np.abs(b))
    assert got.shape == (rows, vocab) and got.dtype == np.float32
    assert np.all(np.abs(got - expect) <= 1e-5 * scale + 1e-6)


@pytest.mark.parametrize("rows,vocab,dim,bias", [
    (2, 32, 1024, False),    # one weight tile, one stage a wave
    (8, 33, 2048, True),     # a last tile that reaches back over the first
    (9, 8193, 3072, False),  # two row passes (the second of one row), a ragged last tile
    (5, 97, 5120, True),     # the largest hidden size of the matrix-core kernel
    (4, 31, 1024, True),     # fewer weight rows than a tile
    (6, 300, 1536, False),   # a hidden size the matrix-core kernel does not take
])
def test_head_logits_several_rows(device, rows, vocab, dim, bias):
    """Several f32 rows (all 24 significant bits) against a bf16 weight, from a buffer that is
    16-byte aligned and from one that is not: both kernels' row, tile and stage edges."""
    model, weight = model_with_head(device, vocab, dim, bias=bias, seed=rows + 30)
    x = torch.randn((rows, dim), generator=torch.Generator().manual_seed(31)) * 3
    b = None if not bias else model.get_output_embeddings().bias.double().cpu().numpy()
    expect = ovjp.head_logits(x.double().numpy(), weight, b)
    scale = np.abs(x.double().numpy()) @ np.abs(weight).T + (0 if b is None else np.abs(b))
    shifted = torch.empty(rows * dim + 1, device=device)[1:].view(rows, dim)
    assert shifted.data_ptr() % 16 == 4
    for hidden in (x.to(device), shifted.copy_(x)):
        got = vjp.last_token_logits_float32(model, hidden).cpu().numpy()
        # the longest f32 chain is 128 sums a row part and eight parts: well under 1e-6 of scale
        assert np.all(np.abs(got - expect) <= 1e-6 * scale)


@pytest.mark.parametrize("rows,vocab,dim,bias", [
    (8, 32, 1024, False), (5, 33, 2048, True), (3, 2047, 3072, False), (4, 2048, 3072, True),
    (2, 16383, 1024, True), (2, 16384, 1024, False), (2, 16384, 4096, False)])
def test_head_logits_both_sides_of_the_kernel_choice(device, rows, vocab, dim, bias):
    """The vocabularies between which two, three and more rows change from one kernel to the other."""
    test_head_logits_several_rows(device, rows, vocab, dim, bias)


def test_head_logits_non_finite_rows_and_weights(device):
    """Infinities and NaN go where f32 arithmetic takes them, and nowhere else."""
    model, weight = model_with_head(device, 64, 1024, seed=40)
    x = torch.randn((3, 1024), generator=torch.Generator().manual_seed(41))
    x[0, 5], x[1, 900] = float("inf"), float("nan")
    clean = vjp.last_token_logits_float32(model, x[2:].repeat(2, 1).to(device))[:1]
    got = vjp.last_token_logits_float32(model, x.to(device)).cpu()
    signs = torch.from_numpy(np.sign(weight[:, 5])).float()
    assert torch.equal(got[0], signs * float("inf")) and torch.isnan(got[1]).all()
    assert torch.equal(got[2], clean[0].cpu())
    w = model.get_output_embeddings().weight
    w[7, 3] = float("-inf")
    x[2, 3] = 2.0  # its second and third pieces are zero
    got = vjp.last_token_logits_float32(model, x.to(device)).cpu()
    assert got[2, 7] == float("-inf") and torch.isfinite(got[2][torch.arange(64) != 7]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,vocab,dim", [(3, 17, 128), (8, 513, 640), (5, 4100, 512),
                                            (11, 1000, 1024), (8, 200, 1000)])
def test_row_hidden_gradients_several_rows(device, dtype, rows, vocab, dim):
    """Ragged weight rows and column blocks, two row passes (8 and 3), and a width that the
    matrix-core kernel does not take (1000)."""
    model, weight = model_with_head(device, vocab, dim, dtype, seed=rows + 50)
    logits = torch.randn((rows, vocab), generator=torch.Generator().manual_seed(51)).to(device) * 3
    _, targets, competitors = vjp.row_margins(logits)
    due = [float(r != 1) for r in range(rows)]
    got = vjp.row_hidden_gradients(model, logits, targets, competitors, due).cpu().numpy()
    l64, t = logits.double().cpu().numpy(), targets.cpu().numpy()
    expect = ovjp.hidden_gradient(l64, t, weight, np.array(due))
    share = np.exp(l64 - l64.max(axis=1, keepdims=True))
    share[np.arange(rows), t] = 0
    scale = np.abs(weight[t]) + (share / share.sum(axis=1, keepdims=True)) @ np.abs(weight)
    # the shares carry expf's and the division's f32 rounding, the sums chains of at most 32 + 251
    assert np.all(np.abs(got - expect) <= 2e-6 * scale)


@pytest.mark.parametrize("rows,vocab,dim", [(3, 58593, 1024), (4, 58594, 1024), (3, 100, 1000)])
def test_row_hidden_gradients_three_and_four_rows(device, rows, vocab, dim):
    """Three and four rows on both sides of the weights at which they change kernels, bf16 and f32
    (whose sums of four rows wait for a whole group of weight rows)."""
    for dtype in (torch.bfloat16, torch.float32):
        test_row_hidden_gradients_several_rows(device, dtype, rows, vocab, dim)


@pytest.mark.parametrize("rows,vocab,dim", [(3, 17, 128), (8, 63, 256), (5, 513, 512)])
def test_row_hidden_gradients_infinite_weights(device, rows, vocab, dim):
    """Infinities in the last weight rows (block and stage remainders) reach the gradients with
    their sign in their own columns, as the f32 sum over the rows has it, and nothing else."""
    model, _ = model_with_head(device, vocab, dim, seed=rows + 60)
    w = model.get_output_embeddings().weight
    w[vocab - 1, 3], w[vocab - 1, dim - 1], w[vocab - 2, 40] = float("inf"), float("-inf"), float("inf")
    logits = torch.randn((rows, vocab), generator=torch.Generator().manual_seed(61)).to(device)
    logits[:, 2] = 9.0  # the target of every row, a finite weight row
    _, targets, competitors = vjp.row_margins(logits)
    got = vjp.row_hidden_gradients(model, logits, targets, competitors, [1.0] * rows).cpu()
    expect = torch.full((rows, dim), 0.0)
    expect[:, 3], expect[:, dim - 1], expect[:, 40] = -float("inf"), float("inf"), -float("inf")
    assert torch.equal(torch.where(torch.isfinite(got), torch.zeros(()), got), expect)


@pytest.mark.parametrize("layers,hidden,width", [(1, 2048, 2048), (11, 2048, 2048),
                                                 (12, 2048, 2048), (6, 2100, 2056), (40, 300, 64)])
def test_pre_gradients_layer_counts_match_per_layer(device, layers, hidden, width):
    """Few layers (a partial row a row block), many (one a reduction group) and both sides of the
    line between them: the per-layer call's sums in the same order, bit for bit."""
    g = torch.Generator(device=device).manual_seed(layers)
    weights = [torch.randn((hidden, width), generator=g, device=device).to(torch.bfloat16)
               for _ in range(layers)]
    posts = [torch.randn(hidden, generator=g, device=device) for _ in range(layers)]
    batched = vjp.pre_gradients(posts, weights, width // 8, 8)
    for post, weight, got in zip(posts, weights, batched):
        assert torch.equal(got, vjp.pre_gradient(post, weight, width // 8, 8))


def test_margins_given_and_argmax(device):
    rng = np.random.default_rng(3)
    logits = (rng.standard_normal((4, 128256)) * 3).astype(np.float32)
    logits[2, 5] = logits[2, 9] = logits[2].max() + 1  # a tie: the first index wins
    dev = torch.from_numpy(logits).to(device)
    margins, targets, competitors = vjp.row_margins(dev)
    expect, expect_targets, _, _ = ovjp.margin_stats(logits)
    np.testing.assert_array_equal(targets.cpu().numpy(), expect_targets)
    assert targets[2].item() == 5
    np.testing.assert_allclose(margins.cpu().numpy(), expect, rtol=0, atol=1e-5 * (1 + np.abs(expect)).max())
    assert torch.isneginf(competitors[np.arange(4), targets]).all()
    single = vjp.one_vs_rest_margin(dev[1:2], 77)
    np.testing.assert_allclose(single.item(), ovjp.margin_stats(logits[1:2], np.array([77]))[0][0],
                               rtol=1e-6, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_hidden_gradient_single_target(device, dtype):
    vocab, dim = 32000, 4096
    model, weight = model_with_head(device, vocab, dim, dtype, seed=4)
    hidden = torch.randn((1, dim), generator=torch.Generator().manual_seed(5)).to(device)
    logits = vjp.last_token_logits_float32(model, hidden)
    target = int(logits.argmax().item())
    got = vjp.one_vs_rest_hidden_gradient(model, logits, target).cpu().numpy()
    l64 = logits.double().cpu().numpy()
    expect = ovjp.hidden_gradient(l64, np.array([target]), weight)
    comp = l64.copy()
    comp[0, target] = -np.inf
    p = np.exp(comp - comp.max()) / np.exp(comp - comp.max()).sum()
    scale = np.abs(weight[target]) + p @ np.abs(weight)
    assert got.shape == (1, dim)
    assert np.all(np.abs(got - expect) <= 1e-5 * scale + 1e-6)


def test_row_hidden_gradients_with_due(device):
    vocab, dim = 5003, 2048
    model, weight = model_with_head(device, vocab, dim, seed=6)
    logits = torch.randn((3, vocab), generator=torch.Generator().manual_seed(7)).to(device) * 2
    margins, targets, competitors = vjp.row_margins(logits)
    got = vjp.row_hidden_gradients(model, logits, targets, competitors, [True, False, True])
    got = got.cpu().numpy()
    l64 = logits.double().cpu().numpy()
    t = targets.cpu().numpy()
    expect = ovjp.hidden_gradient(l64, t, weight, np.array([1.0, 0.0, 1.0]))
    np.testing.assert_array_equal(got[1], 0.0)
    assert np.all(np.abs(got - expect) <= 1e-5 * (np.abs(weight[t]) + np.abs(weight).max()) + 1e-6)


@pytest.mark.parametrize("hidden,width,dtype,gated", [(4096, 4096, torch.bfloat16, False),
                                                      (5120, 6144, torch.bfloat16, True),
                                                      (100, 64, torch.float32, True),
                                                      (2048, 2048, torch.float16, False)])
def test_pre_gradient(device, hidden, width, dtype, gated):
    g = torch.Generator().manual_seed(hidden + width)
    o_weight = (torch.randn((hidden, width), generator=g) * 0.02).to(dtype)
    post = torch.randn(hidden, generator=g)
    gate = torch.rand(width, generator=g) if gated else None
    heads = width // 64
    got = vjp.pre_gradient(post.to(device), o_weight.to(device), heads, 64,
                           None if gate is None else gate.to(device))
    assert got.shape == (heads, 64)
    w = o_weight.double().numpy()
    expect = ovjp.pre_gradient(post.double().numpy(), w,
                               None if gate is None else gate.double().numpy())
    scale = np.abs(post.double().numpy()) @ np.abs(w)
    if gate is not None:
        scale = scale * np.abs(gate.double().numpy())
    assert np.all(np.abs(got.reshape(-1).cpu().numpy() - expect) <= 1e-5 * scale + 1e-6)


@pytest.mark.parametrize("dtype,gated", [(torch.bfloat16, False), (torch.float32, True)])
def test_pre_gradients_all_layers_match_per_layer(device, dtype, gated):
    layers, hidden, heads, dim = 5, 2048, 16, 128
    g = torch.Generator().manual_seed(21)
    weights = [(torch.randn((hidden, heads * dim), generator=g) * 0.02).to(dtype).to(device)
               for _ in range(layers)]
    posts = [torch.randn(hidden, generator=g).to(device) for _ in range(layers)]
    gates = [torch.rand(heads * dim, generator=g).to(device) if gated and l % 2 == 0 else None
             for l in range(layers)]
    batched = vjp.pre_gradients(posts, weights, heads, dim, gates)
    for l in range(layers):
        single = vjp.pre_gradient(posts[l], weights[l], heads, dim, gates[l])
        assert batched[l].shape == (heads, dim)
        torch.testing.assert_close(batched[l], single, rtol=0, atol=0)  # same sums, same order


def test_misaligned_weight_views_rejected(device):
    hidden, heads, dim = 64, 2, 64
    backing = torch.zeros(hidden * heads * dim + 1, dtype=torch.bfloat16, device=device)
    misaligned = backing[1:].view(hidden, heads * dim)  # contiguous, 2 bytes off 16-byte alignment
    assert misaligned.data_ptr() % 16 == 2
    aligned = torch.zeros((hidden, heads * dim), dtype=torch.bfloat16, device=device)
    post = torch.ones(hidden, device=device)
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        vjp.pre_gradient(post, misaligned, heads, dim)
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        vjp.pre_gradients([post, post], [aligned, misaligned], heads, dim)
