"""GPU parity of surprise scoring and salience admission.

* causal_surprise (prior-state front): forward 3e-4, backward 2e-3
  (tests/cuda/test_think_cuda.py:89, 118-120), invalid rows exactly 0,
  causality.
* surprise_from_logits: bit-identical to the C oracle (same exp/log routines
  and summation order), and within a few fp32 ulp of the float64 formula.
* admission: tau and the mask bit-identical to the oracle (torch.quantile
  semantics), and the mask equal to the reference torch path's
  (cross_entropy scores, torch.quantile) on the C2 input and eight more
  C2-shaped seeds.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from koemi_amd import think, workloads

pytestmark = pytest.mark.gpu


def reference_causal_surprise(prior, weight, bias, targets, valid):
    logits = torch.matmul(prior.float(), weight.float().transpose(0, 1)) + bias.float()
    nll = torch.logsumexp(logits, dim=-1) - logits.gather(-1, targets.unsqueeze(-1)).squeeze(-1)
    s = 1.0 - torch.exp(-nll / math.log(weight.shape[0]))
    return torch.where(valid, s, torch.zeros_like(s)).to(prior.dtype)


def build_inputs(device, requires_grad=False):
    torch.manual_seed(17)
    prior = torch.randn(2, 7, 8)
    weight = torch.randn(19, 8)
    bias = torch.randn(19)
    targets = torch.randint(0, 19, (2, 7))
    valid = torch.ones(2, 7, dtype=torch.bool)
    valid[0, -1] = False
    out = [prior, weight, bias]
    out = [t.to(device).requires_grad_(requires_grad) for t in out]
    return (*out, targets.to(device), valid.to(device))


def test_causal_surprise_forward(device):
    inputs = build_inputs(device)
    got = think.causal_surprise(*inputs)
    want = reference_causal_surprise(*inputs)
    torch.testing.assert_close(got, want, rtol=3e-4, atol=3e-4)
    assert got[0, -1].item() == 0.0


def test_causal_surprise_backward(device):
    p, w, b, t, v = build_inputs(device, requires_grad=True)
    out = think.causal_surprise(p, w, b, t, v)
    grads = torch.autograd.grad(out.square().sum(), (p, w, b))
    rp, rw, rb = (x.detach().cpu().double().requires_grad_() for x in (p, w, b))
    ref = reference_causal_surprise(rp, rw, rb, t.cpu(), v.cpu()).double()
    ref_grads = torch.autograd.grad(ref.square().sum(), (rp, rw, rb))
    for got, want in zip(grads, ref_grads):
        torch.testing.assert_close(got.cpu(), want.float(), rtol=2e-3, atol=2e-3)
    assert torch.equal(grads[0][0, -1].cpu(), torch.zeros(8))


def test_causal_surprise_is_causal(device):
    inputs = build_inputs(device)
    base = think.causal_surprise(*inputs)
    changed_prior = inputs[0].clone()
    changed_prior[:, 4:] = torch.randn_like(changed_prior[:, 4:]) * 100.0
    changed_targets = inputs[3].clone()
    changed_targets[:, 4:] = (changed_targets[:, 4:] + 7) % 19
    changed = think.causal_surprise(changed_prior, inputs[1], inputs[2], changed_targets, inputs[4])
    assert torch.equal(changed[:, :4], base[:, :4])


def test_benchmark_reports_synchronized_latency(device):
    m = think.benchmark_causal_surprise(*build_inputs(device), warmup_iterations=2, measured_iterations=5)
    assert m.position_count == 14 and m.measured_iterations == 5 and m.latency_milliseconds > 0


@pytest.mark.parametrize("vocab", [2, 3, 19, 64, 128, 255, 256, 257, 1000, 1030])
def test_surprise_rows_bit_identical_to_oracle(device, vocab):
    rng = np.random.default_rng(vocab)
    logits = rng.normal(0, 2, (333, vocab)).astype(np.float32)
    bias = rng.normal(0, 1, vocab).astype(np.float32)
    targets = rng.integers(0, vocab, 333)
    valid = rng.random(333) > 0.1
    got = think.surprise_from_logits(
        torch.from_numpy(logits).to(device), torch.from_numpy(targets).to(device), torch.from_numpy(valid).to(device),
        content_bias=torch.from_numpy(bias).to(device),
    ).cpu().numpy()
    want = oracle.surprise_rows(logits, targets, valid, bias)
    np.testing.assert_array_equal(got, want)


def test_config2_surprise_and_quantile_admission_bit_exact(device):
    c = workloads.config2()
    s = think.surprise_from_logits(c.logits.to(device), c.targets.to(device), c.valid.to(device))
    mask, tau = think.salience_admission(s, c.valid.to(device), quantile=c.quantile)
    s_cpu = s.cpu().numpy()
    want_s = oracle.surprise_rows(c.logits.numpy(), c.targets.numpy(), c.valid.numpy())
    np.testing.assert_array_equal(s_cpu, want_s)
    want_mask, want_tau = oracle.admission(want_s, c.valid.numpy(), q=c.quantile)
    assert float(tau) == want_tau
    assert float(tau) == float(torch.quantile(torch.from_numpy(want_s), c.quantile))
    np.testing.assert_array_equal(mask.cpu().numpy(), want_mask)
    admitted = int(mask.sum())
    # float64 accuracy of the scores
    f64 = oracle.surprise_rows_f64(c.logits.numpy(), c.targets.numpy(), c.valid.numpy())
    max_abs = float(np.abs(s_cpu - f64).max())
    # torch's own path (network.py:681-687) and its mask
    nll = F.cross_entropy(c.logits, c.targets, reduction="none")
    torch_s = (1.0 - torch.exp(-(nll / math.log(256)))).numpy()
    torch_tau = float(torch.quantile(torch.from_numpy(torch_s), c.quantile))
    torch_mask = torch_s > torch_tau
    differ = np.nonzero(torch_mask != mask.cpu().numpy())[0]
    print(f"C2 admission: admitted={admitted} tau={float(tau):.9g} max_abs_vs_f64={max_abs:.3e} "
          f"mask_diff_vs_torch_path={differ.size}", flush=True)
    assert max_abs <= 4 * np.spacing(np.float32(1.0))
    assert differ.size == 0, "the GPU admission mask differs from the reference torch path's"
    assert admitted == int(np.sum(want_s > want_tau))


@pytest.mark.parametrize("seed", range(1003, 1011))
def test_config2_admission_equals_the_torch_path_over_seeds(device, seed):
    """C2-shaped inputs from eight more seeds: the GPU mask equals the mask of
    the reference's torch path (cross_entropy -> 1 - exp(-nll / ln 256) ->
    s > torch.quantile(s, 0.9), network.py:677-688). The scores themselves
    differ from torch's in the last ulp on ~15% of tokens (different exp/log
    implementations), so the count of torch scores within 4 ulp of its tau is
    reported: a mask can only differ where that count is non-zero."""

    c = workloads.config2(seed=seed)
    s = think.surprise_from_logits(c.logits.to(device), c.targets.to(device), c.valid.to(device))
    mask, tau = think.salience_admission(s, c.valid.to(device), quantile=0.9)
    nll = F.cross_entropy(c.logits, c.targets, reduction="none")
    torch_s = (1.0 - torch.exp(-(nll / math.log(256)))).numpy()
    torch_tau = float(torch.quantile(torch.from_numpy(torch_s), 0.9))
    near = int(np.sum(np.abs(torch_s - torch_tau) <= 4 * np.spacing(np.float32(torch_tau))))
    differ = int(np.sum((torch_s > torch_tau) != mask.cpu().numpy()))
    print(f"seed {seed}: tau={float(tau):.9g} torch_tau={torch_tau:.9g} scores_within_4ulp={near} "
          f"mask_diff={differ}", flush=True)
    assert differ == 0


@pytest.mark.parametrize(
    "case",
    ["single", "pair", "ties", "ties_aligned", "constant", "negative", "wide", "nan", "normal_32k", "odd_32k",
     "ties_32k", "outliers_32k", "zeros_32k", "sorted_32k", "nan_32k", "odd_12k", "normal_100k", "sorted_64k",
     "large"],
)
@pytest.mark.parametrize("q", [0.0, 0.25, 0.9, 1.0])
def test_quantile_admission_edge_cases(device, case, q):
    rng = np.random.default_rng(sum(map(ord, case)))
    scores = {
        "single": np.array([0.4]),
        "pair": np.array([0.9, 0.1]),
        "ties": np.repeat([0.2, 0.5, 0.7], 333),
        "constant": np.full(1000, 0.625),
        "negative": rng.normal(0, 10, 5000),
        "wide": np.concatenate([rng.uniform(0, 1, 4000), [1e-30, 3e38, -3e38, 0.0, -0.0]]),
        "nan": np.array([0.1, np.nan, 0.5, 0.7]),
        "ties_aligned": np.repeat([0.2, 0.5, 0.7], 400),
        "normal_32k": rng.normal(0.63, 0.05, 32768),
        "odd_32k": rng.normal(0.63, 0.05, 32767),
        "ties_32k": rng.choice([0.25, 0.5, 0.75], 32768),
        "outliers_32k": np.concatenate([rng.normal(0.63, 0.05, 32764), [1e-30, 3e38, -3e38, -0.0]]),
        "zeros_32k": rng.choice(np.array([-0.0, 0.0, 0.5, -1.0]), 32768),
        "sorted_32k": np.sort(rng.normal(0.63, 0.05, 32768)),
        "nan_32k": np.concatenate([rng.normal(0.63, 0.05, 20000), [np.nan], rng.normal(0.63, 0.05, 12767)]),
        "odd_12k": rng.normal(0.63, 0.05, 12001),
        "normal_100k": rng.normal(0.63, 0.05, 100_000),
        "sorted_64k": np.sort(rng.normal(0.63, 0.05, 65536)),
        "large": rng.uniform(0.5, 0.9, 300_000),
    }[case].astype(np.float32)
    valid = rng.random(scores.size) > 0.2
    mask, tau = think.salience_admission(torch.from_numpy(scores).to(device), torch.from_numpy(valid).to(device), quantile=q)
    want_mask, want_tau = oracle.admission(scores, valid, q=q)
    if math.isnan(want_tau):
        assert math.isnan(float(tau))
    else:
        assert float(tau) == want_tau
    np.testing.assert_array_equal(mask.cpu().numpy(), want_mask)


def test_fixed_threshold_admission_is_strict(device):
    s = torch.tensor([0.7, 0.75, 0.8, 0.9], device=device)
    valid = torch.tensor([True, True, True, False], device=device)
    mask, tau = think.salience_admission(s, valid, threshold=0.75)
    assert mask.tolist() == [False, False, True, False] and float(tau) == 0.75
    for dtype in (torch.bfloat16, torch.float16):
        m, _ = think.salience_admission(s.to(dtype), valid, threshold=0.75)
        assert m.tolist() == [False, False, True, False]
    assert think.admission_above(s, valid, 0.75).tolist() == [False, False, True, False]
    g = torch.Generator().manual_seed(4)
    big = torch.rand((3, 1000), generator=g).to(device)
    big_valid = (torch.rand((3, 1000), generator=g) < 0.8).to(device)
    assert torch.equal(think.admission_above(big, big_valid, 0.5),
                       think.salience_admission(big, big_valid, threshold=0.5)[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,length,width,vocab", [
    (1, 1, 1, 2), (3, 21, 8, 19), (1, 64, 64, 256), (5, 13, 72, 257), (2, 64, 300, 255), (1, 129, 136, 520),
    (4, 300, 128, 256), (3, 700, 40, 130), (2, 65, 512, 1000), (9, 600, 264, 64),
    # few tiles of a wide state (its width in chunks) and of a long vocabulary (the prior gradient's chunks)
    (1, 70, 2048, 257), (1, 16, 4096, 65), (2, 600, 1030, 100), (1, 40, 600, 700), (1, 1, 513, 2), (1, 33, 72, 3000),
    (1, 5, 24, 20000),  # tiles joined by a wave
])
def test_causal_surprise_head_of_every_tile_shape(device, dtype, batch, length, width, vocab):
    """Scores and gradients at the edges of the head's tiles (64 rows, 256 columns, 128 columns of the
    weight gradients, row chunks, unaligned widths) against float64 autograd.

    With u = 2^-24: a logit's fp32 sum errs by dz = 4 sqrt(D) u sum |terms| (Higham's sqrt(n) model with a
    factor of 4), the row's maximum over columns; a score by (2 dz + 16 u (1 + |lse|)) / ln V; G by |g| / ln V
    times (p (4 dz + 32 u (1 + |lse|)) + 16 u |p - [target]|); the gradients by that through the other factor and
    their own fp32 sums, then half an ulp of the output's type."""

    g = torch.Generator().manual_seed(batch * 1000003 + length * 1009 + width + vocab)
    prior = (0.5 * torch.randn((batch, length, width), generator=g)).to(dtype)
    weight = (2.0 / math.sqrt(width) * torch.randn((vocab, width), generator=g)).to(dtype)
    bias = (0.1 * torch.randn((vocab,), generator=g)).to(dtype)
    targets = torch.randint(0, vocab, (batch, length), generator=g)
    valid = torch.rand((batch, length), generator=g) < 0.85
    up = torch.randn((batch, length), generator=g).to(dtype)
    leaves = [t.to(device).requires_grad_() for t in (prior, weight, bias)]
    score = think.causal_surprise(*leaves, targets.to(device), valid.to(device))
    grads = torch.autograd.grad(score, leaves, up.to(device), retain_graph=True)
    p, w, b = (t.double().requires_grad_() for t in (prior, weight, bias))
    z = p @ w.t() + b
    lse = torch.logsumexp(z, -1)
    nll = lse - z.gather(-1, targets[..., None])[..., 0]
    want = torch.where(valid, 1 - torch.exp(-nll / math.log(vocab)), 0.0)
    want_grads = torch.autograd.grad(want, (p, w, b), up.double())
    u, ln = 2.0**-24, math.log(vocab)
    half_ulp = {torch.float32: u, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[dtype]
    rows = batch * length
    p, w, b, z, lse = p.detach().view(rows, width), w.detach(), b.detach(), z.detach().view(rows, vocab), lse.detach().view(rows, 1)
    dz = (4 * math.sqrt(width) * u * (p.abs() @ w.abs().t() + b.abs())).amax(-1, keepdim=True) + 16 * u * (1 + lse.abs())
    soft = torch.softmax(z, -1)
    hot = torch.nn.functional.one_hot(targets.view(-1), vocab).double()
    gnll = (up.double().view(-1, 1) * torch.exp(-nll.detach().view(-1, 1) / ln) / ln) * valid.view(-1, 1)
    G = gnll * (soft - hot)
    dG = gnll.abs() * (soft * 4 * dz + 2 * dz / ln * (soft - hot).abs() + 16 * u * (soft - hot).abs())
    tiny = 2.0**-25 if dtype == torch.float16 else 1e-37
    checks = [
        (score, want, (2 * dz / ln).view(batch, length) * valid),
        (grads[0], want_grads[0], (dG @ w.abs() + 4 * math.sqrt(vocab) * u * (G.abs() @ w.abs())).view(prior.shape)),
        (grads[1], want_grads[1], dG.t() @ p.abs() + 4 * math.sqrt(rows) * u * (G.abs().t() @ p.abs())),
        (grads[2], want_grads[2], dG.sum(0) + 4 * math.sqrt(rows) * u * G.abs().sum(0)),
    ]
    for got, ref, bound in checks:
        err = (got.detach().double().cpu() - ref.detach()).abs()
        bound = bound + half_ulp * ref.detach().abs() + tiny
        assert bool((err <= bound).all()), float((err / bound).max())
    with_graph = torch.autograd.grad(score, leaves, up.to(device), create_graph=True)
    for got, ref, bound in zip(with_graph, want_grads, (c[2] for c in checks[1:])):
        bound = bound + half_ulp * ref.abs() + tiny
        assert bool(((got.detach().double().cpu() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_causal_surprise_contains_what_is_not_finite(device, dtype):
    """A row of states with infinities or NaN leaves every other row's score and gradient unchanged, and so
    does an invalid row or (unchecked) a target out of range; the out-of-range row scores NaN with no gradient."""

    g = torch.Generator().manual_seed(5)
    prior = (0.5 * torch.randn((2, 70, 96), generator=g)).to(dtype).to(device)
    weight = (0.2 * torch.randn((300, 96), generator=g)).to(dtype).to(device)
    bias = torch.zeros((300,), dtype=dtype, device=device)
    targets = torch.randint(0, 300, (2, 70), generator=g).to(device)
    valid = torch.ones((2, 70), dtype=torch.bool, device=device)
    up = torch.ones((2, 70), dtype=dtype, device=device)
    def run(prior, targets):
        leaf = prior.clone().requires_grad_()
        score = think.causal_surprise(leaf, weight, bias, targets, valid, validate_targets=False)
        return score.detach(), torch.autograd.grad(score, leaf, up)[0]
    clean, clean_grad = run(prior, targets)
    bad, bad_targets = prior.clone(), targets.clone()
    bad[0, 3, 7], bad[1, 40, 0], bad[1, 69, 95] = float("inf"), float("nan"), -float("inf")
    bad_targets[0, 10], bad_targets[1, 1] = 300, -1
    score, grad = run(bad, bad_targets)
    touched = torch.zeros((2, 70), dtype=torch.bool, device=device)
    for i, j in ((0, 3), (1, 40), (1, 69), (0, 10), (1, 1)):
        touched[i, j] = True
    assert torch.equal(score[~touched], clean[~touched]) and torch.equal(grad[~touched], clean_grad[~touched])
    assert bool(torch.isnan(score[touched]).all())
    assert not grad[0, 10].any() and not grad[1, 1].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, vocab, width", [
    (70, 65, 40), (70, 129, 40), (70, 67, 40), (70, 257, 40), (9000, 257, 40), (9000, 300, 40), (70, 64, 40), (9000, 256, 40),
    (70, 257, 600),  # the width in chunks
    (70, 1100, 40),  # tiles joined by a wave
])
def test_causal_surprise_of_nan_and_masked_columns(device, dtype, rows, vocab, width):
    """A NaN in the last weight row or the last bias, in a last tile of one column, of several and among
    minus infinities, makes every valid row's score and gradient NaN, whatever the vocabulary's tiles; a
    last tile whose biases are all minus infinity leaves the scores of the other columns."""

    g = torch.Generator().manual_seed(rows + vocab)
    prior = (0.5 * torch.randn((1, rows, width), generator=g)).to(dtype).to(device)
    weight = (0.2 * torch.randn((vocab, width), generator=g)).to(dtype).to(device)
    bias = (0.1 * torch.randn((vocab,), generator=g)).to(dtype).to(device)
    tile = 64 if rows == 70 else 256
    last = (vocab - 1) // tile * tile  # the last tile's first column
    targets = torch.randint(0, max(last, 1), (1, rows), generator=g).to(device)
    valid = torch.rand((1, rows), generator=g).to(device) < 0.9
    def run(weight, bias):
        leaf = prior.clone().requires_grad_()
        score = think.causal_surprise(leaf, weight, bias, targets, valid)
        return score.detach(), torch.autograd.grad(score, leaf, torch.ones_like(score))[0]
    for where in ("weight", "bias", "bias among minus infinities"):
        w, b = weight.clone(), bias.clone()
        if where == "weight":
            w[vocab - 1, 7] = float("nan")
        else:
            if "among" in where:
                b[last:] = -float("inf")
            b[vocab - 1] = float("nan")
        score, grad = run(w, b)
        assert torch.isnan(score[valid]).all() and torch.isnan(grad[valid]).all(), where
        assert not score[~valid].any()
        if where != "weight":  # a NaN weight reaches an invalid row's gradient as 0 x NaN, as in any product
            assert not grad[~valid].any()
    if last:
        b = bias.clone()
        b[last:] = -float("inf")
        score, grad = run(weight, b)
        z = prior.double() @ weight.double()[:last].t() + bias.double()[:last]
        nll = torch.logsumexp(z, -1) - z.gather(-1, targets[..., None])[..., 0]
        want = torch.where(valid, 1 - torch.exp(-nll / math.log(vocab)), 0.0)
        # the fp32 logits of `width` terms below one and a few roundings, then the score's own type
        assert bool(((score.double() - want).abs() <= 2.0**-19 * width / 40 + (2.0**-8 if dtype == torch.bfloat16 else 0) * want).all())
        assert torch.isfinite(grad).all()


@pytest.mark.parametrize("kind, rows", [(k, r) for k in ("normal", "positive") for r in (1, 2, 7, 64, 1000, 4096)]
                         + [("low planes set", r) for r in (1, 2, 7)])
def test_fp32_products_of_the_head_round_either_way(device, kind, rows):
    """grad_weight = G^T prior in fp32 by itself: with the identity as weight grad_prior is G to the bit.

    In units of 2^-24 of the sum of a product's |terms|: every entry within 4 sqrt(rows) (Higham's sqrt(n)
    model with a factor of 4; one term comes out within 2.3), and the mean of the signed errors over the
    4096 entries within 0.6 for one or two terms (the matrix unit cuts off below its sum's last bit: 0.29
    and 0.18 measured) and 0.3 for more (0.13 and less), where planes cut off at the operand end 0.7 to 1.1
    below. "low planes set": operands a few steps below 1 + 2^-7, whose low planes are the largest; their
    terms are nearly one constant, so what is dropped (at most 1) and cut off (1/2) does not average out,
    bound 1.5 (cut-off planes end 6.9 below), and so would the steps' roundings of many terms, in any fp32
    sum, hence few rows."""

    g = torch.Generator().manual_seed(rows)
    width = 64
    if kind == "normal":
        prior = torch.randn((1, rows, width), generator=g)
    elif kind == "positive":
        prior = torch.rand((1, rows, width), generator=g) + 0.5
    else:
        prior = 1 + 2.0**-7 - 2.0**-23 * (1 + torch.randint(0, 64, (1, rows, width), generator=g))
    prior = prior.to(device).requires_grad_()
    weight = torch.eye(width, device=device).requires_grad_()
    targets = torch.zeros((1, rows), dtype=torch.int64, device=device)  # one target: a column of G has one sign
    score = think.causal_surprise(prior, weight, torch.zeros(width, device=device), targets,
                                  torch.ones((1, rows), dtype=torch.bool, device=device))
    grad, grad_weight = torch.autograd.grad(score, (prior, weight), torch.ones_like(score))
    G, p = grad.view(rows, width).double(), prior.detach().view(rows, width).double()
    units = (grad_weight.double() - G.t() @ p) / (2.0**-24 * (G.t().abs() @ p.abs()))
    assert float(units.abs().max()) <= 4 * math.sqrt(rows), float(units.abs().max())
    mean = float((units * torch.sign(G.t() @ p)).mean())
    assert abs(mean) <= (1.5 if kind == "low planes set" else 0.6 if rows <= 2 else 0.3), mean


@pytest.mark.parametrize("rows, width, vocab", [(1024, 128, 1000), (128, 300, 1000), (64, 1024, 256), (16, 512, 3000)])
def test_fp32_gradients_of_few_tiles_err_no_more_than_the_library(device, rows, width, vocab):
    """For few output tiles the library's fp32 products split K over workgroups, which leaves short sums.
    The head's gradients against float64 are no further off than the same formula in fp32 torch operations
    on those products (1.1: the spread of a norm over this many entries of independent roundings)."""

    g = torch.Generator().manual_seed(rows + width + vocab)
    prior = (0.5 * torch.randn((1, rows, width), generator=g)).to(device)
    weight = (2.0 / math.sqrt(width) * torch.randn((vocab, width), generator=g)).to(device)
    bias = (0.1 * torch.randn((vocab,), generator=g)).to(device)
    targets = torch.randint(0, vocab, (1, rows), generator=g).to(device)
    valid = torch.ones((1, rows), dtype=torch.bool, device=device)
    up = torch.randn((1, rows), generator=g).to(device)
    def composite(p, w, b):
        z = p.view(rows, width) @ w.t() + b
        nll = torch.logsumexp(z, -1) - z.gather(-1, targets.view(rows, 1))[:, 0]
        return (1 - torch.exp(-nll / math.log(vocab))).view(1, rows)
    def grads(front, dtype):
        leaves = [t.to(dtype).requires_grad_() for t in (prior, weight, bias)]
        return torch.autograd.grad(front(*leaves), leaves, up.to(dtype))
    want = grads(composite, torch.float64)
    library = grads(composite, torch.float32)
    got = grads(lambda p, w, b: think.causal_surprise(p, w, b, targets, valid), torch.float32)
    for have, lib, ref in zip(got[:2], library, want):
        err, bar = (float((x.double() - ref).norm() / ref.norm()) for x in (have, lib))
        print(f"{rows} {width} {vocab}: {err:.2e}, library {bar:.2e}", flush=True)
        assert err <= 1.1 * bar
