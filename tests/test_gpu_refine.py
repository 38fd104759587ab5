"""The refine memory of the herm ablation (model/network.py:359-384) on the
GPU against the float64 oracle.

* koemi_local_novelty against oracle.local_novelty (memory.py:354-361):
  carried rings with invalid slots, windows longer and shorter than the
  sliding window, bf16 keys read in place from a wider matrix, rows with no
  eligible slot (novelty 1), a query equal to a key (novelty 0). fp32 cosines
  against float64: within 2e-6.
* koemi_assoc_refine_scan_read (one window, one position) and the windowed
  entry against oracle.herm.associative_scan_read fed the refine terms
  (memory.py:257-268: capped refine decay, surprise x novelty write weight,
  clamped reconstruction error against the fast reads, masking): fp32
  tolerance 1e-4 relative + 1e-5 x max|result|, as for the fast memory; the
  windowed entry equals a window-by-window run within 1e-6.
* koemi_herm_refine_gate (network.py:714-721) against numpy in float64
  (fp32: 1e-5 relative), and its bf16-rounding form against the same
  arithmetic on bf16-rounded inputs.
* A two-layer fp32 stack under the herm ablation against oracle.herm over
  two windows and a decode step (the tolerances of test_gpu_herm.py), and
  the sequence-parallel prefill of a bf16 stack against its window-by-window
  prefill (the bf16 tolerances of the sequence tests).
"""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

import oracle
from koemi_amd import herm, memory
from oracle import herm as oherm

pytestmark = pytest.mark.gpu

PAD = herm.PAD_TOKEN_ID


@pytest.mark.parametrize("rows, cap, length, d, window, key_bf16", [
    (5, 4, 11, 16, 4, False), (3, 16, 40, 64, 16, True), (2, 16, 128, 1024, 16, True), (4, 3, 2, 20, 6, False),
    (3, 0, 9, 8, 3, False),
    # runs of four queries: one short of, equal to and past a run, widths at a register group's edge and past
    # the layout, no carried slots, a window longer than the row
    (3, 16, 7, 504, 16, True), (3, 16, 8, 512, 16, False), (4, 5, 17, 520, 9, True), (2, 0, 33, 1024, 40, True),
    (2, 16, 13, 1032, 16, True), (2, 3, 5, 12, 4, True), (5, 4, 4, 24, 3, True), (5, 4, 3, 24, 3, True),
])
def test_local_novelty_matches_the_oracle(device, rows, cap, length, d, window, key_bf16):
    rng = np.random.default_rng(rows * 100 + length)
    ck = rng.normal(size=(rows, cap, d)).astype(np.float32)
    cv = rng.random((rows, cap)) < 0.7
    wide = rng.normal(size=(rows, length, 3 * d)).astype(np.float32)
    if key_bf16:
        wide = torch.from_numpy(wide).to(torch.bfloat16).float().numpy()
    kv = rng.random((rows, length)) < 0.8
    q = rng.normal(size=(rows, length, d)).astype(np.float32)
    kv[0] = False  # row 0: window entries all invalid
    if cap:
        cv[0] = False  # ... and no carried slot: novelty 1 everywhere
    if length > 3:
        q[1, 3] = 2.5 * wide[1, 2, d:2 * d]  # a query parallel to an eligible key: novelty 0
        kv[1, 2] = True
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(device)
    wide_t = t(wide).to(torch.bfloat16) if key_bf16 else t(wide)
    got = memory.local_novelty(t(ck), t(cv), wide_t[..., d:2 * d], t(kv), t(q), window=window)
    want = oracle.local_novelty(ck, cv, wide[..., d:2 * d], kv, q, window)
    err = np.abs(got.cpu().numpy() - want)
    print(f"novelty rows={rows} L={length} d={d}: max_abs={err.max():.3e}", flush=True)
    assert np.all(err <= 2e-6)
    assert np.all(got.cpu().numpy()[0] == 1.0)
    if length > 3:
        assert abs(float(got[1, 3])) <= 2e-6


@pytest.mark.parametrize("d, key_bf16", [(1024, True), (520, False), (512, True), (24, False), (4, True)])
def test_local_novelty_of_either_layout_has_the_same_bits(device, d, key_bf16):
    """A row that fits the registers is walked for a run of queries at once, a wider one by a wave per
    query. Both add a lane's columns d, d + 64, .. in turn and then the lanes, so a row widened with zeros
    past the registers' 1024 columns has the same novelty to the bit."""
    rows, cap, length = 3, 16, 29
    g = torch.Generator().manual_seed(d)
    ck, keys, q = (torch.randn((rows, n, d), generator=g) for n in (cap, length, length))
    cv, kv = (torch.rand((rows, n), generator=g) < 0.8 for n in (cap, length))
    keys = keys.to(torch.bfloat16 if key_bf16 else torch.float32)
    wide = lambda t: torch.nn.functional.pad(t, (0, 1100 - d))
    on = lambda *ts: (t.to(device) for t in ts)
    got = memory.local_novelty(*on(ck, cv, keys, kv, q), window=16)
    want = memory.local_novelty(*on(wide(ck), cv, wide(keys), kv, wide(q)), window=16)
    assert torch.equal(got, want)


def _refine_terms(proj, surprise, valid, novelty, fast, d, m, rate):
    p64 = proj.astype(np.float64)
    value = np.tanh(p64[..., 2 * d:3 * d])
    features = oherm.softmax(p64[..., 3 * d:3 * d + m])
    qf = oherm.softmax(p64[..., 3 * d + m:3 * d + 2 * m])
    decay = oherm.MIN_DECAY + (oherm.MAX_DECAY - oherm.MIN_DECAY) * oherm.sigmoid(p64[..., 3 * d + 2 * m])
    decay = np.minimum(1.0 - (1.0 - decay) * rate, oherm.MAX_REFINE_DECAY)
    weight = (oherm.sigmoid(p64[..., 3 * d + 2 * m + 1]) * np.clip(surprise, 0, 1) * np.clip(novelty, 0, 1))
    error = np.clip(value - fast.astype(np.float64), -2.0, 2.0)
    return np.where(valid, decay, 1.0), error, features, np.where(valid, weight, 0.0), qf


@pytest.mark.parametrize("b, length, d, m, rate", [(2, 130, 100, 16, 0.0625), (3, 1, 64, 16, 0.25),
                                                    (2, 9, 36, 5, 0.0625), (1, 70, 128, 32, 1.0)])
def test_refine_scan_read_matches_the_oracle(device, b, length, d, m, rate):
    rng = np.random.default_rng(b * 1000 + length + 7)
    proj = rng.normal(size=(b, length, 3 * d + 2 * m + 2)).astype(np.float32)
    surprise = rng.random((b, length)).astype(np.float32)
    novelty = rng.random((b, length)).astype(np.float32)
    valid = rng.random((b, length)) < 0.8
    fast = (rng.normal(size=(b, length, d)) * 0.7).astype(np.float32)  # errors beyond +-2 get clamped
    fast[0, 0, :4] = 3.0
    basis = rng.normal(size=(b, d, m)).astype(np.float32)
    normalizer = rng.random((b, m)).astype(np.float32)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(device)
    read, nb, nn = herm.associative_refine_scan_read(t(proj), t(surprise), t(valid), t(novelty), t(fast), t(basis),
                                                     t(normalizer), width=d, features=m, rate=rate)
    decay, error, features, weight, qf = _refine_terms(proj, surprise, valid, novelty, fast, d, m, rate)
    want = oherm.associative_scan_read(basis.astype(np.float64), normalizer.astype(np.float64), decay, error,
                                       features, weight, qf)
    for got, ref, name in zip((read, nb, nn), want, ("read", "basis", "normalizer")):
        err = np.abs(got.cpu().numpy().astype(np.float64) - ref)
        scale = float(np.abs(ref).max())
        print(f"refine {name} b={b} L={length} d={d} m={m}: max_abs={err.max():.3e} scale={scale:.3e}", flush=True)
        assert np.all(err <= 1e-4 * np.abs(ref) + 1e-5 * scale), name


def test_windowed_refine_equals_window_by_window(device):
    """The windowed entry (every window's terms, the carried refine state,
    every window's reads) against the one-window entry run window by window,
    with bf16 projections and bf16 fast reads read in place from a wider
    matrix."""
    b, windows, window, d, m = 2, 3, 64, 96, 16
    length = windows * window
    g = torch.Generator(device=device).manual_seed(5)
    proj = torch.randn((b, length, 3 * d + 2 * m + 4), generator=g, device=device).to(torch.bfloat16)
    surprise = torch.rand((b, length), generator=g, device=device)
    novelty = torch.rand((b, length), generator=g, device=device)
    valid = torch.rand((b, length), generator=g, device=device) < 0.85
    fast_wide = torch.randn((b, length, 2 * d), generator=g, device=device).to(torch.bfloat16)
    fast = fast_wide[..., d:]
    basis = torch.randn((b, d, m), generator=g, device=device) * 0.1
    norm = torch.rand((b, m), generator=g, device=device)
    read, nb, nn = herm.associative_refine_scan_read(proj, surprise, valid, novelty, fast, basis, norm, width=d,
                                                     features=m, rate=0.0625, window=window)
    cb, cn = basis, norm
    for w in range(windows):
        sl = slice(w * window, (w + 1) * window)
        r, cb, cn = herm.associative_refine_scan_read(proj[:, sl].contiguous(), surprise[:, sl], valid[:, sl],
                                                      novelty[:, sl], fast[:, sl].contiguous(), cb, cn, width=d,
                                                      features=m,
                                                      rate=0.0625)
        torch.testing.assert_close(read[:, sl], r, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(nb, cb, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(nn, cn, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("low", [False, True])
def test_refine_gate_matches_numpy(device, low):
    rows, d = 300, 64
    g = torch.Generator().manual_seed(9)
    ws, fast, refine = (torch.randn((1, rows, d), generator=g) for _ in range(3))
    local = torch.randn((1, rows, d), generator=g)
    w = torch.randn((4 * d,), generator=g) * 0.05
    bias = torch.randn((1,), generator=g)
    dt = torch.bfloat16 if low else torch.float32
    p = {"refine_gate_w": w.to(dt).to(device), "refine_gate_b": bias.to(device)}
    out = torch.empty((1, rows, 2 * d), device=device, dtype=dt)
    got = herm._refine_gate(p, ws.to(device), fast.to(device), refine.to(device), local.to(dt).to(device),
                            out[..., d:], torch.bfloat16 if low else None)
    assert got.data_ptr() == out[..., d:].data_ptr()
    r = (lambda x: x.to(torch.bfloat16).double()) if low else (lambda x: x.double())
    x = torch.cat([r(ws), r(fast), r(refine), r(local)], dim=-1)
    pre = x @ r(w) + bias.double()
    if low:
        pre = pre.float().to(torch.bfloat16).double()
    want = fast.double() + torch.sigmoid(pre)[..., None] * refine.double()
    if low:
        want = want.float().to(torch.bfloat16).double()
    err = (got.double().cpu() - want).abs()
    # bf16: the output's rounding, plus the pre-activation rounded to the
    # neighbouring bf16 value (|d sigmoid| <= 1/4 of one bf16 ulp of pre) times |refine|
    bound = ((2.0 ** -8 * want.abs() + 0.25 * 2.0 ** -7 * pre.abs()[..., None] * refine.double().abs() + 1e-6)
             if low else 1e-5 * want.abs() + 1e-6)
    print(f"refine gate low={low}: max_abs={err.max().item():.3e}", flush=True)
    assert bool((err <= bound).all())


def _settings(**kw):
    base = dict(width=32, memory_features=4, local_memory_size=4, salience_memory_size=3, expert_count=4, top_k=2,
                layers=2, scan_chunk=6, linear_dtype=torch.float32, ablation="herm", salience_threshold=0.5)
    base.update(kw)
    return herm.HermSettings(**base)


def test_refine_stack_prefill_and_decode_match_the_oracle(device):
    """Two layers under the herm ablation, two windows of six then one decode
    step, fp32 projections, against oracle.herm; the head is scaled so that
    admissions (and so novelty-weighted refine writes of surprising tokens)
    happen; tolerances as test_gpu_herm.py (1e-4 relative + 1e-4 x scale)."""
    b, length = 2, 12
    settings = _settings()
    params = herm.init_stack(settings, 17)
    for p in params:
        p["head_w"] *= 8.0
    params_np = [{k: v.double().numpy() for k, v in p.items()} for p in params]
    rng = np.random.default_rng(4)
    ids = rng.integers(0, 256, (b, length))
    ids[1, 2] = PAD
    cfg = settings.oracle_config()
    # a threshold clear of every oracle score
    for tau in (0.5, 0.55, 0.6, 0.45, 0.65, 0.4, 0.7):
        cfg["salience_threshold"] = tau
        _, _, scores, _ = oherm.prefill(params_np, [oherm.initial_state(b, cfg) for _ in params_np], ids, cfg,
                                        settings.scan_chunk, return_layers=True)
        flat = np.concatenate([s[ids != PAD] for s in scores])
        if np.abs(flat - tau).min() >= 2e-3 and (flat > tau).any():
            break
    else:
        pytest.skip("no threshold with a 2e-3 margin for this seed")
    settings = dataclasses.replace(settings, salience_threshold=tau)
    prepared = herm.prepare_stack(params, settings, device)
    states = herm.initial_states(settings, b, device)
    assert "refine_basis" in states[0]
    logits, states = herm.prefill(prepared, settings, torch.from_numpy(ids).to(device), states)
    want_logits, want_states = oherm.prefill(params_np, [oherm.initial_state(b, cfg) for _ in params_np], ids, cfg,
                                             settings.scan_chunk)
    scale = float(np.abs(want_logits).max())

    def close(got, want, sc, what):
        err = np.abs(np.asarray(got, np.float64) - want)
        print(f"{what}: max_abs={err.max():.3e} scale={sc:.3e}", flush=True)
        assert np.all(err <= 1e-4 * np.abs(want) + 1e-4 * sc), what

    close(logits.cpu().numpy(), want_logits, scale, "refine prefill logits")
    for layer, (got, want) in enumerate(zip(states, want_states)):
        for key in ("working", "basis", "refine_basis", "refine_normalizer", "salient_keys"):
            close(got[key].cpu().numpy(), want[key], float(np.abs(want[key]).max()) + 1e-30, f"layer {layer} {key}")
        assert np.abs(want["refine_basis"]).max() > 0
    next_ids = torch.from_numpy(ids[:, -1:]).to(device)
    got_logits, states = herm.stack_window(prepared, settings, next_ids, states)
    want_step, want_states, _ = oherm.stack_window(params_np, want_states, ids[:, -1:], cfg)
    close(got_logits.cpu().numpy(), want_step, scale, "refine decode step logits")
    for layer, (got, want) in enumerate(zip(states, want_states)):
        for key in ("refine_basis", "refine_normalizer"):
            close(got[key].cpu().numpy(), want[key], float(np.abs(want[key]).max()) + 1e-30,
                  f"decode layer {layer} {key}")


def test_refine_sequence_prefill_matches_the_window_prefill(device):
    """A bf16 stack under the herm ablation (width 256, 256-position
    sequences, so the fused gate kernel runs): the sequence-parallel prefill
    against the window-by-window prefill of the same stack, logits within the
    bf16 tolerance of the sequence tests (relative Frobenius 1e-2), refine
    states within 1e-2, ring bits exact."""
    settings = herm.HermSettings(width=256, memory_features=16, layers=2, scan_chunk=128, expert_count=4, top_k=2,
                                 ablation="herm")
    b, length = 2, 256
    params = herm.prepare_stack(herm.init_stack(settings, 23, device), settings, device)
    ids = torch.randint(0, 256, (b, length), generator=torch.Generator().manual_seed(3)).to(device)
    want, want_states = herm.prefill(params, settings, ids, herm.initial_states(settings, b, device))
    got, got_states = herm.stack_sequence(params, settings, ids, herm.initial_states(settings, b, device))
    torch.cuda.synchronize()
    rel = float((got - want).norm() / want.norm())
    print(f"refine sequence vs window logits rel {rel:.3e}", flush=True)
    assert rel <= 1e-2
    for layer, (g, w) in enumerate(zip(got_states, want_states)):
        for key in ("refine_basis", "refine_normalizer", "basis"):
            r = float((g[key] - w[key]).norm() / (w[key].norm() + 1e-30))
            print(f"layer {layer} {key}: rel {r:.3e}", flush=True)
            assert r <= 1e-2, f"layer {layer} {key}"
        for key in ("local_valid", "salient_valid", "last_token"):
            assert torch.equal(g[key], w[key]), f"layer {layer} {key}"
