"""The fp32 attention kernels (every d_head but the fp16 path's 64) at the edges of their 16-row tiles
and 16-value blocks, against the oracle's float64 twin.

Tolerance: everything is fp32 (unit roundoff u = 2^-24). The longest sums here have 300 terms of one
sign at most, so a relative error of sqrt(300) u = 1.0e-6 per reduction; a gradient passes through
three (scores, Delta, the final sum), and dS = P (dP - Delta) cancels to about a third of its terms:
1e-5 in rel-L2 covers it, and 2e-4 * max(1, max|want|) any single value (the reference's own bar)."""
import numpy as np
import pytest

import dfattn
import oracle as O
from conftest import oracle_threads, rel_l2

pytestmark = pytest.mark.gpu


def run(x, n_heads, scale, causal, device, shift=0):
    """O, lse, dQ, dK, dV; shift: every tensor starts `shift` floats past a 16-byte boundary."""
    import torch

    def dev(a):
        buf = torch.empty(a.size + shift, dtype=torch.float32, device=device)
        t = buf[shift:].view(a.shape)
        t.copy_(torch.from_numpy(a))
        return t

    q, k, v, g = (dev(x[n]) for n in ("q", "k", "v", "do"))
    out = dev(np.zeros_like(x["q"]))
    grads = [dev(np.full_like(x["q"], np.nan)) for _ in range(3)]
    o, lse = dfattn.attention_forward(q, k, v, n_heads, scale, causal, out=out)
    dfattn.attention_backward(q, k, v, o, g, lse, n_heads, scale, causal, *grads)
    torch.cuda.synchronize()
    return {n: t.cpu().numpy() for n, t in zip(("o", "lse", "dq", "dk", "dv"), [o, lse] + grads)}


def check(x, n_heads, scale, causal, got):
    t = oracle_threads()
    o, lse = O.mha_forward(x["q"], x["k"], x["v"], n_heads, scale, causal, threads=t)
    want = dict(zip(("o", "lse", "dq", "dk", "dv"), (o, lse, *O.backward(x["q"], x["k"], x["v"], x["do"], n_heads,
                                                                         scale, causal, threads=t))))
    for name, w in want.items():
        top = 2e-4 * max(1.0, float(np.max(np.abs(w))))
        worst = float(np.max(np.abs(got[name] - w)))
        assert worst <= top, f"{name}: max-abs {worst:.2e} (bar {top:.1e})"
        # One key or row leaves dQ and dK exactly zero in the oracle.
        if np.linalg.norm(w) > 1e-3:
            assert rel_l2(got[name], w) <= 1e-5, f"{name}: rel-L2 {rel_l2(got[name], w):.2e}"


@pytest.mark.parametrize("d_head", [1, 5, 16, 31, 48, 64, 72, 80, 100, 127, 128])
@pytest.mark.parametrize("seq,causal", [(1, True), (15, False), (16, True), (17, True), (33, False), (127, True),
                                        (300, True), (300, False)])
def test_tile_edges(device, d_head, seq, causal):
    print(f"[gpu-fp32] D={d_head} S={seq} causal={causal}", flush=True)
    shift = 1 if d_head == 64 else 0  # d_head 64 comes here when a tensor is only 4-byte aligned
    x = O.seeded_inputs(seq, 3, d_head, 40 + d_head + seq)
    check(x, 3, d_head ** -0.5, causal, run(x, 3, d_head ** -0.5, causal, device, shift))


@pytest.mark.parametrize("scale", [0.5, -0.25])
def test_scores_that_move_the_reference_point(device, scale):
    """Scores that climb (or fall) by about 60 over the keys, and a negative scale."""
    print(f"[gpu-fp32] staircase scale={scale}", flush=True)
    x = O.seeded_inputs(200, 2, 32, 77)
    x["q"][:, 0] = x["q"][:, 32] = 8.0
    x["k"][:, 0] = x["k"][:, 32] = np.arange(200, dtype=np.float32) * 0.08 * np.sign(scale)
    check(x, 2, scale, True, run(x, 2, scale, True, device))


@pytest.mark.parametrize("d_head", [5, 64, 80, 128])
@pytest.mark.parametrize("seq,causal", [(1, True), (40, True), (33, False), (48, False)])
def test_scale_zero(device, d_head, seq, causal):
    """Scale 0 weighs every visible key alike (and gives dQ and dK of zero); hidden keys, and those past a
    ragged last tile, stay hidden."""
    print(f"[gpu-fp32] scale 0 D={d_head} S={seq} causal={causal}", flush=True)
    x = O.seeded_inputs(seq, 2, d_head, 60 + d_head)
    got = run(x, 2, 0.0, causal, device, 1 if d_head == 64 else 0)
    assert all(np.isfinite(t).all() for t in got.values())
    check(x, 2, 0.0, causal, got)


def test_lse_error_against_float64(device):
    """The mean rel-L2 error of lse over these (seeded) inputs: 4.42e-8 with one rounding of the reference
    point's and the sum's logarithms together, 4.88e-8 with the log2 domain's sum times ln 2; the row-wise
    kernel these replaced had 4.68e-8."""
    import torch

    print("[gpu-fp32] lse against float64", flush=True)
    errors = []
    for d_head in (16, 32, 48, 64, 100, 128):
        for seq in (64, 200, 512):
            x, scale = O.seeded_inputs(seq, 5, d_head, d_head + seq), float(np.float32(d_head ** -0.5))
            got = run(x, 5, scale, True, device, 1 if d_head == 64 else 0)["lse"]
            q, k = (torch.from_numpy(x[n]).double().view(seq, 5, d_head).transpose(0, 1).contiguous() for n in "qk")
            scores = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
            hidden = torch.ones(seq, seq, dtype=torch.bool).triu(1)
            errors.append(rel_l2(got, torch.logsumexp(scores.masked_fill(hidden, -np.inf), 2).numpy()))
    assert np.mean(errors) <= 4.65e-8, errors


@pytest.mark.parametrize("d_head", [40, 128])
def test_nonfinite_rows_stay_behind_the_mask(device, d_head):
    """Row 40 of V (then of dO) holds an infinity and a NaN: under causal masking no query before row
    40 (no key after it) may see them, also those of row 40's own tile."""
    print(f"[gpu-fp32] non-finite rows D={d_head}", flush=True)
    x = O.seeded_inputs(60, 2, d_head, 90)
    scale = d_head ** -0.5
    clean = run(x, 2, scale, True, device)

    def same(a, b):
        # The sums run on another unit in that tile: at most 60 terms of order one, 60 u = 4e-6.
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-5)

    bad = {n: a.copy() for n, a in x.items()}
    bad["v"][40, 0], bad["v"][40, d_head] = np.inf, np.nan
    got = run(bad, 2, scale, True, device)
    same(got["o"][:40], clean["o"][:40])
    assert not np.isfinite(got["o"][40:, 0]).any() and np.isnan(got["o"][40:, d_head]).all()
    same(got["o"][:, 1:d_head], clean["o"][:, 1:d_head])
    bad = {n: a.copy() for n, a in x.items()}
    bad["do"][40, 0] = bad["do"][40, d_head] = np.inf
    got = run(bad, 2, scale, True, device)
    same(got["dv"][41:], clean["dv"][41:])
    same(got["dk"][41:], clean["dk"][41:])
    same(got["dq"][:40], clean["dq"][:40])
    assert not np.isfinite(got["dv"][:41, 0]).any()
    # dQ_i sums over keys up to i only: an infinite K row after them must not reach it.
    bad = {n: a.copy() for n, a in x.items()}
    bad["k"][40, 0] = bad["k"][40, d_head] = np.inf
    got = run(bad, 2, scale, True, device)
    same(got["o"][:40], clean["o"][:40])
    same(got["dq"][:40], clean["dq"][:40])
