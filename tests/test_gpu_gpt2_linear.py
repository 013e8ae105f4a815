"""The linear layers' products (dfgpt2_linear_*) at the ends of their tiles and past them: rows, columns
and contractions of one value, one short of a tile, one past it, contractions no multiple of a load, and
the sizes at which the tile changes.

Against plain PyTorch in float64. Rounding a value in [1, 2) to bf16 (7 fraction bits) leaves at most half
of 2^-7, so 2^-8 of a value goes to the second term and at most 2^-16 of it is lost; the product of the two
second terms, at most 2^-16 of the product, is left out. 3 * 2^-16 = 4.6e-5 of the sum of the products'
magnitudes bounds a value, to which an fp32 sum of n terms adds at most 2^-23 n. The 2-norm of random data
is held to 6e-6 (measured: 4.4e-6)."""
import pytest

from dfattn import ops

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (1, 5, 3), (3, 2, 65), (63, 31, 33), (64, 64, 64), (65, 33, 97), (100, 36, 50), (127, 130, 95),
         (129, 257, 193), (257, 45, 385), (200, 768, 2304), (1000, 768, 3072), (1025, 200, 1537), (2049, 130, 1601)]


def check(name, got, want, bound, rel=6e-6):
    err = (got.double() - want).abs()
    assert bool((err <= bound).all()), f"{name}: {float((err / bound.clamp_min(1e-300)).max()):.2f} of the bound"
    # The norm is a statistic of many values; a few are held to their bound alone.
    if want.numel() >= 256:
        assert float(err.norm() / want.norm()) <= rel, f"{name}: {float(err.norm() / want.norm()):.1e}"


@pytest.mark.parametrize("rows,k,n", SIZES)
def test_linear_products(device, rows, k, n):
    import torch

    print(f"[gpu-linear] {rows} rows, {k} in, {n} out", flush=True)
    torch.manual_seed(rows * 7 + k * 3 + n)
    F = torch.nn.functional
    x, w, b, dy, h = (torch.randn(*s, device=device) for s in ((rows, k), (n, k), (n,), (rows, n), (rows, k)))
    nan = float("nan")
    y, a = torch.full((2, rows, n), nan, device=device).unbind(0)
    plain, dx, dxg = (torch.full(s, nan, device=device) for s in ((rows, n), (rows, k), (rows, k)))
    dw = torch.full((n, k), nan, device=device)
    ops.linear_forward_into(x, w, b, y, a)
    ops.linear_forward_into(x, w, b, plain)
    ops.linear_backward_input_into(dy, w, dx)
    ops.linear_backward_input_into(dy, w, dxg, h)
    ops.linear_backward_weight_into(dy, x, dw)
    assert torch.equal(y, plain)
    # GELU and its derivative are the elementwise kernels' (tanhf of the same argument).
    assert torch.equal(a, ops.gelu_forward(y))
    assert torch.equal(dxg, ops.gelu_backward(dx, h))
    x, w, b, dy = (t.double() for t in (x, w, b, dy))

    def bound(p, q, terms, extra=0.0):
        return (4.6e-5 + 1.2e-7 * (terms + 3)) * (p.abs() @ q.abs()) + extra

    want = x @ w.t()
    check("y", y, want + b, bound(x, w.t(), k, 1.2e-7 * (want.abs() + b.abs())))
    check("dx", dx, dy @ w, bound(dy, w, n))
    check("dw", dw, dy.t() @ x, bound(dy.t(), x, rows))


def test_rows_at_any_4_byte_address(device):
    import torch

    print("[gpu-linear] operands one float past a 16-byte boundary", flush=True)
    rows, k, n = 130, 68, 97
    flat = [torch.randn(m + 1, device=device) for m in (rows * k, n * k, n, rows * n)]
    x, w, b, dy = (f[1:].view(s) for f, s in zip(flat, ((rows, k), (n, k), (n,), (rows, n))))
    y, dw = torch.empty(rows, n, device=device), torch.empty(n, k, device=device)
    ops.linear_forward_into(x, w, b, y)
    ops.linear_backward_weight_into(dy, x, dw)
    check("y", y, (x.double() @ w.double().t() + b.double()), 6.2e-5 * (x.double().abs() @ w.double().abs().t() + b.abs()))
    check("dw", dw, dy.double().t() @ x.double(), 6.2e-5 * (dy.double().abs().t() @ x.double().abs()))


def test_weight_gradient_of_no_rows_is_zero(device):
    import torch

    print("[gpu-linear] no rows", flush=True)
    dw = torch.full((70, 33), float("nan"), device=device)
    ops.linear_backward_weight_into(torch.empty(0, 70, device=device), torch.empty(0, 33, device=device), dw)
    assert bool((dw == 0).all())


def test_step_with_own_and_library_products(device):
    """A GPT-2 step's gradients with dfgpt2_linear_* at the fast sites against hipBLASLt's exact products:
    the gradients differ by the fast path's error carried through two layers."""
    import torch

    from dfattn.gpt2_step import StaticGPT2, synthetic_batch

    cfg = dict(vocab_size=500, d_model=96, n_heads=3, n_layers=2, d_ff=384, seq_len=130, seed=4)
    tokens, targets = synthetic_batch(500, 130, 5, device)
    print("[gpu-linear] GPT-2 step: own and exact products", flush=True)
    own, exact = StaticGPT2(**cfg), StaticGPT2(**cfg, fast_gemm=False)
    assert own._engine._own_gemms() and not exact._engine._own_gemms()
    assert abs(float(own.step(tokens, targets)) - float(exact.step(tokens, targets))) < 1e-4
    g, ref = own.opt.arena.g, exact.opt.arena.g
    assert float((g - ref).norm() / ref.norm()) < 1e-4


def test_step_with_library_products_at_the_fast_sites(device):
    """The same step with the fast sites on hipBLASLt's fast path (first MLP bias and GELU in a kernel of
    their own, GELU's derivative after the product): the same values to the fast paths' error."""
    import torch

    from dfattn.gpt2_step import StaticGPT2, synthetic_batch

    cfg = dict(vocab_size=500, d_model=96, n_heads=3, n_layers=2, d_ff=384, seq_len=130, seed=4)
    tokens, targets = synthetic_batch(500, 130, 5, device)
    print("[gpu-linear] GPT-2 step: own and library fast products", flush=True)
    own, library = StaticGPT2(**cfg), StaticGPT2(**cfg)
    library._engine.library_products = True
    assert own._engine._own_gemms() and not library._engine._own_gemms()
    assert abs(float(own.step(tokens, targets)) - float(library.step(tokens, targets))) < 1e-4
    g, ref = own.opt.arena.g, library.opt.arena.g
    assert float((g - ref).norm() / ref.norm()) < 1e-4
