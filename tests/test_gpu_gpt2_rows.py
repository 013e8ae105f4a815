"""The GPT-2 step's row kernels where their variants meet: LayerNorm rows of up to 8 float4 a lane and
just past them, several rows per wave in the fused backward, the bias gradient's row blocks, and the
cross-entropy at the ends of its register variants, with rows that start at any 4-byte address.

Against plain PyTorch in float64. Everything is fp32: sums over n terms of either sign carry a relative
error of about sqrt(n) u (u = 6e-8) in 2-norm, at most 6e-6 for the 8200 rows here; single values are
held to 1e-4 of the largest."""
import pytest

from dfattn import ops

pytestmark = pytest.mark.gpu


def check(name, got, want, rel=6e-6):
    got, want = got.detach(), want.detach()
    got, want = got.double(), want.double()
    err = float((got - want).norm() / want.norm().clamp_min(1e-30))
    worst = float((got - want).abs().max() / want.abs().max().clamp_min(1e-30))
    assert err <= rel and worst <= 1e-4, f"{name}: rel {err:.1e}, max {worst:.1e}"


WIDE_ROWS = [(1, 1028), (5, 1536), (7, 1600), (2051, 2048), (9, 2052), (6, 1030)]


@pytest.mark.parametrize("rows,features,workspace", [(*s, True) for s in WIDE_ROWS + [(4097, 768), (8200, 1024)]] +
                         [(*s, False) for s in WIDE_ROWS])
def test_layer_norm_widths(device, rows, features, workspace):
    """With and without a workspace: only rows of at most 1024 features need one."""
    import torch

    print(f"[gpu-rows] LayerNorm {rows} x {features} workspace={workspace}", flush=True)
    torch.manual_seed(rows + features)
    x, y, dy, res = (torch.randn(rows, features, device=device) for _ in range(4))
    gamma, beta = torch.randn(features, device=device), torch.randn(features, device=device)
    total, out, dx = (torch.empty_like(x) for _ in range(3))
    stats = torch.empty(2, rows, device=device)
    dg, db, dbias = (torch.empty(features, device=device) for _ in range(3))
    ops.add_layer_norm_forward_into(x, y, gamma, beta, total, out, stats)
    ws = torch.empty(ops.layer_norm_backward_fused_workspace_bytes(rows, features) // 4 if workspace else 1, device=device)
    ops.layer_norm_backward_fused_into(dy, total, gamma, stats, res, dx, dg, db, dbias, ws)
    dg2, db2, dx2 = (torch.empty_like(t) for t in (dg, db, dx))
    ops.layer_norm_backward_residual_into(dy, total, gamma, stats, res, dx2, dg2, db2)
    t64, g64, b64 = ((x + y).double().requires_grad_(True), gamma.double().requires_grad_(True),
                     beta.double().requires_grad_(True))
    o64 = torch.nn.functional.layer_norm(t64, (features,), g64, b64, 1e-5)
    gt, gg, gb = torch.autograd.grad(o64, (t64, g64, b64), dy.double())
    want = gt + res.double()
    check("sum", total, t64)
    check("out", out, o64)
    for name, got, w in (("dx", dx, want), ("dgamma", dg, gg), ("dbeta", db, gb), ("dbias", dbias, want.sum(0)),
                         ("dx apart", dx2, want), ("dgamma apart", dg2, gg), ("dbeta apart", db2, gb)):
        check(name, got, w)


@pytest.mark.parametrize("rows", [1, 255, 4095, 4096, 4097, 8192])
def test_bias_gradient_row_blocks(device, rows):
    import torch

    print(f"[gpu-rows] bias gradient rows={rows}", flush=True)
    g = torch.randn(rows, 36, device=device)
    check("bias", ops.bias_grad(g), g.double().sum(0))


def test_bias_gradient_of_the_most_rows(device):
    """2^31 - 1 rows of four ones: a row slot's index ends next to 2^31. Each of the 256 slots counts 2^23
    rows (one a row less), exactly; their total rounds to 2^31."""
    import torch

    rows = 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < rows * 16 + (4 << 30):
        pytest.skip("needs 36 GiB of free device memory")
    print(f"[gpu-rows] bias gradient rows={rows}", flush=True)
    g = torch.ones(rows, 4, device=device)
    got = ops.bias_grad(g).tolist()
    del g
    torch.cuda.empty_cache()
    assert got == [2.0 ** 31] * 4


@pytest.mark.parametrize("cols", [1, 3, 511, 512, 513, 2047, 2048, 2049, 4096, 4097, 8192, 8195, 16384, 16385, 30720, 30721, 50257, 51200, 51201])
def test_cross_entropy_lengths(device, cols):
    """One row all -1e30 but its target, and one whose largest logit comes last."""
    import torch

    print(f"[gpu-rows] cross-entropy cols={cols}", flush=True)
    torch.manual_seed(cols)
    rows = 5
    logits = torch.randn(rows, cols, device=device) * 3
    targets = torch.randint(0, cols, (rows,), device=device)
    logits[1] = -1e30
    logits[1, targets[1]] = 2.0
    logits[2, cols - 1] = 60.0
    want = torch.softmax(logits.double(), 1)
    row_loss = -torch.log(want[torch.arange(rows), targets].clamp_min(1e-12)) / 7
    want[torch.arange(rows), targets] -= 1
    guard = torch.full((rows * cols + 8,), 7.0, device=device)
    grad = guard[4:4 + rows * cols].view(rows, cols)
    loss = torch.empty(rows, device=device)
    ops.logit_ce_chunk(logits, targets.int(), grad, loss, 7)
    check("grad", grad, want / 7)
    check("loss", loss, row_loss)
    assert (guard[:4] == 7).all() and (guard[4 + rows * cols:] == 7).all()
    ops.logit_ce_chunk(logits, targets.int(), logits, loss, 7)  # in place
    assert torch.equal(logits, grad)


@pytest.mark.parametrize("cols", [16, 2048, 3000, 5000, 8192, 16384, 30000, 50257])
def test_cross_entropy_masked_logits(device, cols):
    """Logits of -inf (masked) in rows that lie far below and above zero: all the values that one thread
    holds (four adjacent ones, again 2048 further), and all the first ones of every thread. A masked
    logit's gradient is zero."""
    import torch

    print(f"[gpu-rows] cross-entropy masked cols={cols}", flush=True)
    torch.manual_seed(cols)
    rows, at = 5, torch.arange(cols, device=device)
    logits = torch.randn(rows, cols, device=device)
    logits += torch.tensor([-100.0, -300.0, 200.0, -1000.0, -100.0], device=device)[:, None]
    one_thread = at // 4 % 512 == 1
    first = at < min(10240, cols // 2)
    for i, mask in enumerate((one_thread, first, first, at >= 0, one_thread | first)):
        logits[i, mask] = float("-inf")
    targets = torch.tensor([0, cols - 1, cols - 1, cols // 3, cols - 1], device=device)
    logits[torch.arange(rows), targets] = torch.tensor([-101.0, -299.0, 201.0, -1000.0, -100.5], device=device)
    want = torch.softmax(logits.double(), 1)
    row_loss = -torch.log(want[torch.arange(rows), targets].clamp_min(1e-12)) / 7
    masked = logits == float("-inf")
    want[torch.arange(rows), targets] -= 1
    grad, loss = torch.empty_like(logits), torch.empty(rows, device=device)
    ops.logit_ce_chunk(logits, targets.int(), grad, loss, 7)
    assert bool((grad[masked] == 0).all())
    for i in (0, 1, 2, 4):
        check(f"grad {i}", grad[i], want[i] / 7)
    assert bool((grad[3] == 0).all())  # one value left: probability 1
    assert float((loss - row_loss).abs().max()) <= 1e-5
    ops.logit_ce_chunk(logits, targets.int(), logits, loss, 7)  # in place
    assert torch.equal(logits, grad)


@pytest.mark.parametrize("cols", [16, 5000, 16384, 50257])
def test_cross_entropy_nan_logits(device, cols):
    """A NaN among the logits makes its row's gradient NaN, also where one thread holds nothing else, and
    no other row's."""
    import torch

    print(f"[gpu-rows] cross-entropy NaN cols={cols}", flush=True)
    torch.manual_seed(cols)
    logits, at = torch.randn(4, cols, device=device), torch.arange(cols, device=device)
    logits[0, cols // 2] = float("nan")
    logits[1, at // 4 % 512 == 1] = float("nan")
    logits[2, at // 4 % 512 == 1] = float("-inf")
    logits[2, 5] = float("nan")
    grad, loss = torch.empty_like(logits), torch.empty(4, device=device)
    ops.logit_ce_chunk(logits, torch.zeros(4, dtype=torch.int32, device=device), grad, loss, 4)
    assert bool(grad[:3].isnan().all()) and bool(grad[3].isfinite().all())
