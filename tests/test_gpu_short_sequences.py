"""d_head 64: the kernels for short sequences (32 rows a workgroup, tiles split among its waves) at the
edges of their tiles, and the staged kernels at ragged lengths of shapes that go to them. Both through
the one-call pair and the training pair, at the bar of the fp16-operand shapes."""
import pytest

import oracle as O
from test_gpu_parity import compare, oracle_fwd_bwd, run_fwd_bwd, run_training_pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("n_heads,seq", [(1, 1), (2, 31), (2, 32), (2, 33), (3, 63), (3, 64), (2, 95), (2, 97), (3, 128),
                                         (3, 129), (2, 161), (12, 545), (12, 1409)])
def test_short(device, n_heads, seq, causal):
    say(f"short H={n_heads} S={seq} causal={causal}")
    x = O.seeded_inputs(seq, n_heads, 64, 600 + seq)
    want = oracle_fwd_bwd(x, n_heads, 0.125, causal)
    compare("one call", run_fwd_bwd(x, n_heads, 0.125, causal, device), want, scaled=True)
    compare("pair", run_training_pair(x, n_heads, 0.125, causal, device), want, scaled=True)


@pytest.mark.parametrize("n_heads,seq,causal", [(16, 2047, True), (16, 2049, True), (16, 2175, True), (16, 1537, False),
                                                (14, 1537, True), (4, 2049, False)])
def test_staged(device, n_heads, seq, causal):
    say(f"staged H={n_heads} S={seq} causal={causal}")
    x = O.seeded_inputs(seq, n_heads, 64, 700 + seq)
    want = oracle_fwd_bwd(x, n_heads, 0.125, causal)
    compare("one call", run_fwd_bwd(x, n_heads, 0.125, causal, device), want, scaled=True)
    compare("pair", run_training_pair(x, n_heads, 0.125, causal, device), want, scaled=True)
