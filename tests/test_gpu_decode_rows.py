"""Decode with every row layout: caches of up to three keys (one wave per head); 8, 16 or 32 lanes per
cache row, rows that fill their lanes or not, and rows that are not aligned for 4-value loads; groups of
64 and 32 keys that end anywhere. Against the oracle at the decode tests' fp32 bar."""
import numpy as np
import pytest

import dfattn
import oracle as O
from test_gpu_decode import cache, close, dev_any, host, paged_pool, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_head", [1, 4, 20, 31, 33, 48, 62, 68, 80, 127, 128])
@pytest.mark.parametrize("length,page,bf16", [(1, 0, False), (2, 7, True), (3, 2, False), (4, 0, True), (31, 16, True), (65, 0, True), (257, 7, False),
                                              (1500, 64, True), (1537, 0, False)])
def test_rows(device, d_head, length, page, bf16):
    print(f"[gpu-decode-rows] D={d_head} L={length} page={page} bf16={bf16}", flush=True)
    H, scale = 3, d_head ** -0.5
    q, k, v = cache(length, H, d_head, 100 * d_head + length)
    table = None
    if bf16:
        k, v = O.to_bf16_bits(k), O.to_bf16_bits(v)
    if page:
        k, v, table = paged_pool(k, v, page, 5)
        want, want_lse = O.decode(q, k, v, H, length, scale, block_table=table, page_size=page)
    else:
        want, want_lse = O.decode(q, k, v, H, length, scale)
    dk, dv = (dev_any(t.view(np.int16), device) if bf16 else to_dev(t, device) for t in (k, v))
    for ws in ("auto", None):
        out, lse = dfattn.decode(to_dev(q, device), dk, dv, H, length, scale, page_size=page or 1, workspace=ws,
                                 block_table=dev_any(table, device) if page else None)
        close("out", host(out), want)
        close("lse", host(lse), want_lse)


@pytest.mark.parametrize("d_head", [32, 64, 128])
def test_infinite_last_value(device, d_head):
    """The last key's value is infinite in one column: that column is infinite, not NaN (rows past the
    end stand for the last one but are not added), the others are untouched."""
    print(f"[gpu-decode-rows] infinite last value D={d_head}", flush=True)
    q, k, v = cache(70, 2, d_head, 7)
    clean, _ = dfattn.decode(to_dev(q, device), to_dev(k, device), to_dev(v, device), 2, 70)
    v[69, 3] = np.inf
    out, _ = dfattn.decode(to_dev(q, device), to_dev(k, device), to_dev(v, device), 2, 70)
    assert np.isposinf(host(out)[3])
    keep = np.arange(2 * d_head) != 3
    np.testing.assert_array_equal(host(out)[keep], host(clean)[keep])


@pytest.mark.parametrize("length", [2, 3, 40])
@pytest.mark.parametrize("d_head", [64, 80])
def test_first_score_of_minus_infinity(device, d_head, length):
    """A first key whose score is -inf has weight 0: the call is the one without it."""
    print(f"[gpu-decode-rows] -inf first score D={d_head} L={length}", flush=True)
    q, k, v = cache(length, 2, d_head, 8)
    want, want_lse = O.decode(q, k[1:], v[1:], 2, length - 1, d_head ** -0.5)
    for h in (0, d_head):
        k[0, h] = -np.inf if q[h] > 0 else np.inf
    out, lse = dfattn.decode(to_dev(q, device), to_dev(k, device), to_dev(v, device), 2, length)
    close("out", host(out), want)
    close("lse", host(lse), want_lse)
