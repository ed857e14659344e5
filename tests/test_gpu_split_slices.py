"""The split path's K slices, runs of row tiles and activation records.

A workgroup of k_mfv takes one K slice of up to 8 chunks of 256 columns, a wave
per chunk, and an equal run of all (tile, slice, row tile) work: widths of 1,
8 and 9 chunks (one slice whole, two of which the second leaves a wave idle),
11 (6 and 5), and 18 (three of 6) in both products; tiles of one pair and of
16 and 17.  Bar: the split path's, relative L2 1e-4 of the oracle.  A token
with a non-finite activation gives NaN in its own row only.  The path's own
precision is held against 64 bits.
"""
import numpy as np
import pytest

import nexus_amd as nx
import oracle
from moe_cases import Q2_K, Q4_0, Q4_K, Q8_0, Layer, assert_same_bits, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = nx.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("fmt", [Q4_K, Q4_0, Q8_0, Q2_K])
@pytest.mark.parametrize("E,H,F,k,T", [(4, 2304, 256, 2, 3), (3, 256, 2816, 1, 51), (2, 2048, 4608, 2, 17),
                                       (5, 1024, 2304, 2, 1)])
def test_slices(ctx, fmt, E, H, F, k, T):
    print(f"split slices fmt={nx.FORMAT_NAMES[fmt]} E={E} H={H} F={F} k={k} T={T}", flush=True)
    L = Layer(fmt, E, H, F, k, T, seed=E + H + F + T)
    ex = L.upload(nx, ctx)
    got = ex.forward(L.x, L.logits, k, 0, nx.PATH_MFMA_SPLIT)
    assert rel_l2(got, L.oracle_out()) <= 1e-4
    # one row's non-finite activation stays in its row
    if T > 1:
        x = L.x.copy()
        x[1, H - 1] = np.inf
        bad = ex.forward(x, L.logits, k, 0, nx.PATH_MFMA_SPLIT)
        assert np.all(np.isnan(bad[1]))
        keep = np.arange(T) != 1
        assert_same_bits(bad[keep], got[keep])
    ex.close()


@pytest.mark.parametrize("fmt", [Q4_K, Q4_0, Q8_0, Q2_K])
def test_precision(ctx, fmt):
    """Against the layer in 64 bits on the same routes and weights: activations
    carry 22 bits and a sign (2^-23), sums are in 32 bits, three products deep:
    2^-20 (measured 2e-7 to 4e-7; operands left as fp16 subnormals gave 8e-5)."""
    E, H, F, k, T = 6, 1024, 1536, 2, 29
    L = Layer(fmt, E, H, F, k, T, seed=fmt)
    ex = L.upload(nx, ctx)
    got = ex.forward(L.x, L.logits, k, 0, nx.PATH_MFMA_SPLIT)
    ex.close()
    idx, weight, count, _ = oracle.route(L.logits, T, E, k, 0)
    ref = np.zeros((T, H))
    for t in range(T):
        x = L.x[t].astype(np.float64)
        for e, w in list(zip(idx[t], weight[t]))[:count[t]]:
            gate, up, down = (L.dense[(int(e), r)].astype(np.float64).reshape(s)
                              for r, s in ((0, (F, H)), (1, (F, H)), (2, (H, F))))
            g = gate @ x
            ref[t] += w * (down @ (g / (1.0 + np.exp(-g)) * (up @ x)))
    assert rel_l2(got, ref) < 2.0 ** -20
