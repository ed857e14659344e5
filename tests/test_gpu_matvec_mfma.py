"""Dense matvec of five and more tokens on the matrix cores (nx_mfd.hip).

Against the oracle's dequantization of the same payload in 64 bits.  The
sizes cover ragged last row and token tiles, fewer chunks of 256 columns than a
workgroup has waves, rows of several panels, and in INSTANCES each instance on
256 CUs (1, 2 or 4 row tiles of 16 per wave; 8, 4 or 2 chunk groups with 1, 2 or
4 token tiles) over several steps of which the last is ragged; test_plan.py
checks that those sizes choose them.

Bound per output: the operands carry 22 bits, and a product is rounded at
most some 2^5 times on its way (8 MFMAs, the chunks and the 8 waves' sums), so
the error is below 2^5 2^-24 times the sum of the magnitudes of the terms.
These are the products and, for Q4_K, the offsets taken off again, below
twice the products for weights of both signs; sum |w x| <= |w| |x|: in
all 2^-18 |w| |x|.
"""
import numpy as np
import pytest

import nexus_amd as nx
import oracle
from moe_cases import DeviceArray, assert_same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = nx.Context(0)
    yield c
    c.close()


def matrix(ctx, fmt, rows, cols, seed):
    w = (np.random.default_rng(seed).standard_normal(rows * cols) * 0.05).astype(np.float32)
    q = oracle.quantize(fmt, w)
    m = nx.Matrix(ctx, fmt, rows, cols)
    m.load(q)
    return m, oracle.dequantize(fmt, q, rows * cols).reshape(rows, cols).astype(np.float64)


def assert_close(got, w, x):
    x = x.astype(np.float64)
    bound = 2.0 ** -18 * np.linalg.norm(x, axis=1)[:, None] * np.linalg.norm(w, axis=1)[None, :]
    err = np.abs(got - x @ w.T)
    assert np.all(err <= bound), np.nanmax(err / np.maximum(bound, 1e-300), axis=1)


# row tiles per wave, chunk groups, and a size that chooses them
INSTANCES = [(1, 8, 37, 2304, 5), (2, 8, 325, 2304, 200), (4, 8, 500, 3328, 260), (1, 4, 325, 2304, 400),
             (2, 4, 1000, 2304, 260), (1, 2, 1335, 1280, 400), (2, 2, 8197, 1280, 65)]


@pytest.mark.parametrize("fmt", [nx.Q4_K, nx.Q4_0, nx.Q8_0])
@pytest.mark.parametrize("case", INSTANCES, ids=lambda c: "%dx%d-%d-%d-%d" % c)
def test_instances(ctx, fmt, case):
    print(f"matvec instance fmt={nx.FORMAT_NAMES[fmt]} {case}", flush=True)
    rows, cols, T = case[2:]
    m, w = matrix(ctx, fmt, rows, cols, seed=rows + cols + T + fmt)
    x = np.random.default_rng(T).standard_normal((T, cols)).astype(np.float32)
    got = m.matvec(x)
    assert_close(got, w, x)
    # and as close to 64 bits as the kernel's error elsewhere (2.1e-7), per token
    ref = x.astype(np.float64) @ w.T
    assert np.all(np.linalg.norm(got - ref, axis=1) < 2.0 ** -20 * np.linalg.norm(ref, axis=1))
    m.close()


@pytest.mark.parametrize("fmt", [nx.Q4_K, nx.Q4_0, nx.Q8_0])
@pytest.mark.parametrize("rows,cols,T", [(1, 256, 5), (37, 512, 16), (100, 2304, 17), (256, 14336, 33),
                                         (8197, 256, 7), (16389, 256, 9), (16389, 512, 45)])
def test_parity(ctx, fmt, rows, cols, T):
    print(f"matvec fmt={nx.FORMAT_NAMES[fmt]} rows={rows} cols={cols} T={T}", flush=True)
    m, w = matrix(ctx, fmt, rows, cols, seed=rows + cols + T + fmt)
    x = np.random.default_rng(T).standard_normal((T, cols)).astype(np.float32)
    x[0] *= 1e30
    x[-1] *= 1e-25
    x[1] = 0.0
    x[2, ::3] *= 1e4
    got = m.matvec(x)
    assert_close(got, w, x)
    assert np.all(got[1] == 0.0)
    m.close()


@pytest.mark.parametrize("fmt", [nx.Q4_K, nx.Q4_0, nx.Q8_0])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_token(ctx, fmt, bad):
    m, w = matrix(ctx, fmt, 48, 768, seed=fmt)
    x = np.random.default_rng(1).standard_normal((19, 768)).astype(np.float32)
    clean = m.matvec(x)
    x[4, 700] = bad
    got = m.matvec(x)
    assert np.all(np.isnan(got[4]))
    keep = np.arange(19) != 4
    assert_same_bits(got[keep], clean[keep])
    m.close()


def test_unaligned_input(ctx):
    """Rows that are not 16-byte aligned stay on the GEMV, with its results."""
    m, w = matrix(ctx, nx.Q4_K, 80, 512, seed=3)
    x = np.random.default_rng(2).standard_normal((6, 512)).astype(np.float32)
    dx, dy = DeviceArray(x.size + 1), DeviceArray(6 * 80 + 1, fill=7.0)
    dx.upload(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    m.matvec_dev(dx.ptr + 4, x.size, 6, dy.ptr)
    out = dy.download()
    assert_close(out[:480].reshape(6, 80), w, x)
    assert out[480] == 7.0
    m.close()


@pytest.mark.parametrize("fmt,rows,cols", [(nx.Q4_K, 256, 10496), (nx.Q4_K, 17, 14336),
                                           (nx.Q8_0, 256, 4352), (nx.Q8_0, 48, 8192)])
def test_few_long_rows_stay_on_the_gemv(ctx, fmt, rows, cols):
    """Up to six tokens of at most 256 long rows: the GEMV, which gives each
    token the bits of a call of its own."""
    m, w = matrix(ctx, fmt, rows, cols, seed=rows + cols)
    x = np.random.default_rng(9).standard_normal((6, cols)).astype(np.float32)
    alone = np.concatenate([m.matvec(x[t:t + 1]) for t in range(6)])
    for T in (5, 6):
        assert_same_bits(m.matvec(x[:T]), alone[:T])
    assert_close(alone, w, x)
    m.close()


@pytest.mark.parametrize("fmt", [nx.Q4_K, nx.Q4_0, nx.Q8_0])
def test_smallest_normal_values(ctx, fmt):
    """Tokens of the smallest normal numbers keep the precision of others: their
    scaled maximum is at least 1, whose two halves reach 2^-25, so the error of
    a value is some 2^-24 of the maximum and a sum's relative error below 2^-20."""
    m, w = matrix(ctx, fmt, 64, 512, seed=fmt + 5)
    x = np.random.default_rng(7).standard_normal((9, 512)).astype(np.float32)
    x *= np.logspace(-37, -34, 9, dtype=np.float32)[:, None]
    got = m.matvec(x).astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert np.all(err < 2.0 ** -20), err
    m.close()
