"""Exact router logits of 262144 (token, expert) chains and more: the products
come from the matrix cores, and must be the reference's separately rounded
ones (src/engine/mod.rs:775-801), subnormal, infinite and NaN ones included.
Partial tiles of tokens and experts, rows of less than one stage of 64 columns,
of whole stages and with a remainder; bit-identical to the oracle.
"""
import numpy as np
import pytest

import nexus_amd as nx
import oracle
from moe_cases import assert_same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = nx.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("T,E,H", [(1031, 257, 60), (1031, 257, 196), (32768, 8, 64), (2062, 129, 128)])
def test_bits(ctx, T, E, H):
    print(f"router logits outer T={T} E={E} H={H}", flush=True)
    rng = np.random.default_rng(T + E + H)
    w = (rng.standard_normal((E, H)) * 0.05).astype(np.float32)
    x = rng.standard_normal((T, H)).astype(np.float32)
    w[0] *= np.float32(1e-20)  # subnormal products
    x[0] *= np.float32(1e-21)
    x[T - 1] *= np.float32(1e-38)  # subnormal factors
    x[1, 5] = np.inf
    w[3, 5] = 0.0  # inf * 0
    x[2, 7] = np.nan
    x[3] = -0.0
    w[4] = 3e38  # overflow inside the chain
    w[5, ::2] = 3e38
    w[5, 1::2] = -3e38
    got = ctx.router_logits(w, x, E, H, exact=True)
    ref = np.stack([oracle.matvec(w, E, H, xt) for xt in x])
    assert_same_bits(got, ref)
    assert not np.signbit(got[3]).any()
    assert 0.0 < abs(got[0, 0]) < 1.2e-38
