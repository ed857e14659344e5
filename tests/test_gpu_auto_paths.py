"""NX_PATH_AUTO on layers large enough for its wider ranges (7 M weights a
matrix): the bits of the path it chooses, through nx_moe_forward_dev.  Experts
are built on the device; no oracle is needed, the paths have their own tests.
"""
import numpy as np
import pytest

import nexus_amd as nx
from moe_cases import Q2_K, Q4_0, Q4_K, Q8_0, DeviceArray, assert_same_bits

pytestmark = pytest.mark.gpu

GEMV, SPLIT, BF16 = nx.PATH_GEMV, nx.PATH_MFMA_SPLIT, nx.PATH_MFMA_BF16


@pytest.fixture(scope="module")
def ctx():
    c = nx.Context(0)
    yield c
    c.close()


def device_experts(ctx, fmt, E, H, F, Fs):
    """Experts of uniform weights, quantized by the library.  Every expert and
    the shared one hold the same three matrices: which path ran is seen in the
    bits whatever the weights."""
    ex = nx.Experts(ctx, fmt, E, H, F, Fs)
    rng = np.random.default_rng(E + H + F + fmt)
    src = DeviceArray(H * F)
    nb = nx.quant_bytes(fmt, H * F)
    q = DeviceArray(nb // 4 + 1)
    for role in (nx.ROLE_GATE, nx.ROLE_UP, nx.ROLE_DOWN):
        src.upload((rng.random(H * F, dtype=np.float32) - np.float32(0.5)) * np.float32(0.07))
        ctx.quantize_dev(fmt, src.ptr, H * F, q.ptr, nb)
        for e in range(E):
            ex.load_dev(e, role, q.ptr, nb)
        if Fs:
            assert Fs <= F
            ex.load_dev(nx.EXPERT_SHARED, role, q.ptr, nx.quant_bytes(fmt, H * Fs))
        ctx.sync()  # src and q are reused
    return ex


def forward(call, T, E, H, k, path, shift=0):
    """The call's output; x starts `shift` floats after an aligned address."""
    rng = np.random.default_rng(T + H)
    x = DeviceArray(T * H + shift)
    x.upload(rng.standard_normal(T * H).astype(np.float32), shift)
    lg = DeviceArray(T * E)
    lg.upload(rng.standard_normal(T * E).astype(np.float32))
    out = DeviceArray(T * H, fill=np.nan)
    call(x.ptr + 4 * shift, lg.ptr, T, k, out.ptr, path=path)
    got = out.download()
    assert np.isfinite(got).all()
    return got


# fmt, E, H, F, k, shared F, T, path with x unaligned
UNALIGNED = [
    (Q4_K, 4, 2048, 3584, 2, 0, 2, GEMV),     # 1.3 tokens per expert
    (Q4_0, 4, 2048, 3584, 2, 0, 5, GEMV),     # 2.6
    (Q8_0, 4, 2048, 3584, 2, 0, 5, GEMV),
    (Q4_K, 4, 2048, 3584, 2, 0, 25, BF16),    # 12.5
    (Q4_0, 4, 2048, 3584, 2, 3584, 4, GEMV),  # a shared expert, 4 tokens
    (Q8_0, 4, 2048, 3584, 2, 3584, 8, BF16),  # ... 8 tokens
    (Q4_K, 4, 512, 512, 2, 512, 4, GEMV),
    (Q2_K, 4, 512, 512, 2, 0, 9, GEMV),
]


@pytest.mark.parametrize("case", UNALIGNED, ids=lambda c: "-".join(map(str, c)))
def test_unaligned_input(ctx, case):
    """x on a 4-byte address: AUTO runs on a path that takes it, with the bits
    that path has for the same values at an aligned address; the split path
    asked for by name refuses it."""
    fmt, E, H, F, k, Fs, T, want = case
    print("auto unaligned", nx.FORMAT_NAMES[fmt], case, flush=True)
    ex = device_experts(ctx, fmt, E, H, F, Fs)
    ref = forward(ex.forward_dev, T, E, H, k, want)
    for shift in (1, 2):
        assert_same_bits(forward(ex.forward_dev, T, E, H, k, nx.PATH_AUTO, shift), ref)
        with pytest.raises(nx.NexusError, match="16-byte aligned") as e:
            forward(ex.forward_dev, T, E, H, k, SPLIT, shift)
        assert e.value.code == nx.NX_ERR_UNSUPPORTED
    ex.close()


# fmt, E, H, F, k, shared F, T, path: both sides of the limits of the rule
# (nexus_amd/csrc/nx_plan.hpp)
CHOICE = [
    (Q4_K, 8, 2048, 4608, 2, 0, 2, GEMV), (Q4_K, 8, 2048, 4608, 2, 0, 3, SPLIT),
    (Q4_K, 8, 2048, 4608, 2, 0, 51, SPLIT), (Q4_K, 8, 2048, 4608, 2, 0, 53, BF16),
    (Q4_0, 8, 2048, 4608, 2, 0, 4, GEMV), (Q4_0, 8, 2048, 4608, 2, 0, 5, SPLIT),
    (Q4_0, 8, 2048, 4608, 2, 0, 51, SPLIT), (Q4_0, 8, 2048, 4608, 2, 0, 53, BF16),
    (Q8_0, 8, 2048, 4608, 2, 0, 6, GEMV), (Q8_0, 8, 2048, 4608, 2, 0, 7, SPLIT),
    (Q8_0, 8, 2048, 4608, 2, 0, 47, SPLIT), (Q8_0, 8, 2048, 4608, 2, 0, 49, BF16),
    (Q4_0, 8, 2048, 4608, 2, 4608, 3, GEMV), (Q4_0, 8, 2048, 4608, 2, 4608, 4, SPLIT),
    (Q4_0, 8, 2048, 4608, 2, 4608, 47, SPLIT), (Q4_0, 8, 2048, 4608, 2, 4608, 49, BF16),
    (Q8_0, 8, 2048, 4608, 2, 4608, 5, GEMV), (Q8_0, 8, 2048, 4608, 2, 4608, 6, SPLIT),
    (Q8_0, 8, 2048, 4608, 2, 4608, 31, SPLIT), (Q8_0, 8, 2048, 4608, 2, 4608, 33, BF16),
    (Q4_K, 8, 1024, 2048, 2, 0, 4, GEMV), (Q4_K, 8, 1024, 2048, 2, 0, 5, SPLIT),
    (Q8_0, 64, 1024, 768, 8, 0, 5, GEMV), (Q8_0, 64, 1024, 768, 8, 0, 6, SPLIT),
]


@pytest.mark.parametrize("case", CHOICE, ids=lambda c: "-".join(map(str, c)))
def test_choice(ctx, case):
    fmt, E, H, F, k, Fs, T, want = case
    print("auto choice", nx.FORMAT_NAMES[fmt], case, flush=True)
    ex = device_experts(ctx, fmt, E, H, F, Fs)
    outs = {p: forward(ex.forward_dev, T, E, H, k, p) for p in (GEMV, SPLIT, BF16)}
    assert_same_bits(forward(ex.forward_dev, T, E, H, k, nx.PATH_AUTO), outs[want])
    for p, out in outs.items():  # the bits tell the paths apart
        assert p == want or not np.array_equal(out, outs[want])
    ex.close()


def test_choice_in_the_scratch_array(ctx):
    """12.6 tokens per expert, whose split workspace is above the scratch array:
    the no-allocation call runs on the grouped GEMM, which fits."""
    E, H, F, k, T = 64, 2304, 4096, 8, 101
    print("auto choice, no allocation", E, H, F, k, T, flush=True)
    ex = device_experts(ctx, Q4_K, E, H, F, 0)
    assert_same_bits(forward(ex.forward_noalloc, T, E, H, k, nx.PATH_AUTO),
                     forward(ex.forward_dev, T, E, H, k, BF16))
    assert_same_bits(forward(ex.forward_dev, T, E, H, k, nx.PATH_AUTO),
                     forward(ex.forward_dev, T, E, H, k, SPLIT))
    ex.close()
