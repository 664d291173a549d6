"""What a test of the f32 GEMM's split product has to notice, on a CPU model of
it: with any one of its six products left out, sums and single products are
further from 64 bits than the bounds that the GPU tests hold the kernel to."""
import numpy as np
import pytest

# (term of the weight, term of the activation), as the kernel multiplies them
PRODUCTS = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]

# One product alone: the sum of its six parts rounds once at full size (2^-23
# where the matrix unit rounds down), the three left out are under 2^-25.
SINGLE_BOUND = 1.5 * 2.0**-23


def sum_bound(inner):
    """Norm-wise error of a sum of `inner` products: 3 inner / 8 additions to
    the accumulator, each off by up to 2^-23 of a partial sum, whose sizes grow
    as a random walk: about 2.2e-8 sqrt(inner); the kernel shows 1.5e-8."""
    return 2.5e-8 * np.sqrt(inner)


def bf16(x):
    bits = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    return ((bits + 0x7fff + (bits >> 16 & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def terms(x):
    x = x.astype(np.float32)
    hi = bf16(x)
    mid = bf16(x - hi)
    return [t.astype(np.float64) for t in (hi, mid, bf16(x - hi - mid))]


def product(a, w, without=None):
    at, wt = terms(a), terms(w)
    return sum(at[j] @ wt[i] for i, j in PRODUCTS if (i, j) != without)


@pytest.mark.parametrize("without", [None] + PRODUCTS)
@pytest.mark.parametrize("inner", [64, 1024, 4096])
def test_sums(inner, without):
    rng = np.random.default_rng(inner)
    a, w = (rng.standard_normal(s).astype(np.float32) for s in ((32, inner), (inner, 64)))
    want = a.astype(np.float64) @ w.astype(np.float64)
    error = np.linalg.norm(product(a, w, without) - want) / np.linalg.norm(want)
    assert (error > sum_bound(inner)) == (without is not None)


@pytest.mark.parametrize("without", [None] + PRODUCTS)
def test_single_products(without):
    rng = np.random.default_rng(1)
    a, w = rng.standard_normal((64, 1)).astype(np.float32), rng.standard_normal((1, 64)).astype(np.float32)
    want = a.astype(np.float64) @ w.astype(np.float64)
    assert (np.max(np.abs(product(a, w, without) / want - 1)) > SINGLE_BOUND) == (without is not None)


def test_terms_are_exact_down_to_the_smallest_scaled_subnormal():
    bits = np.random.default_rng(2).integers(0, 1 << 23, 4096)
    x = (bits.astype(np.float64) * 2.0**-149 * 2.0**24).astype(np.float32)
    parts = terms(x)
    np.testing.assert_array_equal(sum(parts), x.astype(np.float64))
    assert all((np.abs(p[p != 0]) >= 2.0**-126).all() for p in parts)
