"""The f32 palette GEMM's split product (three bf16 terms per operand) on
every tile: edges of the tiles and K tails, several palette groups in one
tile, and operands that have no split (infinite, NaN, beyond the largest
bf16), which come from the f32 matrix units instead."""
import numpy as np
import pytest

from test_gpu_parity import Scope, run_case
from test_split_product import SINGLE_BOUND, sum_bound

pytestmark = pytest.mark.gpu


@pytest.fixture
def scope(ctx):
    s = Scope(ctx)
    yield s
    s.close()


def exact(workloads, case):
    codes = case.weight.codes.astype(np.int64)
    lut = case.weight.palette.astype(np.float64).reshape(-1, 1 << case.weight.bits)
    n = codes.shape[1]
    group = np.minimum(np.arange(n) // max(n // lut.shape[0], 1), lut.shape[0] - 1)
    with np.errstate(invalid="ignore", over="ignore"):
        y = case.a.astype(np.float64) @ lut[group[None, :], codes]
        if case.bias is not None:
            y = y + case.bias.astype(np.float64)
        if case.activation == "relu":
            y = np.maximum(y, 0)
    return y


@pytest.mark.parametrize("rows,inner,columns,bits,groups", [
    (1, 64, 128, 5, 1), (31, 32, 16, 6, 1), (33, 96, 160, 5, 1), (65, 160, 272, 6, 1), (97, 192, 96, 6, 3),
    (129, 320, 384, 5, 3), (193, 1024, 528, 6, 1), (40, 4096, 64, 5, 1)])
def test_split_product_on_every_tile(abi, ctx, scope, workloads, rows, inner, columns, bits, groups):
    case = workloads.gemm_case(rows + inner, rows, inner, columns, bits, dtype=np.float32, groups=groups,
                               bias=True, activation="relu" if rows % 2 else "none")
    want = exact(workloads, case)
    for variant in [None] + list(range(abi.variant_count("f32"))):
        got = run_case(abi, ctx, scope, case, variant=variant)
        error = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(rows, inner, columns, "variant", variant, "error", error, flush=True)
        assert error <= sum_bound(inner)


def test_single_products_are_exact(abi, ctx, scope, workloads):
    """One operand per row that is not zero, at every k of five K blocks: each
    output is one product of full significands."""
    case = workloads.gemm_case(5, 320, 320, 160, 6, dtype=np.float32)
    case.a[...] = np.diag(np.diag(case.a))
    want = exact(workloads, case)
    assert (want != 0).all()
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant)
        error = np.max(np.abs(got / want - 1))
        print("variant", variant, "error", error, flush=True)
        assert error <= SINGLE_BOUND


def test_wide_range_of_magnitudes(abi, ctx, scope, workloads):
    """Rows scaled from 1e-30 to 1e30: each row's own error stays that of f32
    (twice the bound: 128 outputs each, the large rows from the f32 units)."""
    case = workloads.gemm_case(3, 61, 256, 128, 5, dtype=np.float32)
    case.a *= (10.0 ** np.arange(-30, 31)[:, None]).astype(np.float32)
    want = exact(workloads, case)
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant).astype(np.float64)
        assert (np.linalg.norm(got - want, axis=1) <= 2 * sum_bound(256) * np.linalg.norm(want, axis=1)).all()


@pytest.mark.parametrize("where", ["a", "palette"])
def test_operands_without_a_split(abi, ctx, scope, workloads, where):
    """Infinity, NaN and 3.4e38 in A or in the palette: the outputs are what
    f32 arithmetic gives (infinities of the right sign, NaN where they meet)
    and the rows and columns without them keep their values."""
    case = workloads.gemm_case(9, 70, 192, 160, 5, dtype=np.float32)
    if where == "a":
        case.a[3, 5], case.a[40, 100], case.a[65, 7], case.a[69, 191] = np.inf, np.nan, -np.inf, 3.4e38
    else:
        case.weight.palette[...] = np.where(np.arange(32) == 7, np.inf, case.weight.palette)
        case.weight.codes[:, 3:] = np.where(case.weight.codes[:, 3:] == 7, 8, case.weight.codes[:, 3:])
        case.weight.packed[...] = workloads.pack_codes(case.weight.codes, 5)
    want = exact(workloads, case)
    finite = np.isfinite(want)
    assert 0 < finite.sum() < finite.size
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
        error = np.abs(got[finite] - want[finite]) / np.maximum(np.abs(want[finite]), 1.0)
        assert error.max() <= 8 * sum_bound(192)  # the largest of 11,000 outputs


def test_sums_have_no_offset(abi, ctx, scope, workloads):
    """The matrix unit rounds its sums down; subtracting half of the K
    blocks cancels that. The mean error of 65,536 outputs, each off by up to
    1e-6 of their size at random, is below 1e-6 / 256; uncancelled runs may
    leave a tenth of the 3e-7 that the offset is without them."""
    case = workloads.gemm_case(11, 512, 4096, 128, 5, dtype=np.float32)
    want = exact(workloads, case)
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant)
        offset = np.mean(got - want) / np.mean(np.abs(want))
        print("variant", variant, "offset", offset, flush=True)
        assert abs(offset) <= 3.4e-8


@pytest.mark.parametrize("exponent", [-100, -112, -120, -126, -140])
@pytest.mark.parametrize("where", ["a", "palette"])
def test_operands_down_to_the_smallest_subnormals(abi, ctx, scope, workloads, where, exponent):
    """Operands of about 2^exponent against ones of about 2^60: the bits that
    bf16's exponent range has no room for count like any other's."""
    case = workloads.gemm_case(17, 70, 320, 160, 5, dtype=np.float32)
    w = case.weight.palette
    small, large = (case.a, w) if where == "a" else (w, case.a)
    small[...] = np.ldexp(small.astype(np.float64) / small.std(), exponent).astype(np.float32)
    large[...] = np.ldexp(large.astype(np.float64) / large.std(), 60).astype(np.float32)
    want = exact(workloads, case)
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant)
        error = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(where, exponent, "variant", variant, "error", error, flush=True)
        assert error <= sum_bound(320)


def test_an_output_depends_on_its_own_row_and_column_alone(abi, ctx, scope, workloads):
    """A row that is not finite leaves the other rows of its tile as they are, to the bit."""
    case = workloads.gemm_case(19, 96, 256, 160, 5, dtype=np.float32)
    clean = case.a.copy()
    for variant in range(abi.variant_count("f32")):
        case.a[...] = clean
        want = run_case(abi, ctx, scope, case, variant=variant)
        case.a[[2, 70], 9] = np.nan, 3e38
        got = run_case(abi, ctx, scope, case, variant=variant)
        others = np.setdiff1d(np.arange(96), [2, 70])
        assert np.isnan(got[2]).all()
        np.testing.assert_array_equal(got[others].view(np.uint32), want[others].view(np.uint32))


@pytest.mark.parametrize("inner", [96, 128, 192, 256])
def test_short_sums_have_no_offset(abi, ctx, scope, workloads, inner):
    """Sums of two to four K blocks, on every tile: the mean error of a million
    outputs (each off by at most 2.5e-7 of their size at random) stays under
    7e-9 of their mean size; with every block added it is 1.0e-8 to 1.7e-8."""
    case = workloads.gemm_case(inner, 2048, inner, 512, 5, dtype=np.float32)
    want = exact(workloads, case)
    for variant in range(abi.variant_count("f32")):
        got = run_case(abi, ctx, scope, case, variant=variant)
        offset = np.mean(got - want) / np.mean(np.abs(want))
        print(inner, "variant", variant, "offset", offset, flush=True)
        assert abs(offset) <= 7e-9
