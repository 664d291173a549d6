"""The small-M kernel's 32 x 32 tile with activation rows through LDS (more
than one row group): its sums are those of the form that reads fragments
from memory (one row group), bit for bit, and match the oracle."""
import numpy as np
import pytest

from test_gpu_parity import Scope, assert_f16_parity, run_case, small_m_variants, variant_names

pytestmark = pytest.mark.gpu


@pytest.fixture
def scope(ctx):
    s = Scope(ctx)
    yield s
    s.close()


# both forms at their border, uneven shares, four and more K blocks each; and
# below it, where every row count reads fragments from memory
@pytest.mark.parametrize("rows,inner,columns,bits,scale", [
    (33, 64, 32, 5, None), (34, 512, 96, 6, 0.5), (63, 704, 160, 5, None), (61, 768, 160, 5, None),
    (90, 832, 64, 6, None), (64, 1024, 4096, 5, None),
    (95, 2112, 64, 6, None), (188, 4096, 1024, 5, 0.5), (300, 2624, 96, 5, None)])
def test_staged_rows_match_fragments(abi, ctx, scope, oracle, workloads, rows, inner, columns, bits, scale):
    names = variant_names(abi, ctx, scope, workloads)
    variant = next(i for i in small_m_variants(abi, ctx, scope, workloads) if "_k8_m1n1" in names[i])
    case = workloads.gemm_case(rows, rows, inner, columns, bits, activation="silu", residual_scale=scale)
    got = run_case(abi, ctx, scope, case, variant=variant)
    assert_f16_parity(oracle, got, case)
    for active in (1, 17, 32):
        prefix = run_case(abi, ctx, scope, case, variant=variant, active_rows=active)
        print(rows, inner, columns, "prefix", active, flush=True)
        np.testing.assert_array_equal(prefix[:active].view(np.uint16), got[:active].view(np.uint16))
