"""Windows around and above 256 frames in every planned range of query tiles
(few: key-split wavefronts, above 256 frames with the next tile prefetched,
then the shared kernels), at tile edges, against the oracle."""
import pytest

from test_gpu_attention import assert_attention_parity, run_attention
from test_gpu_parity import Scope

pytestmark = pytest.mark.gpu


@pytest.fixture
def scope(ctx):
    s = Scope(ctx)
    yield s
    s.close()


@pytest.mark.parametrize("row_major", [False, True])
@pytest.mark.parametrize("batch,frames,valid,kernel", [
    (1, 33, [33], "q32_w4"), (2, 129, [129, 1], "q32_w4"), (3, 256, [256, 0, 65], "q32_w4"),
    (1, 257, [257], "q32_w4"), (2, 300, [289, 33], "q32_w4"), (1, 1024, [1000], "q32_w4"),
    (4, 320, [320, 1, 129, 0], "q2x32_shared"), (5, 320, [320, 64, 200, 31, 96], "q4x32_shared")])
def test_long_windows_match_oracle(abi, ctx, scope, oracle, workloads, batch, frames, valid, kernel, row_major):
    case = workloads.attention_case(90 + frames, batch, frames, valid=valid)
    print(f"attention f16 B={batch} T={frames} row_major={row_major}", flush=True)
    got, name = run_attention(abi, ctx, scope, case, row_major=row_major)
    assert name.endswith(kernel)
    assert_attention_parity(oracle, got, case)
