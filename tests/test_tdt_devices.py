"""A TDT op made on one GPU while another is current asks its own GPU what it
holds. Runs on the CPU: a child process loads the library with a HIP runtime
stub of eight devices that counts the queries made with the wrong one current."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r"""
#include <stdlib.h>
static int current, expected = -1;
int stub_wrong, stub_queries;
void stub_expect(int device) { expected = device; }
static void query(void) { ++stub_queries; stub_wrong += expected >= 0 && current != expected; }
int hipGetDeviceCount(int* n) { *n = 8; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipGetDevice(int* d) { *d = current; return 0; }
int hipStreamCreateWithFlags(void** s, unsigned f) { *s = 0; return 0; }
int hipStreamDestroy(void* s) { return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipFuncSetAttribute(const void* f, int a, int v) { query(); return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t l) { query(); *n = 1; return 0; }
int hipMalloc(void** p, size_t n) { query(); *p = malloc(n); return 0; }
int hipFree(void* p) { free(p); return 0; }
"""

CHILD = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import parakeet_wgsl_amd.palette_abi as abi
class Buffer:
    def __init__(self, nbytes=1 << 40):
        self.ptr, self.nbytes = 4096, nbytes
def weight(name, size):
    count = (2560 if "lstm" in name else 640 if "projector" in name else 1032) if "bias" in name else 640 * (
        1025 if "embedding" in name else 5120 if "lstm" in name else 640 if "projector" in name else 1032)
    return Buffer(count * (4 if "bias" in name else size))
any_size = Buffer()
own, other = abi.Context(3), abi.Context(0)
for precision in ("f16", "f32"):
    stub.hipSetDevice(0)
    stub.stub_expect(3)
    weights = {n: weight(n, 2 if precision == "f16" else 4) for n in abi.TDT_WEIGHT_NAMES}
    slices = ("encoder_projected", "encoded_lengths", "decode_starts", "decode_ends", "flush_finals", "tokens",
              "token_frames", "token_durations", "metadata", "state", "predictor_scratch")
    op = abi.TdtDecoderOp(own, weights=weights, batch_size=4, frames=188, max_tokens=64, precision=precision,
                          **{n: any_size for n in slices})
    assert op.resident_windows()
    stub.hipSetDevice(0)
    op.set_team_size(0)
    assert op.resident_windows()
    op.release()
wrong, queries = (ctypes.c_int.in_dll(stub, n).value for n in ("stub_wrong", "stub_queries"))
print("wrong", wrong, "of", queries)
assert queries and not wrong
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc is not installed")
def test_queries_go_to_the_ops_own_device(abi, tmp_path):
    source, stub = tmp_path / "hip_stub.c", tmp_path / "hip_stub.so"
    source.write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", str(source), "-o", str(stub)], check=True)
    preload = ":".join(p for p in (str(stub), os.environ.get("LD_PRELOAD")) if p)
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=ROOT)
    child = subprocess.run([sys.executable, "-c", CHILD, str(stub)], cwd=ROOT, env=env, capture_output=True, text=True,
                           timeout=120)
    assert child.returncode == 0, child.stdout + child.stderr
