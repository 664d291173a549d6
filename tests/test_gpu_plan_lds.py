"""pk_gemm_plan against the code objects of the library: the kernel that a plan
names and its LDS are those of the compiled kernel, for every f32 tile, the
small-M forms on both sides of their rule, the other f16 families and a group."""
import os
import re
import struct
import subprocess

import numpy as np
import pytest

from test_gpu_parity import Scope

pytestmark = pytest.mark.gpu
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture
def scope(ctx):
    s = Scope(ctx)
    yield s
    s.close()


@pytest.fixture(scope="module")
def compiled(abi, tmp_path_factory):
    """Static LDS of every kernel in the library, by mangled name."""
    if not os.path.exists(READELF):
        pytest.skip("llvm-readelf is not installed")
    with open(abi.LIB_PATH, "rb") as f:
        library = f.read()
    magic, lds = b"__CLANG_OFFLOAD_BUNDLE__", {}
    path = str(tmp_path_factory.mktemp("code") / "object.co")
    at = library.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", library, at + len(magic))
        entry = at + len(magic) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", library, entry)
            target = library[entry + 24:entry + 24 + name].decode()
            entry += 24 + name
            if "gfx950" not in target:
                continue
            with open(path, "wb") as f:
                f.write(library[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True, check=True).stdout
            sizes = re.findall(r"\.group_segment_fixed_size:\s*(\d+)", notes)
            names = re.findall(r"^\s+\.name:\s+(_Z\S+)", notes, re.M)
            assert len(sizes) == len(names)
            lds.update(zip(names, map(int, sizes)))
        at = library.find(magic, at + 1)
    assert lds
    return lds


def parameters(kernel, *values):
    """Mangled template arguments: integers as Li..E, truth values as Lb..E."""
    return kernel + "I" + "".join(f"Lb{int(v)}E" if isinstance(v, bool) else f"Li{v}E" for v in values) + "E"


def of(compiled, part):
    found = {v for k, v in compiled.items() if part in k}
    assert len(found) == 1, (part, found)
    return found.pop()


def gemm(abi, ctx, scope, workloads, rows, inner, columns, bits, dtype):
    case = workloads.gemm_case(1, rows, inner, columns, bits, dtype=dtype)
    w = case.weight
    return abi.GemmOp(ctx, a=scope.put(case.a), packed=scope.put(w.packed), palette=scope.put(w.palette),
                      output=scope.empty((rows, columns), dtype), bits=bits, rows=rows, inner=inner, columns=columns)


@pytest.mark.parametrize("bits", [5, 6])
def test_f32_plans(abi, ctx, scope, workloads, compiled, bits):
    op = gemm(abi, ctx, scope, workloads, 64, 128, 256, bits, np.float32)
    try:
        for variant in range(abi.variant_count("f32")):
            op.set_variant(variant)
            plan = op.plan()
            wn, ks, mb, nb = map(int, re.fullmatch(rb"pk_gemm_f32_b\d_n(\d)k(\d)_m(\d)n(\d)", plan.kernel).groups())
            assert plan.lds_bytes == of(compiled, parameters("gemm_f32_kernel", bits, wn, mb, nb, ks))
    finally:
        op.release()


# one row group, rows through LDS from K = 768 on, an upper half of padding
@pytest.mark.parametrize("rows,inner,staged", [(32, 1024, False), (33, 704, False), (33, 768, True), (64, 1056, False),
                                               (64, 1024, True)])
@pytest.mark.parametrize("bits", [5, 6])
def test_small_m_plans(abi, ctx, scope, workloads, compiled, bits, rows, inner, staged):
    op = gemm(abi, ctx, scope, workloads, rows, inner, 64, bits, np.float16)
    try:
        plan = op.plan()
        assert plan.kernel.decode() == f"pk_gemm_f16s_b{bits}_k8_m1n1d" + ("4rows" if staged else "2")
        general = inner % 64 != 0
        assert plan.lds_bytes == of(compiled, parameters("gemm_f16s_kernel", bits, 8, 1, 1, 4 if staged else 2,
                                                         general, staged))
        assert op.plan(32).kernel.decode().endswith("d2")
    finally:
        op.release()


def test_pair_code_operand_order_and_group_plans(abi, ctx, scope, workloads, compiled):
    ops = [gemm(abi, ctx, scope, workloads, 64, 512, 128, bits, np.float16) for bits in (5, 6)]
    group = abi.GemmGroup(ctx, ops)
    try:
        plan = group.plan()
        kind, w, rw, cb, d, occ = re.fullmatch(rb"pk_gemm_f16s_(group|stream)_k(\d)_m(\d)n(\d)d(\d)(?:o(\d))?",
                                               plan.kernel).groups()
        values = [int(x) for x in (w, rw, cb, d, occ) if x]
        assert plan.lds_bytes == of(compiled, parameters(f"gemm_f16s_{kind.decode()}_kernel", *values))
    finally:
        group.release()
        for op in ops:
            op.release()
    for bits in (5, 6):
        op = gemm(abi, ctx, scope, workloads, 128, 512, 256, bits, np.float16)
        try:
            for variant in range(abi.variant_count("f16")):
                op.set_variant(variant)
                plan = op.plan()
                m = re.fullmatch(rb"pk_gemm_f16_b\d_w(\d)x(\d)_m(\d)n(\d)", plan.kernel)
                if m:
                    name = parameters("gemm_f16_kernel", bits, *map(int, m.groups()), False)
                    assert plan.lds_bytes == of(compiled, name)
                m = re.fullmatch(rb"pk_gemm_f16p_b\d_n(\d)k(\d)_m(\d)n(\d)", plan.kernel)
                if m:
                    name = parameters("gemm_f16k_kernel", bits, *map(int, m.groups()), False)[:-1]
                    stored = f"Lb0ELb{int(plan.stream_stores)}EE"
                    found = {v for k, v in compiled.items() if name in k and stored in k}
                    assert found == {plan.lds_bytes}, (plan.kernel, plan.lds_bytes, found)
        finally:
            op.release()
