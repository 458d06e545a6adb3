"""Barriers among workgroups, in the code that the compiler makes of them: an
arrival tells the other workgroups that every wave's stores have reached memory,
and a workgroup barrier alone does not wait for the other waves' stores."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = """
#include "dev_common.h"
using namespace upside;
__device__ __forceinline__ Ctx context(const RunArgs* a, float* f, int* words, int local) {
    extern __shared__ int lds[];
    Ctx c;
    c.args = cmem(a);
    c.G = 8;
    c.rank = (int)blockIdx.x;
    c.local = local;
    c.tid = (int)threadIdx.x;
    c.lost = (lp<int>)lds;
    c.bar = (gp<unsigned long long>)words;
    c.bar_flag = (gp<unsigned>)(words + 2);
    c.bar_next = 8;
    c.spin_limit = a->spin_limit;
    c.prof = nullptr;
    f[blockIdx.x * NT + threadIdx.x] = 1.f;
    return c;
}
extern "C" __global__ void on_one_xcd(const RunArgs* a, float* f, int* w) { Ctx c = context(a, f, w, 1); team_sync(c); }
extern "C" __global__ void spread(const RunArgs* a, float* f, int* w) { Ctx c = context(a, f, w, 0); team_sync(c); }
extern "C" __global__ void all_systems(const RunArgs* a, float* f, int* w) {
    Ctx c = context(a, f, w, 1);
    grid_sync(c, c.args->rex);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_stores_are_waited_for_before_an_arrival(tmp_path):
    src, out = tmp_path / "barriers.hip", tmp_path / "barriers.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(PKG, "csrc"), "--cuda-device-only", "-S", str(src), "-o",
                    str(out)], check=True, capture_output=True, timeout=300)
    text = out.read_text()
    for kernel in ("on_one_xcd", "spread", "all_systems"):
        body = text[text.index("\n%s:" % kernel):]
        ops = [line.split(";")[0].strip() for line in body[:body.index("s_endpgm")].splitlines()]
        store = next(i for i, op in enumerate(ops) if op.startswith("global_store_dword"))
        barrier = next(i for i, op in enumerate(ops) if i > store and op == "s_barrier")
        arrival = next(i for i, op in enumerate(ops) if op.startswith("global_atomic_add_x2"))
        assert store < barrier < arrival, kernel
        assert any(op.startswith("s_waitcnt") and "vmcnt(0)" in op for op in ops[store:barrier]), kernel
