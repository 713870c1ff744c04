"""Launches with more LDS than a kernel gets by default raise that kernel's limit first.  The limit belongs to the kernel, not to the call:
threads that raise it for launches of their own must not take it from each other, so whatever the size a kernel asks for one value, and
its launches stay inside it.  Runs without a GPU: stand-ins for the runtime's launch calls write down what they are asked for."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAND_INS = r"""
#include <cstddef>
#include <cstdio>
struct dim3 { unsigned x, y, z; };
static dim3 grid_, block_; static size_t lds_; static void* stream_;
extern "C" {
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) { grid_ = g; block_ = b; lds_ = lds; stream_ = s; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) { *g = grid_; *b = block_; *lds = lds_; *s = stream_; return 0; }
int hipFuncSetAttribute(const void* f, int, int v) { std::printf("limit %p %d\n", f, v); return 0; }
int hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, void*) { std::printf("launch %p %zu\n", f, lds); return 0; }
int hipGetLastError() { return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
}
"""
CALLS = r"""
import ctypes as C, importlib.util, sys
C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)                    # ahead of the runtime
spec = importlib.util.spec_from_file_location("_lib", sys.argv[2])
_lib = importlib.util.module_from_spec(spec); spec.loader.exec_module(_lib)
lib, at = _lib.lib(), 1 << 20                              # (addresses that nothing reads)
def scan(lanes, waves):
    p = _lib.QaSScanParams()
    p.batch, p.dim, p.seqlen, p.dstate, p.n_groups, p.delta_softplus, p.token_major = 1, 64, 900, 16, 1, 1, 1
    for n in ("u", "delta", "z", "out"):
        setattr(p, n + "_batch_stride", 900 * 64); setattr(p, n + "_l_stride", 64); setattr(p, n + "_d_stride", 1)
    p.B_batch_stride = p.C_batch_stride = 900 * 32; p.B_l_stride = p.C_l_stride = 32; p.B_dstate_stride = p.C_dstate_stride = 1
    p.A_d_stride, p.A_dstate_stride = 16, 1
    for n in ("u", "delta", "z", "A_log", "B", "C", "out", "scale_u", "scale_delta", "scale_A", "scale_B", "scale_C", "scale_z"): setattr(p, n, at)
    p.mapping = 0x40000000 | ((64 if lanes == 4 else 96) + waves - 1) << 20
    assert lib.qa_sscan_fwd(C.byref(p), None) == 0
def hadamard(dim, rows):
    p = _lib.QaHadamardParams()
    p.rows, p.dim, p.scale, p.x_row_stride, p.out_row_stride, p.x, p.out = rows, dim, 1.0, dim, dim, at, at
    assert lib.qa_hadamard_quant(C.byref(p), None) == 0
if sys.argv[3] == "scan":
    for lanes, waves in ((4, 12), (4, 8), (4, 3), (8, 16), (8, 13), (8, 12), (8, 8), (8, 5), (4, 12)): scan(lanes, waves)
else:
    for rows in (1, 1000):
        for dim in (32768, 16384, 24576, 20480, 32768): hadamard(dim, rows)
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no C++ compiler")
@pytest.mark.parametrize("calls", ["scan", "hadamard"])
def test_a_kernel_has_one_limit(tmp_path, calls):
    (tmp_path / "stand_ins.cpp").write_text(STAND_INS)
    built = str(tmp_path / "stand_ins.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(tmp_path / "stand_ins.cpp"), "-o", built], check=True)
    run = subprocess.run([sys.executable, "-c", CALLS, built, os.path.join(ROOT, "quamba_amd", "_lib.py"), calls], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    limits, launches = {}, {}
    for kind, kernel, value in re.findall(r"(limit|launch) (\S+) (\d+)", run.stdout):
        (limits if kind == "limit" else launches).setdefault(kernel, set()).add(int(value))
    large = {k: v for k, v in launches.items() if max(v) > 65536}
    assert large and any(len(v) > 1 for v in large.values())               # (kernels that are launched with one size and another)
    for kernel, sizes in large.items():
        assert len(limits[kernel]) == 1 and max(sizes) <= max(limits[kernel]) <= 160 * 1024, (limits[kernel], sizes)
