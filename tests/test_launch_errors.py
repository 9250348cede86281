"""A call any of whose kernels fails to launch reports it: every path of the linears and of the attention
entry points runs against a stand-in for HIP's launch functions (no device), with each of its launches
failing in turn."""

from __future__ import annotations

import json
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
LIBRARY = HERE.parent / "quantized-llm-inference-engine-_amd" / "llmopt" / "kernels" / "libllmopt_qlinear.so"

# The library is loaded in a process of its own, behind the stand-in, whose symbols come first there.
CHILD = r"""
import ctypes, json, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
launches, fail = (ctypes.c_int.in_dll(stub, "llmopt_stub_" + n) for n in ("launches", "fail"))
i64, i32, ptr, f32 = ctypes.c_int64, ctypes.c_int, ctypes.c_void_p, ctypes.c_float
size = ctypes.c_size_t
for name in ("llmopt_q_linear_workspace_ex", "llmopt_q_linear_swiglu_workspace_ex"):
    getattr(lib, name).restype = size
P = ptr(1 << 20)  # never read: nothing is launched
W = ptr(1 << 24)

def linear(m, n, k, act, bits, group, swiglu=False, symmetric=1, short=False):
    ws = lib.llmopt_q_linear_swiglu_workspace_ex if swiglu else lib.llmopt_q_linear_workspace_ex
    need = 0 if short else ws(i64(m), i64(n), i64(k), bits, group, act)
    f = lib.llmopt_q_linear_swiglu if swiglu else lib.llmopt_q_linear
    return f(P, i64(m), i64(k), i64(k), P, i64(k if bits == 8 else k // 2), P, None if symmetric else P, P, P, i64(n),
             i64(n // 2 if swiglu else n), act, bits, group, symmetric, 1 if bits == 8 and symmetric else 0,
             W if need else None, size(need), None)

def prefill(seqs, q_len, heads, kv, d):
    return lib.llmopt_paged_attention_prefill(
        P, 2, i64(q_len * heads * d), i64(heads * d), i64(d), P, P, 2, i64(64), i64(16), i64(kv), i64(d), P, i64(8), P,
        i64(seqs), i64(heads), i64(q_len), f32(1), f32(0), P, i64(q_len * heads * d), i64(heads * d), i64(d), None)

case = json.loads(sys.argv[3])
call = lambda: globals()[case[0]](*case[1])
rc = call()
total = launches.value
got = []
for at in range(1, total + 1):
    launches.value, fail.value = 0, at
    got.append(call())
fail.value = 0
print(json.dumps({"rc": rc, "launches": total, "failed": got, "after": call()}))
"""

CASES = {  # name: (call, arguments, launches)
    "one decode launch": ("linear", [1, 4096, 4096, 2, 4, 128], 1),
    "K slices and their reduction": ("linear", [16, 4096, 14336, 2, 4, 128], 2),
    "byte codes in K slices": ("linear", [16, 4096, 14336, 1, 8, 128], 2),
    "GEMM, split K, bf16": ("linear", [300, 4096, 14336, 2, 4, 128], 2),
    "GEMM, split K, fp16": ("linear", [300, 4096, 14336, 1, 4, 128], 2),
    "GEMM, split K, bytes": ("linear", [300, 4096, 14336, 2, 8, 128], 2),
    "GEMM, split K, groups of 64": ("linear", [300, 4096, 4096, 1, 4, 64], 2),
    "GEMM, split K, SwiGLU in the reduction": ("linear", [100, 2048, 4096, 2, 4, 128, True], 2),
    "GEMM, whole K": ("linear", [600, 28672, 4096, 2, 4, 128], 1),
    "GEMM, SwiGLU": ("linear", [300, 28672, 4096, 1, 4, 128, True], 1),
    "fp32 GEMM, split K": ("linear", [24, 6144, 4096, 0, 4, 64], 3),
    "fp32 GEMM, SwiGLU": ("linear", [1536, 28672, 4096, 0, 4, 64, True], 2),
    "fp32 decode pieces": ("linear", [4, 4096, 14336, 0, 4, 64], None),
    "generic": ("linear", [5, 7, 12, 2, 4, 12], 1),
    "prefill attention": ("prefill", [2, 100, 8, 2, 128], 1),
}


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    cc = shutil.which("cc") or shutil.which("gcc")
    if cc is None:
        pytest.skip("no C compiler")
    out = tmp_path_factory.mktemp("stub") / "libhip_launch_stub.so"
    subprocess.run([cc, "-shared", "-fPIC", "-O1", str(HERE / "hip_launch_stub.c"), "-o", str(out)], check=True)
    return out


@pytest.mark.parametrize("name", CASES)
def test_a_failed_launch_is_reported(stub, name):
    call, args, launches = CASES[name]
    proc = subprocess.run([sys.executable, "-c", CHILD, str(stub), str(LIBRARY), json.dumps([call, args])],
                          capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0, proc.stderr[-2000:]
    got = json.loads(proc.stdout.splitlines()[-1])
    assert got["rc"] == 0 and got["launches"] >= 1 and got["after"] == 0
    if launches is not None:
        assert got["launches"] == launches
    assert all(rc != 0 for rc in got["failed"]), got
