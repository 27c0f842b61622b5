"""CPU check that a launch the runtime refuses is reported with its reason:
the library runs in a process whose HIP launch calls are a counting stub."""

from __future__ import annotations

import subprocess
import sys

import pytest

from conftest import submodule

# hipLaunchKernel number FAIL_AT (from 1) leaves hipErrorOutOfMemory; hipGetLastError returns and clears it.
STUB = r"""
#include <stddef.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3;
static struct { dim3 grid, block; size_t shared; void* stream; } pushed;
static int launches, last;
int fail_at, *launch_count = &launches;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, void* stream) {
  pushed.grid = grid, pushed.block = block, pushed.shared = shared, pushed.stream = stream;
  return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, void** stream) {
  *grid = pushed.grid, *block = pushed.block, *shared = pushed.shared, *stream = pushed.stream;
  return 0;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t shared, void* stream) {
  if (++launches == fail_at) last = 2;
  return last;
}
int hipGetLastError(void) {
  int e = last;
  last = 0;
  return e;
}
"""

# 300 rows x 4096 columns run on the grouped GEMM, which needs the weight's
# code flag: split, clear the flag, scan, product.  No address is followed.
CALL = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
ctypes.c_int.in_dll(stub, "fail_at").value = int(sys.argv[3])
lib = ctypes.CDLL(sys.argv[2])
I, P, Z = ctypes.c_int64, ctypes.c_void_p, ctypes.c_size_t
lib.glm53_fp8_linear.argtypes = [P, I, I, P, I, P, P, P, P, Z, P]
lib.glm53_last_error.restype = ctypes.c_char_p
status = lib.glm53_fp8_linear(4096, 300, 128, 4096, 4096, 4096, None, 4096, 4096, 1 << 30, None)
print(status, ctypes.cast(P.in_dll(stub, "launch_count"), ctypes.POINTER(ctypes.c_int))[0])
print(lib.glm53_last_error().decode())
"""


@pytest.mark.parametrize("fail_at,what", [(1, "split launch"), (2, "scan launch"), (3, "scan launch"),
                                          (4, "grouped gemm launch")])
def test_refused_launches_of_the_several_row_linear_keep_their_reason(tmp_path, fail_at, what):
    N = submodule("_native")
    (tmp_path / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", tmp_path / "stub.so", tmp_path / "stub.c"], check=True)
    run = subprocess.run([sys.executable, "-c", CALL, tmp_path / "stub.so", N.LIB_PATH, str(fail_at)], check=True,
                         capture_output=True, text=True)
    counts, message = run.stdout.splitlines()
    assert counts.split() == [str(N.DEVICE_ERROR), str(max(fail_at, 3) if what == "scan launch" else fail_at)]
    assert message == f"{what}: out of memory"
