"""The LDS limit of a kernel, raised by two threads that launch it for the first time with different needs: the header's
host code compiled with a runtime of a few lines in which the larger limit is set first and its call returns last."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_RUNTIME = """
#pragma once
#include <stddef.h>
typedef int hipError_t;
typedef void* hipStream_t;
constexpr int hipSuccess = 0, hipDeviceAttributeMultiprocessorCount = 0, hipFuncAttributeMaxDynamicSharedMemorySize = 0;
inline int hipGetDevice(int* d) { *d = 0; return 0; }
inline int hipDeviceGetAttribute(int* n, int, int) { *n = 256; return 0; }
int hipFuncSetAttribute(const void*, int, int bytes);
"""

_PROGRAM = """
#include <chrono>
#include <cstdio>
#include <thread>
#include "kernels.h"
std::atomic<int> limit{0}, small_done{0};
int hipFuncSetAttribute(const void*, int, int bytes) {
  limit = bytes;
  if (bytes == 2000)  // the other thread gets its whole call in before this one returns, if it can
    for (int x = 0; x < 300 && !small_done; ++x) std::this_thread::sleep_for(std::chrono::milliseconds(1));
  return 0;
}
static mlstm::LdsLimit lds;
int main() {
  std::thread large([] { lds.allow(nullptr, 2000); });
  while (limit != 2000) std::this_thread::yield();
  std::thread small([] { lds.allow(nullptr, 1000); small_done = 1; });
  large.join();
  small.join();
  const bool allowed = lds.allow(nullptr, 2000);
  printf("allowed %d, limit %d\\n", (int)allowed, limit.load());
  return allowed && limit >= 2000 ? 0 : 1;
}
"""


def test_two_first_launches(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(_RUNTIME)
    (tmp_path / "main.cpp").write_text(_PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{ROOT}/mlstm_kernels_amd/csrc",
                    str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    run = subprocess.run([str(tmp_path / "main")], capture_output=True, text=True, timeout=30)
    assert run.returncode == 0, run.stdout
