"""Settings made once per device (csrc/per_device.h), compiled for the CPU: one call for each device, another after a
failure, and every time for devices past the 64 that are remembered."""

from __future__ import annotations

import subprocess

from conftest import PACKAGE, ROOT

MAIN = r"""
#include <cstdio>
#include "per_device.h"
int main() {
  std::atomic<uint64_t> done{0};
  int calls = 0, status = 0;
  auto on = [&](int device) { return oxr::once_per_device(done, device, [&] { ++calls; return status; }); };
  auto show = [&](int result) { printf("%d:%d ", result, calls); };
  show(on(0)); show(on(0)); show(on(1)); show(on(1)); show(on(0));
  status = 7;
  show(on(2)); show(on(2)); show(on(1));
  status = 0;
  show(on(2)); show(on(2)); show(on(63)); show(on(63)); show(on(64)); show(on(64));
}
"""


def test_once_per_device(tmp_path) -> None:
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", f"-I{ROOT / PACKAGE / 'csrc'}", str(tmp_path / "main.cpp"), "-o",
                    str(tmp_path / "main")], check=True)
    out = subprocess.run([str(tmp_path / "main")], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["0:1", "0:1", "0:2", "0:2", "0:2", "7:3", "7:4", "0:4", "0:5", "0:5", "0:6", "0:6", "0:7", "0:8"]
