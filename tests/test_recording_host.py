"""What a graph recording refuses (no GPU).

Growing a buffer or reading a count back while a stream records would free
memory that recorded kernels use, or spoil the recording: both are refused
before any runtime call.
"""
from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "chui-dev_amd" / "csrc"
HIPCC = shutil.which("hipcc") or shutil.which("hipcc", path="/opt/rocm/bin")

PROGRAM = r"""
#include "common.hpp"
#include <cstdio>
template <class F> bool refused(F f) {
  try { f(); } catch (const std::logic_error&) { return true; } catch (...) {}
  return false;
}
int main() {
  chui::DeviceBuffer b;
  char memory[64];
  b.ptr = memory;  // stands for memory that recorded kernels use
  b.bytes = sizeof(memory);
  chui::PinnedReadback r;
  char host[8];
  bool ok = true;
  {
    const chui::RecordingScope outer(true);
    ok = ok && !refused([&] { b.reserve(64); });
    ok = ok && refused([&] { b.reserve(65); }) && b.ptr == memory && b.bytes == 64;
    { const chui::RecordingScope inner(false); ok = ok && refused([&] { b.reserve(65); }); }
    ok = ok && refused([&] { r.read(host, memory, 8, nullptr); }) && r.ptr == nullptr;
  }
  ok = ok && !chui::t_recording;
  b.ptr = nullptr;
  std::puts(ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
"""


@pytest.mark.skipif(HIPCC is None, reason="hipcc is not installed")
def test_buffers_neither_grow_nor_read_back_while_recording(tmp_path):
    src = tmp_path / "recording.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "recording"
    subprocess.run([HIPCC, "--offload-host-only", "-x", "hip", "-std=c++20", "-O1", f"-I{CSRC}", str(src), "-o",
                    str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout.strip() == "ok"
