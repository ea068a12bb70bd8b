"""The one-time kernel setup under several host threads (csrc/once.h, which
needs no HIP): compiled here as host code."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "once.h"

int main() {
  sj::OncePerDevice once;
  std::atomic<int> runs{0}, early{0}, wrong{0}, ready[2] = {{0}, {0}};
  std::vector<std::thread> threads;
  for (int t = 0; t < 16; t++)
    threads.emplace_back([&, t] {
      const int device = t & 1;
      const int status = once(device, [&] {
        runs++;
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        ready[device] = 1;
        return 7 + device;
      });
      if (!ready[device]) early++;
      if (status != 7 + device) wrong++;
    });
  for (auto& t : threads) t.join();
  for (int i = 0; i < 2; i++) once(1000, [&] { return runs++, 0; });  // past the table: every call
  printf("%d %d %d\n", runs.load(), early.load(), wrong.load());
}
"""


def test_nobody_passes_before_the_setup_is_done(tmp_path):
    src, exe = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "sejong_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    assert out == ["4", "0", "0"]  # once on each of two devices, twice past the table


def test_every_setup_goes_through_it():
    """No kernel source keeps a flag of its own that is set before its setup is done."""
    csrc = os.path.join(ROOT, "sejong_amd", "csrc")
    for name in sorted(os.listdir(csrc)):
        text = open(os.path.join(csrc, name)).read()
        assert "static int done" not in text, name
        if "hipFuncAttributeMaxDynamicSharedMemorySize" in text:
            assert "OncePerDevice" in text, name
