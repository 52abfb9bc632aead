"""elm_device_once.h, which raises a kernel's dynamic-LDS limit: once on every device (not once in the process), whichever
device comes first and however many threads call, and again where it failed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "elm_device_once.h"
#include <cstdio>
#include <thread>
#include <vector>

int main() {
  elmh::DeviceOnce once;
  std::atomic<int> ran[80];
  for (auto& r : ran) r = 0;
  bool ok = true;
  auto on = [&](int d, bool result) { return once.run(d, [&] { ++ran[d]; return result; }); };
  ok &= !on(3, false) && ran[3] == 1;  // refused: asked again
  ok &= on(3, true) && on(3, true) && ran[3] == 2;
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] {
      for (int i = 0; i < 200; ++i)
        for (int d = 0; d < 64; ++d) on(d, true);
    });
  for (auto& t : ts) t.join();
  for (int d = 0; d < 64; ++d) ok &= ran[d] == (d == 3 ? 2 : 1);
  ok &= on(70, true) && on(70, true) && ran[70] == 2;  // past the recorded devices: every call
  puts(ok ? "ok" : "bad");
  return !ok;
}
"""


def test_runs_once_on_every_device(tmp_path):
    src, exe = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "edgelm_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
