"""sma_abi::OncePerDevice, compiled for the host: a setting is made once for each
device, not once for the process, again after a failure, and by every device
beyond the 64 it remembers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "once_per_device.hpp"
#include <cstdio>
#include <thread>
#include <vector>
int main() {
  sma_abi::OncePerDevice once;
  std::atomic<int> made[70] = {};
  auto use = [&](int dev, int rc) { return once(dev, [&] { ++made[dev]; return rc; }); };
  int bad = use(2, 7) != 7;                     // a failure is not remembered
  for (int k = 0; k < 3; ++k)
    for (int dev : {0, 1, 2, 63, 64}) bad += use(dev, 0) != 0;
  bad += made[0] != 1 || made[1] != 1 || made[2] != 2 || made[63] != 1 || made[64] != 3;
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] { for (int k = 0; k < 1000; ++k) for (int dev = 3; dev < 20; ++dev) use(dev, 0); });
  for (auto& t : ts) t.join();
  for (int dev = 3; dev < 20; ++dev) bad += made[dev] < 1 || made[dev] > 8;
  std::printf("%d\n", bad);
  return bad != 0;
}
'''


def test_once_for_each_device(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    (tmp_path / "o.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I" + os.path.join(ROOT, "alya_sma_amd", "csrc"),
                    str(tmp_path / "o.cpp"), "-o", str(tmp_path / "o")], check=True)
    assert subprocess.run([str(tmp_path / "o")]).returncode == 0


def test_no_setting_is_kept_for_the_process():
    """The library's calls of hipFuncSetAttribute, whose limits hold for one
    device, are made through OncePerDevice."""
    text = open(os.path.join(ROOT, "alya_sma_amd", "csrc", "surrogate.hip")).read()
    assert "static bool" not in text
    assert text.count("hipFuncSetAttribute(") == 1
