"""sma_abi::StagePool (the host stages of sma160_eval and read-back between
calls), compiled for the host with a stage that counts: as many callers as came
at once find their stages again, on each of several devices, within the limits of
stages and bytes."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "stage_pool.hpp"
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
std::atomic<int> made{0}, ended{0}, dropped{0};
struct Stage {
  int device;
  size_t bytes = 0;
  Stage* next = nullptr;
  std::atomic<int> users{0};
  explicit Stage(int d) : device(d) { ++made; }
  void drop_block() { bytes = 0; ++dropped; }
};
using Pool = sma_abi::StagePool<Stage>;
Stage* lease(Pool& p, int dev, size_t want) {
  Stage* s = p.take(dev);
  if (!s) s = new Stage(dev);
  if (s->bytes < want) s->bytes = want;
  return s;
}
void back(Pool& p, Stage* s) {
  if (!p.give(s)) { ++ended; delete s; }
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d\n", __LINE__); return 1; } } while (0)
// `n` callers at once on each of `devs` devices
void round(Pool& p, int n, int devs, size_t want) {
  std::vector<Stage*> v;
  for (int k = 0; k < n; ++k)
    for (int d = 0; d < devs; ++d) v.push_back(lease(p, d, want));
  for (Stage* s : v) back(p, s);
}
int main() {
  Pool p(64, 1000);
  CHECK(p.take(0) == nullptr);
  round(p, 12, 3, 8);
  CHECK(made == 36 && ended == 0 && dropped == 0);
  for (int k = 0; k < 5; ++k) round(p, 12, 3, 8);
  CHECK(made == 36 && ended == 0 && dropped == 0);
  round(p, 70, 1, 0);                         // beyond the limit of a device
  CHECK(made == 36 + 58 && ended == 6);
  round(p, 2, 8, 8);                          // the others are not pushed out
  CHECK(made == 36 + 58 + 10 && ended == 6);
  Pool q(4, 100);
  made = ended = dropped = 0;
  Stage *a = lease(q, 0, 60), *b = lease(q, 0, 60), *c = lease(q, 1, 500), *e = lease(q, 1, 40);
  back(q, a);
  back(q, b);                                 // 120 bytes: kept without its block
  CHECK(dropped == 1 && ended == 0 && b->bytes == 0);
  back(q, c);                                 // larger than all that may be kept
  CHECK(dropped == 2 && ended == 0 && c->bytes == 0);
  back(q, e);
  CHECK(dropped == 2 && e->bytes == 40);
  CHECK(q.take(0) == b && q.take(0) == a && q.take(0) == nullptr && q.take(1) == e);
  back(q, b);
  b->bytes = 0;
  Pool t(64, 1 << 20);
  made = ended = 0;
  std::atomic<int> shared{0};
  std::vector<std::thread> ts;
  for (int k = 0; k < 8; ++k)
    ts.emplace_back([&, k] {
      for (int i = 0; i < 20000; ++i) {
        Stage* s = lease(t, k & 1, 16);
        if (s->users.fetch_add(1) || s->device != (k & 1)) ++shared;
        s->users.fetch_sub(1);
        back(t, s);
      }
    });
  for (auto& x : ts) x.join();
  CHECK(shared == 0 && made <= 8 && ended == 0);
  return 0;
}
'''


def test_pool(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    (tmp_path / "p.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I" + os.path.join(ROOT, "alya_sma_amd", "csrc"),
                    str(tmp_path / "p.cpp"), "-o", str(tmp_path / "p")], check=True)
    r = subprocess.run([str(tmp_path / "p")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
