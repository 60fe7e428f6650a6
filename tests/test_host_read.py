"""The pages that entry points read their counts back through (csrc/host_read.h), compiled for the host with a stand-in
for the device: a page goes back to the list only once its stream has been waited for, also where a call leaves early."""
import pathlib
import shutil
import subprocess

import pytest

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>
#include "host_read.h"

struct Stream { int waits = 0; bool fails = false; };
static std::set<void*> live;
static std::mutex m;
struct Fake {
  using Stream = ::Stream*;
  using Status = int;
  static constexpr int kDone = 0;
  static bool alloc(void** p) {
    std::lock_guard<std::mutex> lock(m);
    live.insert(*p = std::malloc(8));
    return true;
  }
  static void release(void* p) {
    std::lock_guard<std::mutex> lock(m);
    live.erase(p);
    std::free(p);
  }
  static int wait(::Stream* s) { ++s->waits; return s->fails ? 1 : 0; }
};
using Read = bf::PinnedRead<Fake>;
#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }

int main() {
  Stream s, broken;
  broken.fails = true;
  int* first;
  {
    Read r(&s);
    first = r.as<int>();
    CHECK(r.ok() && r.wait() == 0);
  }
  CHECK(s.waits == 1);                       // waited for once, by the call
  {
    Read r(&s);
    CHECK(r.as<int>() == first);             // the page came back
  }
  CHECK(s.waits == 2);                       // left early: waited for on the way out
  {
    Read r(&broken);
    CHECK(r.as<int>() == first);
    if (broken.waits < 0) r.wait();          // left early, and the stream cannot be waited for
  }
  CHECK(broken.waits == 1);
  {
    Read r(&broken);
    CHECK(r.as<int>() != first && r.wait() != 0);
  }
  {
    Read a(&s), b(&s);
    CHECK(a.as<int>() != first && b.as<int>() != first && a.as<int>() != b.as<int>());
  }
  std::vector<std::thread> threads;          // many calls in flight: the list keeps kHostPagesKept pages
  std::mutex gate;
  gate.lock();
  for (size_t i = 0; i < 2 * bf::kHostPagesKept; ++i)
    threads.emplace_back([&gate] {
      Stream own;
      Read r(&own);
      std::lock_guard<std::mutex> lock(gate);
      r.wait();
    });
  for (;;) {
    std::lock_guard<std::mutex> lock(m);
    if (live.size() >= 2 * bf::kHostPagesKept) break;
  }
  gate.unlock();
  for (auto& t : threads) t.join();
  CHECK(live.size() == bf::kHostPagesKept + 2);   // and the two pages never handed out again
  return 0;
}
"""


def test_pages_go_back_once_their_stream_is_waited_for(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    csrc = pathlib.Path(__file__).resolve().parents[1] / "budgetformer_amd" / "csrc"
    (tmp_path / "t.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-pthread", "-I", str(csrc), str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")],
                   check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
