"""Who shares a scratch block (tessera_amd/csrc/stream_scratch.hpp): nobody but the launches of one owner,
which is a stream's eager launches or one capture's launches on one stream.  The header has no HIP in it
and is run here as a small C++ program."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include <utility>
#include <vector>
#include "stream_scratch.hpp"
using qmm::ScratchBlock;
using qmm::StreamScratch;

static unsigned char* const kBase = reinterpret_cast<unsigned char*>(uintptr_t{1} << 40);
static size_t taken = 0;
static bool closed = false;
static void* grow(size_t n) {
  if (closed) return nullptr;
  void* p = kBase + taken;
  taken += n;
  return p;
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

int main() {
  static StreamScratch s;
  const size_t MB = 1 << 20;
  auto stream = [](uintptr_t i) { return reinterpret_cast<const void*>(i * 64); };
  CHECK(s.reserve(grow) && taken == StreamScratch::kFirstSlab && s.reserve(grow) && taken == StreamScratch::kFirstSlab);
  ScratchBlock* a = s.find(0, stream(0), 5 * MB, grow);            // the null stream is an owner like any other
  ScratchBlock* b = s.find(0, stream(1), MB, grow);
  CHECK(a && b && a != b && a->bytes == StreamScratch::kSmallBlock);
  CHECK(s.find(0, stream(0), 16 * MB, grow) == a && s.find(0, stream(1), 1, grow) == b);
  ScratchBlock* large = s.find(0, stream(0), 16 * MB + 1, grow);   // besides the small one
  CHECK(large && large != a && large->bytes == StreamScratch::kBlockBytes && s.find(0, stream(0), 128 * MB, grow) == large);
  CHECK(s.find(0, stream(0), 128 * MB + 1, grow) == nullptr);
  // captures: own blocks, also on a stream that has an eager one; a larger need, another block
  ScratchBlock* c = s.find(7, stream(1), 3 * MB, grow);
  ScratchBlock* d = s.find(7, stream(2), 3 * MB, grow);
  ScratchBlock* e = s.find(8, stream(1), 3 * MB, grow);
  CHECK(c && d && e && s.find(7, stream(1), 2 * MB, grow) == c);
  ScratchBlock* f = s.find(7, stream(1), 4 * MB, grow);
  CHECK(f && f != c && s.find(7, stream(1), 4 * MB, grow) == f);
  std::vector<ScratchBlock*> all{a, b, large, c, d, e, f};
  // a caller's workspace is set: what was reserved is still given out, nothing is allocated
  closed = true;
  for (uintptr_t i = 3;; ++i) {
    ScratchBlock* more = s.find(0, stream(i), MB, grow);
    if (more == nullptr) break;
    all.push_back(more);
    CHECK(all.size() < 100);
  }
  CHECK(taken == StreamScratch::kFirstSlab && s.find(0, stream(1), MB, grow) == b);
  closed = false;
  // a block that needs a slab of its own leaves the rest of the last one to others
  ScratchBlock* whole = s.find(0, stream(900), 100 * MB, grow);
  CHECK(whole && taken == StreamScratch::kFirstSlab + StreamScratch::kSlab);
  all.push_back(whole);
  // and without one no more than the bound, however many owners ask
  for (uintptr_t i = 1000; i < 20000; ++i) {
    ScratchBlock* more = i % 2 ? s.find(0, stream(i), MB, grow) : s.find(i, stream(5), 700000, grow);
    if (more != nullptr) all.push_back(more);
  }
  CHECK(taken <= StreamScratch::kMaxBytes && taken > StreamScratch::kMaxBytes - StreamScratch::kSlab);
  std::set<std::pair<unsigned char*, unsigned char*>> spans;
  for (ScratchBlock* x : all) {
    unsigned char* p = static_cast<unsigned char*>(x->ptr);
    CHECK(p >= kBase && p + x->bytes <= kBase + taken && (p - kBase) % 256 == 0);
    CHECK(spans.insert({p, p + x->bytes}).second);
  }
  unsigned char* last = nullptr;
  for (const auto& x : spans) {
    CHECK(x.first >= last);
    last = x.second;
  }
  std::printf("%zu blocks\n", all.size());
  // limits of its own: another pool with small blocks, used up by captures, and what is given out still found
  static StreamScratch small({MB, MB, 64 << 10, 4 * MB, 4 * MB, 8 * MB});
  taken = 0;
  CHECK(small.reserve(grow) && taken == 4 * MB && small.find(0, stream(1), MB + 1, grow) == nullptr);
  ScratchBlock* eager = small.find(0, stream(1), 100, grow);
  ScratchBlock* first = small.find(1, stream(1), 100, grow);
  CHECK(eager && eager->bytes == MB && first && first->bytes == 64 << 10);
  size_t given = 0;
  for (uint64_t i = 2; i < 1000; ++i) given += small.find(i, stream(1), 100, grow) != nullptr;
  CHECK(given == (7 * MB) / (64 << 10) - 1 && taken == 8 * MB);
  CHECK(small.find(1, stream(1), 64 << 10, grow) == first && small.find(0, stream(1), MB, grow) == eager);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_every_owner_has_a_block_of_its_own(tmp_path):
    src, exe = tmp_path / "scratch.cpp", tmp_path / "scratch"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Wextra", "-I" + os.path.join(ROOT, "tessera_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True, capture_output=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
