"""The room for the LM-head products' K pieces (pcp_amd/csrc/lm_pieces.hpp), compiled and run on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "lm_pieces.hpp"
using namespace pcp;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  // A warm-up of n tokens leaves room for every call of fewer tokens, also where a smaller
  // call is cut into more pieces.
  const int64_t shapes[][2] = {{256, 20000}, {896, 151936}, {2048, 50257}, {256, 1000}, {64, 130}, {4096, 151936}};
  for (auto& s : shapes)
    for (int want = 1; want < 4; ++want) {
      size_t most = 0;
      for (int64_t n = 1; n < 5000; ++n) {
        const LmPieces p = lm_pieces(n, s[0], s[1], want & 1, want & 2);
        CHECK(p.split_d >= 1 && p.split_w >= 1 && ((want & 1) || p.split_d == 1) && ((want & 2) || p.split_w == 1));
        if (p.bytes > most) most = p.bytes;
        if (n % 61 == 0 || n % 64 < 2) CHECK(lm_pieces_room(n, s[0], s[1], want & 1, want & 2) >= most);
      }
    }
  CHECK(lm_pieces(4352, 256, 20000, true, true).bytes > lm_pieces(4353, 256, 20000, true, true).bytes);

  // An allocator with a limit per allocation: what is held, and what was asked of it.
  std::set<void*> live;
  size_t limit = 8 << 20;
  int asked = 0, fault = 0;
  auto alloc = [&](size_t want, void** p) -> int {
    ++asked;
    if (fault) return fault;
    if (want > limit) return OptionalRoom::kRefused;
    live.insert(*p = std::malloc(want));
    return OptionalRoom::kHeld;
  };
  auto retire = [&](void* p) { live.erase(p); std::free(p); };
  OptionalRoom r;
  CHECK(r.have(0, alloc, retire) == OptionalRoom::kHeld && asked == 0);
  CHECK(r.have(3 << 20, alloc, retire) == OptionalRoom::kHeld && asked == 1);
  void* held = r.buf;
  // A refused size frees nothing, and is not asked for again.
  for (int i = 0; i < 3; ++i) {
    CHECK(r.have(9 << 20, alloc, retire) == OptionalRoom::kRefused && asked == 2);
    CHECK(r.have(20 << 20, alloc, retire) == OptionalRoom::kRefused && asked == 2);
    CHECK(r.buf == held && live.count(held) && r.bytes == size_t(3) << 20);
    CHECK(r.have(2 << 20, alloc, retire) == OptionalRoom::kHeld && asked == 2);
  }
  // A size between the held and the refused one may still grow; the old buffer then goes.
  CHECK(r.have(5 << 20, alloc, retire) == OptionalRoom::kHeld && asked == 3);
  CHECK(r.buf != held && live.size() == 1 && live.count(r.buf));
  // An error is passed on and is not taken for a refusal.
  fault = 77;
  held = r.buf;
  CHECK(r.have(6 << 20, alloc, retire) == 77 && r.buf == held && r.refused == size_t(9) << 20);
  fault = 0;
  CHECK(r.have(6 << 20, alloc, retire) == OptionalRoom::kHeld);
  retire(r.buf);
  r.reset();
  limit = 64 << 20;
  CHECK(r.buf == nullptr && r.have(9 << 20, alloc, retire) == OptionalRoom::kHeld);
  retire(r.buf);
  std::puts("ok");
  return 0;
}
"""


def test_room_for_k_pieces(tmp_path):
    src, exe = tmp_path / "pieces.cpp", tmp_path / "pieces"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "pcp_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
