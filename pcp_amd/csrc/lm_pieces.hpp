// The K pieces of the cached LM-head backward's products: into how many each product is
// cut, and the room that they take. Host code without HIP, so it is tested on the CPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace pcp {

// The cached backward's dhidden has few, long tiles (one per 256 tokens x 256 hidden
// columns, K = the vocabulary: 2374 stages at V = 151,936), dW many short ones, so with
// few tokens a handful of CUs ran dhidden for milliseconds after dW was done: 288 live
// tokens at H = 896 took 2.89 ms for the launch, 8 CUs busy. A product whose tile is longer
// than half of a CU's even share of the launch is therefore cut along K into pieces of
// half that share (the share counts every token, and about half of them are live, so a
// piece is then a CU's live share), at least 16 stages (below that a piece's f32 tile
// costs more than its products). Each piece stores its own f32 partial tile, and the pieces
// are added in order, so results stay deterministic. Whole calls, ms, before and with
// pieces of 1/2, 1/4, 1/8 and 1/16 of the share (tokens x H x V):
//    64 x  256 x 151936  3.70 |  .254  .253  .254  .251
//   512 x  896 x 151936  3.39 |  .740  .745  .785  .800
//  1024 x 4096 x 151936  5.30 |  3.12  3.09  3.12  3.17
//  2048 x 2048 x  50257  1.70 |  1.02  1.03  1.07  1.14
//  4096 x  896 x 151936  4.60 |  2.60  2.63  2.65  2.70
// 16384 x  256 x   1000  .319 |  .165  .166  .165  .165   (here dW is the long one)
// Configuration 5 (its dhidden tiles are an eighth of the share) stays whole.
// K pieces per tile: `tiles` tiles of `stages` 64-deep stages each, in a launch whose other
// product adds `other` tile-stages (at all tokens).
inline int lm_ksplit(int64_t tiles, int64_t stages, int64_t other) {
  constexpr int64_t kCus = 256, kMin = 16;
  const int64_t share = (tiles * stages + other) / kCus;   // stages per CU, evenly dealt
  if (tiles <= 0 || 2 * stages <= share) return 1;
  const int64_t piece = share / 2 > kMin ? share / 2 : kMin;
  return static_cast<int>((stages + piece - 1) / piece);
}

// The pieces of a call of n tokens: dhidden's compact [n, H] f32 buffers one after the other,
// then dW's [V, H] ones. A tile's prologue and epilogue count as four stages.
struct LmPieces {
  int split_d = 1, split_w = 1;
  size_t d_bytes = 0, bytes = 0;   // dhidden's; both
};

inline LmPieces lm_pieces(int64_t n, int64_t H, int64_t V, bool want_d, bool want_w) {
  constexpr int64_t kTile = 256, kStage = 64;
  const int64_t nvt = (V + kTile - 1) / kTile, nht = (H + kTile - 1) / kTile, ntk = (n + kTile - 1) / kTile;
  const int64_t sd = (V + kStage - 1) / kStage + 4, sw = (n + kStage - 1) / kStage + 4;
  LmPieces p;
  if (want_d) p.split_d = lm_ksplit(ntk * nht, sd, want_w ? nvt * nht * sw : 0);
  if (want_w) p.split_w = lm_ksplit(nvt * nht, sw, want_d ? ntk * nht * sd : 0);
  if (p.split_d > 1) p.d_bytes = (4 * static_cast<size_t>(n) * H * p.split_d + 255) & ~static_cast<size_t>(255);
  p.bytes = p.d_bytes + (p.split_w > 1 ? 4 * static_cast<size_t>(V) * H * p.split_w : 0);
  return p;
}

// Room for the pieces of every call of up to n tokens (their number falls as n grows), so
// that a call of fewer tokens than the one before it needs no larger buffer.
inline size_t lm_pieces_room(int64_t n, int64_t H, int64_t V, bool want_d, bool want_w) {
  size_t room = 0;
  for (int64_t m = 64;; m += 64) {
    room = std::max(room, lm_pieces(std::min(m, n), H, V, want_d, want_w).bytes);
    if (m >= n) return room;
  }
}

// A grow-only buffer that a call can do without. A larger one is allocated before the held
// one is given up, so a refusal costs nothing that was held (captured graphs keep their
// pointers), and the refused size is remembered: later calls of that size or more allocate
// nothing and synchronise nothing (a call can be captured after one that was refused), and
// take the same route. reset() forgets both.
struct OptionalRoom {
  enum { kHeld = 0, kRefused = -1 };   // other values: the allocator's own error
  void* buf = nullptr;
  size_t bytes = 0;
  size_t refused = SIZE_MAX;   // the smallest size that was refused

  // alloc(size, &p): kHeld, kRefused or an error; retire(p): frees a buffer that earlier
  // calls may still use.
  template <typename Alloc, typename Retire>
  int have(size_t need, Alloc alloc, Retire retire) {
    if (need <= bytes) return kHeld;
    if (need >= refused) return kRefused;
    void* p = nullptr;
    const size_t want = (need + 0xFFFFF) & ~static_cast<size_t>(0xFFFFF);
    const int rc = alloc(want, &p);
    if (rc == kRefused) refused = need;
    if (rc != kHeld) return rc;
    if (buf) retire(buf);
    buf = p;
    bytes = want;
    return kHeld;
  }
  void reset() { *this = OptionalRoom{}; }
};

}  // namespace pcp
