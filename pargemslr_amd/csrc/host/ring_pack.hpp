// Layout of a ring-packed level (TrsvPack with window > 0) as the ring kernel
// reads it: the packing's slabs turned into step boundaries, lane records,
// (slot, row id) pairs and pivots by position.  Plain host code, templated over
// the value that the device holds (4, 8 or 16 bytes), so that the upload and
// the host replay (tests/cpp/ring_check.cpp) share it.
//
// Factor entries.  A row takes four lanes, a lane five
// entries: entry j of the row is entry j / 4 of lane j % 4.  A lane's record is
// its five values and five 16-bit ring slots, cut into pieces of at most 16
// bytes:
//   4-byte values   [v0 v1 v2 v3] [v4 s01 s23 s4]
//   8-byte values   [v0 v1] [v2 v3] [v4 s01 s23] [s4]
//   16-byte values  [v0] [v1] [v2] [v3] [v4] [s01 s23 s4 -]
// (s01: slots 0 and 1 in one word).  The rows of a step are cut into groups of
// 16 (the rows of one wave); a group of n rows at position p starts at byte
// p * ring_row_bytes<V>() of its block and holds piece 0 of its 4 n lanes, then
// piece 1, ...: every copy of a wave is one contiguous run of memory at a
// wave-uniform base, and lands in LDS as the solving lanes read it.
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <vector>

#include "csr.hpp"
#include "trsv_pack.hpp"

namespace pgs {

constexpr int kRingWidth = 20;  // entries of a row's records
constexpr int kRingGroup = 16;  // rows of a group

template <typename V>
constexpr int ring_row_bytes() {
  return 4 * (5 * (int)sizeof(V) + (sizeof(V) == 16 ? 16 : 12));
}

constexpr int kRingOut = 0x7ffffff0;  // a byte offset past every resource of the ring kernel

// The ring kernel addresses a block's rows of all columns, its records (two
// positions per row) and, both shorter, its pairs and step boundaries with 32-bit
// byte offsets; lanes with nothing to load or store aim at offset kRingOut, which
// must stay past each of them.  A level may hold any number of such blocks.
template <typename V>
constexpr bool ring_offsets_fit(int64_t max_block_rows, int nrhs) {
  return max_block_rows * nrhs * (int64_t)sizeof(V) <= kRingOut && 2 * max_block_rows * ring_row_bytes<V>() <= kRingOut;
}

// The row id of the dummy row: shifted by 2 to 10 bits it is a byte offset past
// every resource.
constexpr int kRingDummyRow = 0x3fe00000;

// A position's ring slot (times the size of a value) and block-local row id.
struct RingInfo {
  int slot, row;
};

// Index of a block's first pair, ri0 its first position: the blocks' pairs lie two
// apart.  A block has an even number of positions, so that each block's pairs start
// at a multiple of 16 bytes (one pair apart, an apply at 1023x1021 x 8 columns took
// 1436 us, like this 1427 to 1430).
constexpr int64_t ring_info0(int64_t ri0, int64_t b) { return ri0 + 2 * b; }

// Byte of entry j of row t in a group of n rows: its value's and its slot's.
template <typename V>
void ring_entry_bytes(int n, int t, int j, int& value, int& slot) {
  const int lane = 4 * t + j % 4, e = j / 4;
  int s01, s4;  // the words of slots 0 and 1 and of slot 4
  if constexpr (sizeof(V) == 4) {
    const int b = n * 64 + lane * 16;
    value = e < 4 ? lane * 16 + e * 4 : b;
    s01 = b + 4;
    s4 = b + 12;
  } else if constexpr (sizeof(V) == 8) {
    value = (e / 2) * n * 64 + lane * 16 + (e % 2) * 8;
    s01 = n * 128 + lane * 16 + 8;
    s4 = n * 192 + lane * 4;
  } else {
    value = e * n * 64 + lane * 16;
    s01 = n * 320 + lane * 16;
    s4 = s01 + 8;
  }
  slot = e < 4 ? s01 + 2 * e : s4;
}

template <typename V>
struct RingPack {
  int rows = 0;                         // slots of a ring: position p is in slot p % rows
  // Boundaries of the whole steps: blk_step[b + 1] - blk_step[b] + 1 values per
  // block, from blk_step[b] + b; the first of them is 0.
  std::vector<int> pos;
  // The same for half steps (half_steps) with their own step ranges.
  std::vector<int> pos_h, step_h, stepU_h;
  int64_t max_block_steps = 0, max_block_steps_h = 0;
  std::vector<unsigned char> rec;       // records, ring_row_bytes<V>() per position
  std::vector<RingInfo> info;           // per position, and two of the dummy row after a block's last
};

// Step boundaries of every block from the step descriptors (4 per step, the
// first position at 0 and the rows at 2).
inline std::vector<int> step_bounds(const std::vector<int>& desc, const std::vector<int>& blk_step) {
  const int nb = (int)blk_step.size() - 1;
  std::vector<int> pos((size_t)blk_step[nb] + nb);
  for (int b = 0; b < nb; ++b) {
    int* q = pos.data() + blk_step[b] + b;
    int end = 0;
    for (int s = blk_step[b]; s < blk_step[b + 1]; ++s) {
      *q++ = desc[4 * s];
      end = desc[4 * s] + desc[4 * s + 2];
    }
    *q = end;
  }
  return pos;
}

// val(x): the device's value of the packing's.
template <typename V, typename T, typename F>
RingPack<V> ring_pack(const TrsvPack<T>& P, F val) {
  RingPack<V> R;
  // the packed slots are positions modulo a power of two; the device's ring
  // holds just the rows needed (a fifth less LDS at 128^3: room for more
  // columns or stages): slot = position modulo those
  const int W = P.window, wn = std::max(P.window_needed, 1);
  if (wn > 0xffff) throw std::runtime_error("sweep window too large for 16-bit slots");
  R.rows = wn;
  R.pos = step_bounds(P.desc, P.blk_step);
  std::vector<int> dh;
  half_steps(P.desc, P.blk_step, P.blk_stepU, dh, R.step_h, R.stepU_h);
  R.pos_h = step_bounds(dh, R.step_h);
  for (int b = 0; b < P.nblocks; ++b) {
    R.max_block_steps = std::max<int64_t>(R.max_block_steps, P.blk_step[b + 1] - P.blk_step[b]);
    R.max_block_steps_h = std::max<int64_t>(R.max_block_steps_h, R.step_h[b + 1] - R.step_h[b]);
  }
  constexpr int RB = ring_row_bytes<V>();
  const int64_t nr = (int64_t)P.rows.size();
  R.rec.resize((size_t)nr * RB);
  R.info.resize((size_t)ring_info0(nr, P.nblocks), RingInfo{wn * (int)sizeof(V), kRingDummyRow});
  parallel_for(P.nblocks, [&](int b) {
    for (int s = P.blk_step[b]; s < P.blk_step[b + 1]; ++s) {
      const int* d4 = &P.desc[4 * (size_t)s];
      const int end = d4[0] + d4[2];  // a row the step reads is at most W positions before it
      for (int t = 0; t < d4[2]; ++t) {
        const int64_t q = P.blk_ri0[b] + d4[0] + t;
        R.info[ring_info0(q, b)] = RingInfo{(d4[0] + t) % wn * (int)sizeof(V), P.rows[q]};
        const int t0 = t / kRingGroup * kRingGroup;  // first row of t's group
        unsigned char* g = R.rec.data() + (P.blk_ri0[b] + d4[0] + t0) * RB;
        for (int j = 0; j < d4[3]; ++j) {
          const int64_t e = P.blk_ent0[b] + d4[1] + (int64_t)t * d4[3] + j;
          // (padded entries weigh zero, whatever row they name)
          const int p = std::max(0, end - 1 - ((end - 1 - P.col[e]) & (W - 1)));
          const V v = val(P.val[e]);
          const uint16_t slot = (uint16_t)(p % wn);
          int bv, bs;
          ring_entry_bytes<V>(std::min(kRingGroup, d4[2] - t0), t - t0, j, bv, bs);
          std::memcpy(g + bv, &v, sizeof(V));
          std::memcpy(g + bs, &slot, sizeof(slot));
        }
      }
    }
  });
  return R;
}

}  // namespace pgs
