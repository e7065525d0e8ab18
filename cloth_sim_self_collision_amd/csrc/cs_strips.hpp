// Strip plan of the triangular sweeps: the rows cut into contiguous strips,
// each swept by one wave (cs_strips.hip), with everything a wave reads laid
// out in the order it reads it.  Host-only; built from the mesh's pattern and
// level schedules when a cloth is created.
#pragma once

#include <string>
#include <vector>

#include "cs_setup.hpp"

namespace cs {

constexpr int kStripRows = 8;       // rows per sub-level of a strip (eight lanes each)
constexpr int kStripImports = 16;   // rows imported beside a sub-level at most (four lanes each)
constexpr int kStripMaxRing = 32;   // sub-levels of the LDS ring at most (16-bit offsets)
constexpr int kStripGroup = 4;      // a strip's sub-levels are padded to a multiple of this
constexpr int kStripTail = 8;       // empty sub-levels after the last strip (read ahead)
constexpr int kStripZero = 32;      // LDS bytes before the ring: an entry that holds +0.0
constexpr int kStripEntry = 32;     // bytes of a row's ring entry (three components, one unused)
// ring bytes per sub-level: the rows, imports 0, 2, .., 14, entries that the lanes
// without a result write, imports 1, 3, .., 15
constexpr int kStripSub = 4 * kStripRows * kStripEntry;
constexpr unsigned kStripNone = 0xffffffffu;  // offset of a lane without a store or an import

// One sweep direction.  Strip s owns the sub-levels ptr[s] .. ptr[s + 1] - 1;
// slot = sub-level * kStripRows + row within it.
struct StripSweep {
  std::vector<int> ptr;
  int nsub = 0;                   // sub-levels of all strips, without the tail
  std::vector<int> row;           // row of each slot, -1: none
  std::vector<int> slot;          // slot of each row
  // per slot and block: LDS offset of the column row's entry (the zero entry
  // past the row's blocks)
  std::vector<unsigned short> col;
  // kStripImports per sub-level: the rows imported beside it (from strips
  // swept before this one), -1: none
  std::vector<int> import;
};

struct StripPlan {
  bool ok = false;
  int k = 0;      // blocks per row of both sweeps (the packed width)
  int ring = 0;   // sub-levels in the LDS ring, a power of two
  StripSweep fwd, bwd;
};

// Strips of s, or ok = false when the mesh does not fit the layout (more than
// kStripImports imports in reach of a sub-level, a dependency further back than
// the ring, rows too wide for the packed sweeps).
void build_strips(const MeshSetup& s, StripPlan& p);

// Walks both sweeps strip by strip with the ring as the wave would keep it
// and checks that every block of every row reads its column row's entry,
// written earlier; empty string when it holds.
std::string validate_strips(const MeshSetup& s, const StripPlan& p);

}  // namespace cs
