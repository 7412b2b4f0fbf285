// Which slab and which part of K a workgroup of the K-split slab GEMM takes
// (plain C++, no HIP: also compiled into a test on the CPU).
//
// Eight consecutive workgroups run on eight XCDs, from a first XCD that
// depends on the hardware queue, so workgroups 8 apart share an XCD: the parts
// of slab s are workgroups s % 8 + 8 (parts (s / 8) + q), q = 0 .. parts - 1.
// The place follows the workgroup's index and nothing else, so every part of
// every slab has a workgroup wherever the workgroups run.  Were a part on
// another XCD than part 0 of its slab, part 0 would not see its sums in its L2
// and its wait would give up, which the call reports.  (Taken from the XCC_ID
// register, two workgroups of one XCD had one place and another had none; with
// a part 0 among the missing nobody waited, and 16 outputs kept what the
// memory held.)
#pragma once

namespace hk {

constexpr int kPlaceXcds = 8;  // XCDs that consecutive workgroups go round

struct SlabPlace {
  int slab, part;
};

constexpr SlabPlace slab_place(int workgroup, int parts) {
  const int turn = workgroup / kPlaceXcds;
  return {workgroup % kPlaceXcds + kPlaceXcds * (turn / parts), turn % parts};
}

// Workgroups of a launch over `slabs` slabs (those past the last one leave).
constexpr int slab_places(int slabs, int parts) { return parts * kPlaceXcds * ((slabs + kPlaceXcds - 1) / kPlaceXcds); }

}  // namespace hk
