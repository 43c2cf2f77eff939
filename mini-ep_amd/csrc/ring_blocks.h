// The blocks of K that ring_loop (ring_gemm.h) walks, in plain C++: a CPU test
// sweeps every index that the loop issues.
#pragma once

namespace mep {
namespace {
namespace ring {

constexpr int AHEAD = 2;                      // blocks (two K-steps) of loads in flight

// Block that load b of a loop over nb blocks reads, the walk starting at block
// rot < nb.  The loop issues loads up to b = nb + AHEAD - 1; those from nb on are
// not used, but must stay in the row: a row's next line may belong to rows that
// another workgroup is still writing, and a copy of it in the L1 would outlive
// the write.  b is wrapped before rot is added: with nb = 4 and rot = 3 the sum
// reaches 2 nb.
constexpr int block_at(int b, int rot, int nb) {
  const int at = (b >= nb ? b - nb : b) + rot;
  return at >= nb ? at - nb : at;
}

}  // namespace ring
}  // namespace
}  // namespace mep
