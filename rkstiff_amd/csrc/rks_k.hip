// Persistent stepping kernels of one precision, nonlinearity and method: every grid size,
// tile and proposer variant that exists for them.  Compiled once per combination with
//   RKS_R, RKS_RN   state / FFT and NL storage precision (double or float)
//   RKS_NLK         NLK_ADVECT, NLK_CUBIC or NLK_HANKEL
//   RKS_METH        a method id, or RKS_METH_ANY
//   RKS_TABLE       the name of this unit's lookup function
// The proposer variant exists for the sizes whose workgroups can be whole waves (n >= 128;
// the host refuses smaller rfft grids), the second tile for n = 2^9 .. 2^12, with and
// without the proposer.  Without it also (rks_host.hip default_tile) twice the threads for
// the cubic n = 2^13, four times for n = 2^10 and the cubic n = 2^11.  The Hankel kind has the
// size classes 2^4 .. 2^10 and one tile.
#include "rks_kernels.h"

namespace {

template <int LOG2N, bool LEARN, int TILE>
bool entry_of(rks_kernel_entry* e) {
  constexpr int T = rks_threads(LOG2N, RKS_NLK) << TILE;
  e->fn = (const void*)&rks_kernel<RKS_R, RKS_RN, LOG2N, RKS_NLK, LEARN, TILE, RKS_METH>;
  e->threads = T;
  e->lds = rks_lds_bytes<RKS_R, LOG2N, T, RKS_NLK>();
  return true;
}

// the sizes LO..HI
template <int LO, int HI, bool LEARN, int TILE>
bool find(int log2n, rks_kernel_entry* e) {
  if constexpr (LO > HI) {
    return false;
  } else {
    return log2n == LO ? entry_of<LO, LEARN, TILE>(e) : find<LO + 1, HI, LEARN, TILE>(log2n, e);
  }
}

}  // namespace

bool RKS_TABLE(int log2n, bool learn, int tile, rks_kernel_entry* e) {
  if constexpr (RKS_NLK == NLK_HANKEL) {
    return !learn && tile == 0 && find<4, 10, false, 0>(log2n, e);
  } else {
    if (tile == 1)
      return learn ? find<9, 12, true, 1>(log2n, e) : find<9, RKS_NLK == NLK_CUBIC ? 13 : 12, false, 1>(log2n, e);
    if (tile == 2) return !learn && find<10, RKS_NLK == NLK_CUBIC ? 11 : 10, false, 2>(log2n, e);
    if (tile != 0) return false;
    return learn ? find<7, 13, true, 0>(log2n, e) : find<4, 13, false, 0>(log2n, e);
  }
}
