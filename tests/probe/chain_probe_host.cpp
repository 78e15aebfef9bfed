// Host build of the choice of the chain's wavefront (tests/test_chain_wave.py).
#include "veig_chain.hpp"

// a workgroup of `waves` wavefronts, each with its own registers: picks[w] is
// the wavefront that w takes for the chain's
extern "C" void probe_chain(int waves, const unsigned *hw_id, const unsigned *lds_alloc, int *picks) {
  int notes[16];
  for (int w = 0; w < waves; ++w) notes[w] = veig::chain_note(w, hw_id[w], lds_alloc[w]);
  for (int w = 0; w < waves; ++w) picks[w] = veig::chain_pick(notes, waves);
}
