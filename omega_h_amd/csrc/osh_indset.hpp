// The rounds of the independent sets (indset::find,
// src/Omega_h_indset.cpp:5-35), shared by the sweeps over a mesh's nodes and
// those over a swap pass's candidates.
#pragma once

#include <utility>

#include "osh_passes.hpp"

namespace osh {

// one round of indset::find (src/Omega_h_indset.cpp:5-35).  In the first
// round the states come straight from the candidate marks (2 for a
// candidate, 0 otherwise), so no node is in the set yet.
template <bool FIRST>
__device__ __forceinline__ I8 indset_state(I8 const* old_state, LO x) {
  I8 s = old_state[x];
  return FIRST ? I8(s ? 2 : 0) : s;
}

// A node joins the set once every neighbor that beats it (higher quality,
// or the same quality and a higher index) is out, and leaves once one of
// them is in: a neighbor it beats can be in only after the node is out, so
// this is the round above restated over the beating neighbors alone.  The
// first round records, per candidate, which row positions hold candidates
// that beat it (bits of `dom`); later rounds read the states at those
// positions only, not the qualities.  A row longer than 64 positions is
// read whole every round.
constexpr int kDomBits = 64;

// Each batch of rounds ends with a wait for two words: kUndecidedWord, set by
// the last round's nodes that stay undecided, and kCandWord, set by the first
// round's candidates, so that no reduction over the states is needed.
constexpr int kUndecidedWord = 0;
constexpr int kCandWord = 1;

// one lane a wave stores, and only where the word does not hold the tag yet
__device__ __forceinline__ void tell(bool is, unsigned* word, unsigned tag) {
  unsigned long long b = __ballot(is);
  if (b == 0ull || int(threadIdx.x & 63) != __ffsll(static_cast<long long>(b)) - 1) return;
  if (__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != tag)
    __hip_atomic_store(word, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct IndsetWords {
  unsigned* words;
  unsigned cand_tag;  // 0: not the first round
  unsigned last_tag;  // 0: not the last round of its batch
};

__device__ __forceinline__ void tell_round(I8 before, I8 after, IndsetWords w) {
  if (w.cand_tag) tell(before == 2, w.words + kCandWord, w.cand_tag);
  if (w.last_tag) tell(after == 2, w.words + kUndecidedWord, w.last_tag);
}

// Runs rounds until no node is undecided.  round(first, in, out, words)
// launches one; the first reads `cands` (nonzero: a candidate), later ones the
// states of the round before, which alternate between a and b.  Returns the
// final states: 1 in the set, 0 not.  *any_cands tells whether there was a
// candidate.  `stop` as in find_indset.
//
// Rounds leave decided nodes as they are and take no node from the set, so
// extra rounds after convergence change nothing: two rounds run before each of
// the first four waits, then 4, 8 and 16 (long chains of decreasing quality,
// as on the first coarsening passes of a large smooth mesh, take some 200
// rounds and would otherwise spend a wait every two).
template <class Round>
Bytes indset_rounds(Ctx& c, LO n, Bytes const& cands, Bytes a, Bytes b, bool* any_cands,
    Round const& round_of, StopWord const* stop = nullptr) {
  for (LO round = 0;;) {
    OSH_CHECK(round <= n + 1, "independent set does not converge");
    int batch = round < 8 ? 2 : (round < 16 ? 4 : (round < 32 ? 8 : 16));
    unsigned tag = c.wait_tag();
    for (int k = 0; k < batch; ++k, ++round) {
      bool first = round == 0;
      IndsetWords w{c.words, first ? tag : 0u, k == batch - 1 ? tag : 0u};
      round_of(first, first ? cands.data() : a.data(), b.data(), w);
      std::swap(a, b);
    }
    c.wait();
    if (any_cands && round == 2) *any_cands = c.word_set(kCandWord, tag);
    if (stop && c.word_set(stop->word, stop->tag)) return a;
    if (!c.word_set(kUndecidedWord, tag)) return a;
  }
}

}  // namespace osh
