// The next work item of a persistent workgroup, handed from the one thread that
// draws it to all waves: at the end of item r the drawing thread puts the item
// that follows, the workgroup passes one barrier, every wave gets it.
#pragma once

namespace tce_t {

// Two words, used in turn.  An item may have no barrier but that one (a half
// item without any element), so the drawing thread can reach the put of item
// r + 1 while other waves have yet to get what was put at the end of item r;
// with a single word they would read the later item and leave the workgroup's
// barriers.  A word is written again two items later, past the barrier of the
// item between, which every wave reaches only after its get.  Plain (constexpr)
// code: the hand-over test runs it on host threads.
struct NextItem {
  long word[2];
  constexpr void put(long r, long item) { word[r & 1] = item; }
  constexpr long get(long r) const { return word[r & 1]; }
};

}  // namespace tce_t
