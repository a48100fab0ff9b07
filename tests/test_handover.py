"""The hand-over of a workgroup's next item (nwchem_amd/csrc/handover.h) under
every interleaving of its waves.

A host program includes the header the kernel includes and walks three waves
through the item loop: wave 0 puts the next item, all pass the barrier at the
item's end and get it; an item with elements has a barrier of its own before
that, an empty half has none.  A depth-first search over all schedules checks
that the waves meet only at the same barrier of the same item and take the same
items.  The same search over a single shared word (planted here) finds the
schedule that breaks it, so the search sees what it looks for.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r"""
#include "handover.h"
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>
#include <tuple>

struct OneWord {  // the planted mistake
  long word[2];
  void put(long, long item) { word[0] = item; }
  long get(long) const { return word[0]; }
};
#ifdef SINGLE
typedef OneWord Words;
#else
typedef tce_t::NextItem Words;
#endif

constexpr int NW = 3;
enum Pc { ITEM, INNER, PUT, END, GET, DONE };
struct Wave {
  int pc;
  long r, g;
  bool operator<(const Wave &o) const { return std::tie(pc, r, g) < std::tie(o.pc, o.r, o.g); }
};
struct State {
  Wave w[NW];
  Words words;
  bool operator<(const State &o) const {
    for (int k = 0; k < NW; ++k) {
      if (w[k] < o.w[k]) return true;
      if (o.w[k] < w[k]) return false;
    }
    return std::tie(words.word[0], words.word[1]) < std::tie(o.words.word[0], o.words.word[1]);
  }
};

std::string items;  // 'x' an item with elements, '.' an empty one
long n;
std::set<State> seen;

bool waits(const Wave &w) { return w.pc == INNER || w.pc == END; }

// false: some schedule breaks the workgroup
bool walk(const State &s) {
  if (!seen.insert(s).second) return true;
  int done = 0, waiting = 0;
  for (const Wave &w : s.w) done += w.pc == DONE, waiting += waits(w);
  if (done == NW) return true;
  if (waiting == NW) {  // the barrier opens
    State t = s;
    for (Wave &w : t.w) {
      if (w.pc != s.w[0].pc || w.r != s.w[0].r || w.g != s.w[0].g) return false;
    }
    for (Wave &w : t.w) w.pc = s.w[0].pc == INNER ? PUT : GET;
    return walk(t);
  }
  if (done && done + waiting == NW) return false;  // some left, the rest wait
  for (int k = 0; k < NW; ++k) {
    if (waits(s.w[k]) || s.w[k].pc == DONE) continue;
    State t = s;
    Wave &w = t.w[k];
    switch (w.pc) {
      case ITEM: w.pc = w.g < 0 ? DONE : (items[w.g] == 'x' ? INNER : PUT); break;
      case PUT:
        if (k == 0) t.words.put(w.r, w.g + 1 < n ? w.g + 1 : -1);
        w.pc = END;
        break;
      case GET:
        w.g = t.words.get(w.r);
        ++w.r;
        w.pc = ITEM;
        break;
    }
    if (!walk(t)) return false;
  }
  return true;
}

int main(int argc, char **argv) {
  for (int a = 1; a < argc; ++a) {
    items = argv[a];
    n = (long)items.size();
    seen.clear();
    State s{};
    s.words.put(-1, 0);
    for (Wave &w : s.w) w = Wave{GET, -1, 0};  // past the barrier before the loop
    if (!walk(s)) {
      printf("%s\n", items.c_str());
      return 1;
    }
  }
  return 0;
}
"""

SEQUENCES = ["x", ".", "xx", "x.", ".x", "..", "x.x", "x..x", ".x.x.", "x...x", "..x..x.", "xxx.xx"]


def _build(tmp_path, *flags):
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "nwchem_amd", "csrc"),
                    *flags, "-o", str(exe), str(src)], check=True)
    return str(exe)


def test_waves_take_the_same_items_under_every_schedule(tmp_path):
    r = subprocess.run([_build(tmp_path), *SEQUENCES], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, f"a schedule of items {r.stdout.strip()} breaks the workgroup"


@pytest.mark.parametrize("items,breaks", [("xxx", False), ("x.x", True), (".x", True)])
def test_the_search_finds_the_fault_of_a_single_word(tmp_path, items, breaks):
    r = subprocess.run([_build(tmp_path, "-DSINGLE"), items], timeout=60)
    assert r.returncode == (1 if breaks else 0)
