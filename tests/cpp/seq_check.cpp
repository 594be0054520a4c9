// seq_check.cpp - CPU check of the iterations' numbers and status words (hoc_seq.hpp): the word gives back
// its number and flags, and the order of numbers holds for as many iterations as a handle may run, over the
// wrap and where 32-bit arithmetic on the word (4 seq) would change sign.  Prints "OK" and exits 0.
#include <cstdio>

#include "hoc_seq.hpp"

using namespace hoc;

int main() {
  int bad = 0;
  const int at[] = {0, (1 << 29) - 3, kSeqStart, kSeqMod - 3};
  for (int base : at)
    for (int i = 0; i < 8; ++i) {
      const int s = seq_add(base, i);
      bad += s < 0 || s >= kSeqMod;
      for (int f = 0; f < 4; ++f) {
        const uint32_t v = status_word(s, (f & 2) != 0, (f & 1) != 0);
        bad += status_seq(v) != s || status_near(v) != ((f & 2) != 0) || status_active(v) != ((f & 1) != 0);
      }
      // a wait for s: not ended by any of the 1000 iterations before it, ended by it and those after
      for (int d = 1; d <= 1000; ++d) bad += seq_reached(seq_add(s, -d), s) || !seq_reached(seq_add(s, d), s);
      bad += !seq_reached(s, s);
    }
  std::printf(bad ? "%d failures\n" : "OK\n", bad);
  return bad != 0;
}
