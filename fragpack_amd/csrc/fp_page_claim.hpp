// Page space of a coded record: the claim-mode encoder's atomic protocol on a
// block's page fill.  Plain C++ over the atomics ``Fill`` supplies, so that a
// host program can run every interleaving of it.
#pragma once

namespace fp {

// Polls a record waits for other records' pending adds (each a round trip to
// the coherence point, >= 0.5 us; one pending add lasts a few microseconds).
constexpr int kPageWaitPolls = 8192;

// A record claims ``need`` bytes of its block's page by one atomic add to the
// fill; ``was`` is what the add returned.  Returns its offset in the page, or
// -1 if it spills.
//
// An add that passes the page's end places nothing and is taken back at once.
// Until then the fill is the placed bytes F plus the pending adds.  Records
// cannot overlap as long as ANY TWO RECORDS EXCEED ANY ONE (asserted where the
// sizes are defined): the first pending add was made on F itself and did not
// fit, so while any is pending less than one record's largest size is left
// behind F, a pending add and another record together never fit there, and a
// record that is placed saw F alone.
//
// A record that finds the fill past the page's end after taking its own add
// back cannot tell F from what is pending and looks again; one that finds it
// at or before the end claims by compare-and-swap, or spills if it does not
// fit behind what it sees (F and perhaps a pending record that fits and will
// be placed by itself).  After the last one no spilled record fits what is
// left.
//
// A fill that rests past the page's end (an encode into pages smaller than
// those it was filled under) looks the same as a pending add, so the wait is
// bounded by ``polls``: then the record spills, and ``polls`` is left 0 for
// the caller to hand to its next record.
template <typename Fill>
__host__ __device__ inline int page_claim(Fill&& fill, int was, int need, long long page_bytes, int& polls) {
  if (was + need <= page_bytes) return was;
  int cur = fill.sub(need) - need;
  for (int n = polls;;) {
    if (cur > page_bytes) {
      if (n-- <= 0) {
        polls = 0;
        return -1;
      }
      cur = fill.load();
    } else if (cur + need <= page_bytes) {
      const int prev = fill.cas(cur, cur + need);
      if (prev == cur) return cur;
      cur = prev;
    } else {
      return -1;
    }
  }
}

}  // namespace fp
