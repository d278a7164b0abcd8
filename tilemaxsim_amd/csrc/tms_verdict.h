// A check's verdict words: int64s in pinned host memory that its workgroups store to and the
// host polls. Plain C++, so the host's side builds and runs without a GPU.
//
// Every check has a tag of its own and stores the tag with its outcome, so a word answers for
// one check only: a store of an earlier check, left over or still to come after a call that
// failed, is never taken for this one's.
#pragma once
#include <stdint.h>

namespace tms {

constexpr int64_t kVerdictFine = 1, kVerdictBad = 2;  // in a word's low byte, the tag above it

inline int64_t verdict_tag(int64_t sequence) { return sequence << 8; }

enum VerdictState { VERDICT_PENDING, VERDICT_FINE, VERDICT_BAD };

struct VerdictPoll {
  const int64_t* words;
  int parts;
  int64_t tag;
  int seen = 0;
  bool bad = false;

  // The outcome so far; PENDING until each of the `parts` words is this check's.
  VerdictState poll() {
    while (seen < parts) {
      const int64_t v = __atomic_load_n(words + seen, __ATOMIC_ACQUIRE);
      if ((v & ~(int64_t)0xff) != tag) return VERDICT_PENDING;
      bad |= (v & 0xff) == kVerdictBad;
      seen++;
    }
    return bad ? VERDICT_BAD : VERDICT_FINE;
  }
};

enum StreamState { STREAM_BUSY, STREAM_DRAINED, STREAM_FAILED };

// Polls until the check has answered, or until the stream has drained (a last look at the
// words) or failed without its answer: PENDING then. `query` gives the stream's state, `nap`
// sleeps; the first `spins` polls do neither.
template <class Query, class Nap>
VerdictState await_verdict(VerdictPoll& p, int64_t spins, Query query, Nap nap) {
  for (int64_t spin = 0;; spin++) {
    VerdictState s = p.poll();
    if (s != VERDICT_PENDING) return s;
    if (spin < spins) {
#if defined(__x86_64__)
      __builtin_ia32_pause();
#endif
      continue;
    }
    const StreamState st = query();
    if (st != STREAM_BUSY) return p.poll();
    nap();
  }
}

}  // namespace tms
