// Host side of the bounds checks' verdict words (tms_verdict.h), without a GPU: stores of an
// earlier check stand in for a kernel that a failed call left behind.
#include <stdio.h>
#include <stdlib.h>

#include "tms_verdict.h"

using namespace tms;

static int64_t words[64];

static void store(int i, int64_t tag, int64_t outcome) { __atomic_store_n(words + i, tag | outcome, __ATOMIC_RELEASE); }

static void expect(bool ok, const char* what) {
  if (ok) return;
  printf("failed: %s\n", what);
  exit(1);
}

int main() {
  auto nap = []() {};
  const int64_t older = verdict_tag(7), mine = verdict_tag(8);
  expect(older != mine && (mine & 0xff) == 0, "tags differ above the outcome");

  // the earlier check's late "fine" is not this one's, whatever word it lands in
  for (int i = 0; i < 3; i++) store(i, older, kVerdictFine);
  VerdictPoll p{words, 3, mine};
  expect(p.poll() == VERDICT_PENDING, "an older check's words");
  int asked = 0;
  VerdictState s = await_verdict(
      p, 4,
      [&]() {  // busy for two queries, the check's stores in between
        asked++;
        if (asked == 1) store(0, mine, kVerdictFine), store(1, mine, kVerdictFine);
        if (asked == 2) store(2, mine, kVerdictBad);
        return STREAM_BUSY;
      },
      nap);
  expect(s == VERDICT_BAD && asked == 2, "bad although an older check said fine");

  // a late "bad" of the earlier check refuses nothing
  for (int i = 0; i < 3; i++) store(i, older, kVerdictBad);
  VerdictPoll q{words, 3, mine};
  expect(q.poll() == VERDICT_PENDING, "an older check's bad words");
  for (int i = 0; i < 3; i++) store(i, mine, kVerdictFine);
  expect(q.poll() == VERDICT_FINE, "fine although an older check said bad");

  // drained or failed: a last look at the words, then no answer
  for (int i = 0; i < 3; i++) store(i, older, kVerdictFine);
  VerdictPoll r{words, 3, mine};
  expect(await_verdict(r, 0, []() { return STREAM_DRAINED; }, nap) == VERDICT_PENDING, "drained without an answer");
  VerdictPoll f{words, 3, mine};
  expect(await_verdict(f, 0, []() { return STREAM_FAILED; }, nap) == VERDICT_PENDING, "failed without an answer");
  VerdictPoll t{words, 1, mine};
  s = await_verdict(
      t, 0,
      [&]() {
        store(0, mine, kVerdictFine);  // seen between the poll and the query
        return STREAM_DRAINED;
      },
      nap);
  expect(s == VERDICT_FINE, "the last look after the stream has drained");
  printf("ok\n");
  return 0;
}
