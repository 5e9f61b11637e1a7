// Checks unfinished_code (rate_search.h) on made-up run records.
#include <stdio.h>
#include <initializer_list>
#include "../../dvc_amd/csrc/rate_search.h"

using namespace dvc;

struct Record { int x, y, z, w; };
static int failures = 0;
static void expect(const char *what, int got, int want) {
  if (got != want) {
    printf("%s: %d, expected %d\n", what, got, want);
    failures++;
  }
}

int main() {
  const int C = 65, none = -1;
  Record r[C];
  auto fill = [&](int status) {
    for (auto &q : r) q = Record{7, status, -1, 0};
  };
  for (int step = 0; step < 2; step++) {
    // a search that ran: failures and mismatches below the accepted code
    fill(REC_FAILED);
    for (int l = 0; l < C; l += 3) r[l].y = REC_CRC_MISMATCH;
    r[24].y = REC_ACCEPTED;
    expect("finished", unfinished_code(r, 10, 24, step), none);
    // codes above the accepted one and below the start do not matter
    for (int l = 25; l < C; l++) r[l].y = l & 1 ? REC_CANCELLED : REC_NOT_RUN;
    for (int l = 0; l < 10; l++) r[l].y = REC_NOT_RUN;
    expect("outside", unfinished_code(r, 10, 24, step), none);
    // accepted at the start code, or the start code is the full rate
    expect("at the start", unfinished_code(r, 24, 24, step), none);
    expect("full rate at once", unfinished_code(r, C - 1, C - 1, step), none);
    expect("start above", unfinished_code(r, C, C - 1, step), none);
    // a launch that ended early: nothing ran, and the full rate was taken
    fill(REC_NOT_RUN);
    r[C - 1].y = REC_ACCEPTED;
    expect("nothing ran", unfinished_code(r, 11, C - 1, step), 11);
    // a code lost or cancelled below the accepted one, each offset in turn
    for (int bad : {(int)REC_NOT_RUN, (int)REC_CANCELLED, (int)REC_ACCEPTED})
      for (int off = 0; off < 30; off++) {
        fill(REC_FAILED);
        r[40].y = REC_ACCEPTED;
        r[10 + off].y = bad;
        const bool tried = !step || off == 0 || off == 1 || off == 3 || off == 6 || off == 10 || off == 14 ||
                           off == 18 || off == 22 || off == 26;
        expect("one code", unfinished_code(r, 10, 40, step), tried ? 10 + off : none);
      }
  }
  puts(failures ? "FAILED" : "ok");
  return failures != 0;
}
