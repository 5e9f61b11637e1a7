// Checks run_pair (host_pair.h): both parts run, their results come back, and
// neither part's exception ends the process or is lost.
#include <stdio.h>
#include <atomic>
#include <stdexcept>
#include "../../dvc_amd/csrc/host_pair.h"

using namespace dvc;

int main() {
  int failures = 0;
  for (int a = 0; a < 4; a++)
    for (int b = 0; b < 4; b++) {
      std::atomic<int> ran{0};
      auto part = [&ran](int kind) {
        return [&ran, kind]() -> int {
          ran++;
          if (kind == 1) throw std::bad_alloc();
          if (kind == 2) throw std::runtime_error("a text longer than a string keeps in itself");
          return kind == 3 ? -5 : 0;
        };
      };
      int rc[2] = {99, 99};
      std::string what[2];
      run_pair(part(a), part(b), -4, rc, what);
      const int want[4] = {0, -4, -4, -5};
      const char *text[4] = {"", "out of memory", "a text longer than a string keeps in itself", ""};
      if (ran != 2 || rc[0] != want[a] || rc[1] != want[b] || what[0] != text[a] || what[1] != text[b]) {
        printf("parts %d, %d: %d ran, results %d %d, '%s' '%s'\n", a, b, (int)ran, rc[0], rc[1], what[0].c_str(),
               what[1].c_str());
        failures++;
      }
    }
  puts(failures ? "FAILED" : "ok");
  return failures != 0;
}
