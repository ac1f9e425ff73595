// Every place of a head's state that the threads of the kernels for single tokens read, for sizes as the kernels are chosen for: inside the head, and each float of
// it the row of exactly one thread.  Prints the sizes of which that does not hold.
#include <cstdio>
#include <vector>

#include "../state_rows.h"

int main() {
  constexpr int MOST = 32;  // rows a thread holds registers for: 4 to 32 (delta rule), 16 (retention), or eight at a time (state spaces)
  long bad = 0, sizes = 0;
  for (int width = 4; width <= 1024; width += width < 64 ? 4 : 12)
    for (int rows = 1; rows <= 1024; rows += rows < 64 ? 1 : 47) {
      const int groups = 256 / (width >> 2), held = (rows + groups - 1) / groups;
      ++sizes;
      bool ok = true;
      std::vector<unsigned char> seen((size_t)rows * width, 0);
      for (int tid = 0; tid < 256; ++tid) {
        const StateRows s = state_rows(tid, rows, width);
        for (int i = 0; i < (held < MOST ? MOST : held + 7); ++i) ok &= s.at(i) >= 0 && s.at(i) + 4 <= rows * width;
        for (int i = 0; ok && i < s.count; ++i) {
          ok &= s.at(i) == (s.group + i * s.groups) * width + s.col;
          for (int e = 0; ok && e < 4; ++e) ok &= !seen[s.at(i) + e]++;
        }
      }
      for (unsigned char n : seen) ok &= n == 1;
      if (!ok && bad++ < 10) std::printf("%d rows of %d: out of the head, or not each once\n", rows, width);
    }
  std::printf("%ld sizes, %ld bad\n", sizes, bad);
  return bad != 0;
}
