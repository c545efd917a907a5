// Prints what awflcloud_amd/csrc/awfl_cut.hpp answers, one line per line of
// standard input: "adj n lines" -> lines per work-group.
#include <cstdio>
#include <cstring>

#include "../../awflcloud_amd/csrc/awfl_cut.hpp"

int main() {
  char what[16];
  while (std::scanf("%15s", what) == 1) {
    if (!std::strcmp(what, "adj")) {
      int n;
      long long lines;
      if (std::scanf("%d %lld", &n, &lines) != 2) return 1;
      std::printf("%d\n", awfl_cut::adj_cols(n, lines));
    } else {
      return 1;
    }
  }
  return 0;
}
