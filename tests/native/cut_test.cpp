// Prints what awflcloud_amd/csrc/awfl_cut.hpp answers, one line per line of
// standard input: "adj n lines" -> lines per work-group; "tile dir n nline other
// periodic whole" -> lines, rows, segments, segment length, threads and LDS bytes of
// an FP64 tile; "form bits dir ord nx ny nz periodic" -> the faster form by the models;
// "tracers dir ord nx ny nz ntr" -> form, lines per work-group of the tile and its LDS bytes.
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
    } else if (!std::strcmp(what, "tile")) {
      int dir, n, nline, other, per, whole;
      if (std::scanf("%d %d %d %d %d %d", &dir, &n, &nline, &other, &per, &whole) != 6) return 1;
      const awfl_cut::TileCut t = awfl_cut::tile_cut(dir, n, nline, other, per, awfl_cut::rates_f64(dir, 5), whole);
      std::printf("%d %d %d %d %d %zu\n", t.p.cols, t.p.rows, t.p.nseg, t.p.seglen, t.threads,
                  sizeof(double) * awfl_cut::lds_elems(t.p, 2));
    } else if (!std::strcmp(what, "form")) {
      int bits, dir, ord, nx, ny, nz, per;
      if (std::scanf("%d %d %d %d %d %d %d", &bits, &dir, &ord, &nx, &ny, &nz, &per) != 7) return 1;
      const awfl_cut::Rates& r = bits == 64 ? awfl_cut::rates_f64(dir, ord) : awfl_cut::rates_f32(dir, ord);
      const int n = dir == 1 ? ny : nz, other = dir == 1 ? nz : ny;
      std::puts(awfl_cut::tile_cut(dir, n, nx, other, per, r).us <= awfl_cut::walk_cut(n, nx, other, r).us ? "tile" : "walker");
    } else if (!std::strcmp(what, "tracers")) {
      int dir, ord, nx, ny, nz, ntr;
      if (std::scanf("%d %d %d %d %d %d", &dir, &ord, &nx, &ny, &nz, &ntr) != 6) return 1;
      const int n = dir == 0 ? nx : dir == 1 ? ny : nz;
      const awfl_cut::TtCut t = awfl_cut::tt_cut(dir, n, (long long)nx * ny * nz / n, (ord - 1) / 2, ntr);
      const bool tile = t.cols && (dir == 0 || n < 8 ||
                                   awfl_cut::tt_tile(t, dir, ord, n, (long long)((nx + 3) / 4) * (dir == 1 ? nz : ny), ntr));
      std::printf("%s %d %zu\n", tile ? "tile" : "walker", t.cols, awfl_cut::tt_lds(n, t.cols, (ord - 1) / 2, ntr));
    } else {
      return 1;
    }
  }
  return 0;
}
