// Host check of the pencil sweep's records of long rows (Geometry::pen_wide)
// on one image.
//
//   pencil_wide_check <raw image> <nx> <ny> <nz> <fluid layers> <wall order> <rows per strip>
//
// Every record's oriented x, taken back from the cell its slot belongs to; and,
// where the image's rows are short, the records of long rows against those of
// short ones, word by word.  Prints "wide W records N bad B"; exit status 1 if
// B > 0.
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <vector>

#include "geometry.h"
#include "wallprog.h"

using namespace piks;

int main(int argc, char** argv) {
  if (argc < 8) return 2;
  std::ifstream fh(argv[1], std::ios::binary);
  std::vector<uint8_t> raw((std::istreambuf_iterator<char>(fh)), {});
  GeomInput in{std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6])};
  in.pencil_rows = std::atoi(argv[7]);
  const int vs = in.pencil_vs = 16;
  Geometry g;
  std::string err;
  if (build_geometry(in, raw.data(), (int64_t)raw.size(), g, err) || !g.raster) {
    std::printf("no row records: %s\n", err.c_str());
    return 2;
  }
  const bool wide = g.pen_wide;
  const std::vector<uint32_t> first = g.pen_rec;
  if (!wide && !build_pencil_schedule(g, in.pencil_rows, vs, 4, true)) return 2;
  constexpr int W = Geometry::kTaskWords;
  constexpr uint32_t kFlags = 0xf0000000u;
  std::vector<int32_t> cell_of((size_t)g.nstore + 1, -1);
  for (int64_t c = 0; c < g.Ntotal; ++c) cell_of[(size_t)g.pos[0][(size_t)c]] = (int32_t)c;
  int64_t bad = 0, n = 0;
  for (int o = 0; o < 8; ++o)
    for (int64_t p = g.pen_off[o]; p < g.pen_off[o + 1]; ++p) {
      const Geometry::Pencil& pen = g.pen[(size_t)p];
      for (uint32_t q = 0; q < (pen.n & 0x3fffffffu); ++q, ++n) {
        const size_t at = ((size_t)pen.rec + q) * W;
        const uint32_t* r = &g.pen_rec[at];
        const int i = cell_of[pen.lo + (r[0] & 0x0fffffffu) / vs] - (int)pen.cell;
        if (i < 1 || i > g.Nx || (int)(r[1] & ~kFlags) != (osx(o) > 0 ? i : g.Nx + 1 - i)) ++bad;
        if (wide) continue;
        const uint32_t* s = &first[at];
        if ((int)(s[1] & 0x3fffu) != i || ((s[1] ^ r[1]) & kFlags)) ++bad;
        for (int w = 0; w < W; ++w) bad += w != 1 && s[w] != r[w];
      }
    }
  if (!wide && first.size() != g.pen_rec.size()) ++bad;
  std::printf("wide %d records %lld bad %lld\n", (int)wide, (long long)n, (long long)bad);
  return bad ? 1 : 0;
}
