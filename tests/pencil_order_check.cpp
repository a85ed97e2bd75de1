// Host check of the pencil sweep's records over the two raster storage orders,
// on one image: z layer by layer, and y layer by layer, taken where only that
// keeps a row's window within 32-bit offsets (here asked for with `slot`
// elements per slot, which no memory has to hold).
//
//   pencil_order_check <raw image> <nx> <ny> <nz> <fluid layers> <wall order> <rows per strip> <slot>
//
// Every row and record of the second names the cells, octants, marks and waits
// of the first.  Prints "z A B records N bad M", A and B the storage index of
// the cell above (1, 1, 1) less that of (1, 1, 1)'s neighbour along y in either
// order (positive: z is the outer axis); exit status 1 if M > 0.
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <vector>

#include "geometry.h"
#include "wallprog.h"

using namespace piks;

namespace {

constexpr int W = Geometry::kTaskWords;

// A record's sources as cells, tagged (a far source: octant and cell, or a
// corner store entry).
struct Cells {
  const Geometry& g;
  int64_t vs;
  std::vector<int32_t> cell_of;
  Cells(const Geometry& g_, int64_t vs_) : g(g_), vs(vs_), cell_of((size_t)g_.nstore + 1, -1) {
    for (int64_t c = 0; c < g.Ntotal; ++c)
      if (g.pos[0][(size_t)c] != g.nstore) cell_of[(size_t)g.pos[0][(size_t)c]] = (int32_t)c;
  }
  int64_t near(const Geometry::Pencil& p, int64_t off) const {
    if (off % vs || off / vs > p.len) return -2;
    return off / vs == p.len ? -1 : cell_of[(size_t)(p.lo + off / vs)];
  }
  int64_t source(const Geometry::Pencil& p, uint32_t w) const {
    if (!(w & Geometry::kPenFar)) return w % 8 ? -2 : near(p, w / 8);
    const int64_t f = w & 0x3fffffffu;
    if (w & Geometry::kPenFw) return (int64_t)1 << 40 | f;
    return (f / (g.nstore + 1)) << 36 | (int64_t)1 << 41 | cell_of[(size_t)(f % (g.nstore + 1))];
  }
};

}  // namespace

int main(int argc, char** argv) {
  if (argc < 9) return 2;
  std::ifstream fh(argv[1], std::ios::binary);
  std::vector<uint8_t> raw((std::istreambuf_iterator<char>(fh)), {});
  GeomInput in{std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6])};
  in.pencil_rows = std::atoi(argv[7]);
  Geometry a, b;
  std::string err;
  in.pencil_vs = 16;
  if (build_geometry(in, raw.data(), (int64_t)raw.size(), a, err) || !a.raster) return 2;
  in.pencil_vs = std::atoi(argv[8]);
  if (build_geometry(in, raw.data(), (int64_t)raw.size(), b, err) || !b.raster) {
    std::printf("no row records: %s\n", err.c_str());
    return 2;
  }
  const Cells ca(a, 16), cb(b, in.pencil_vs);
  int64_t bad = a.nstore != b.nstore || a.pen.size() != b.pen.size() || a.pen_rec.size() != b.pen_rec.size(), n = 0;
  for (size_t q = 0; !bad && q < a.pen.size(); ++q) {
    const Geometry::Pencil &p = a.pen[q], &r = b.pen[q];
    if (p.rec != r.rec || p.n != r.n || p.id != r.id || p.cell != r.cell) ++bad;
    for (uint32_t t = 0; t < (p.n & 0x3fffffffu); ++t, ++n) {
      const uint32_t* x = &a.pen_rec[((size_t)p.rec + t) * W];
      const uint32_t* y = &b.pen_rec[((size_t)r.rec + t) * W];
      if (ca.near(p, x[0] & 0x0fffffffu) != cb.near(r, y[0] & 0x0fffffffu) || ca.near(p, x[0] & 0x0fffffffu) < 0) ++bad;
      if ((x[0] ^ y[0]) >> 28 || x[1] != y[1] || ((x[7] ^ y[7]) & 7u)) ++bad;
      for (int s = 2; s < 8; ++s) {
        const uint32_t m = s == 7 ? ~7u : ~0u;
        const int64_t u = s >= 6 && x[s] == 0 ? -3 : ca.source(p, x[s] & m), v = s >= 6 && y[s] == 0 ? -3 : cb.source(r, y[s] & m);
        if (u == -2 || (u != v && u != -3 && v != -3)) ++bad;
      }
    }
  }
  auto outer = [](const Geometry& g) {
    return g.pos[0][(size_t)g.cell(1, 1, 2)] - g.pos[0][(size_t)g.cell(1, 2, 1)];
  };
  std::printf("z %d %d records %lld bad %lld\n", outer(a), outer(b), (long long)n, (long long)bad);
  return bad ? 1 : 0;
}
