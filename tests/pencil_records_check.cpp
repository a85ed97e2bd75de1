// Host check of the pencil sweep's schedule (build_pencil_schedule) on one
// image, against the hyperplane schedule of the same image.
//
//   pencil_records_check <raw image> <nx> <ny> <nz> <fluid layers> <wall order> <rows per strip> [plant]
//
// With "plant" one wait mark is cleared and one source is moved before the
// checks, which must report both.  Checks, per octant:
//  * the rows hold every task of the hyperplane schedule once, in the
//    octant's x direction, with its flags;
//  * a source read from a register is the row's previous task (or the one
//    before), every other source the cell and octant the hyperplane kernels
//    read, switched wall slots included (the views of Geometry::wall_views);
//  * along y and z the nearest neighbour that the octant sweeps, and only it,
//    is waited for, and its row comes earlier in the octant's list, so the
//    claims drain whatever number of waves runs.
// Prints "bad N"; exit status 1 if N > 0.
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <string>
#include <vector>

#include "geometry.h"
#include "wallprog.h"

using namespace piks;

int main(int argc, char** argv) {
  if (argc < 8) return 2;
  const bool plant = argc > 8 && std::string(argv[8]) == "plant";
  std::ifstream fh(argv[1], std::ios::binary);
  std::vector<uint8_t> raw((std::istreambuf_iterator<char>(fh)), {});
  GeomInput in{std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6])};
  Geometry h, g;
  std::string err;
  if (build_geometry(in, raw.data(), (int64_t)raw.size(), h, err)) {
    std::printf("geometry: %s\n", err.c_str());
    return 2;
  }
  in.pencil_rows = std::atoi(argv[7]);
  const int64_t vs = in.pencil_vs = 48;  // elements per slot
  if (build_geometry(in, raw.data(), (int64_t)raw.size(), g, err) || !g.raster) {
    std::printf("pencil geometry: %s\n", err.c_str());
    return 2;
  }
  constexpr int W = Geometry::kTaskWords;
  if (plant) {
    bool wait = false, src = false;
    for (size_t t = 0; t < g.pen_rec.size() / W && !(wait && src); ++t)
      for (int q = 1; q <= 5; ++q) {
        uint32_t& w = g.pen_rec[t * W + q];
        if (q == 1 && !wait && (w & Geometry::kPenWaitY)) {
          w &= ~Geometry::kPenWaitY;
          wait = true;
        } else if (q > 1 && !src && !(w & Geometry::kPenFar)) {
          w += (uint32_t)vs * 8u;
          src = true;
        }
      }
    std::printf("planted: wait mark %d, source %d\n", (int)wait, (int)src);
  }
  int64_t bad = 0, switched = 0, corner = 0, regs = 0;
  auto fail = [&](const char* what, int o, int64_t c) {
    if (bad++ < 10) std::printf("FAIL %s (octant %d, cell %lld)\n", what, o, (long long)c);
  };
  if (g.nstore != h.nstore) fail("stored cells", -1, g.nstore);
  std::vector<int32_t> cell_of((size_t)g.nstore + 1, -1);
  for (int64_t c = 0; c < g.Ntotal; ++c)
    if (g.pos[0][(size_t)c] != g.nstore) {
      if (h.pos[0][(size_t)c] == h.nstore) fail("stored cell", -1, c);
      cell_of[(size_t)g.pos[0][(size_t)c]] = (int32_t)c;
    }
  std::vector<int32_t> hp_task((size_t)g.Ntotal), row_at((size_t)g.Ny * g.Nz);
  for (int o = 0; o < 8; ++o) {
    std::fill(hp_task.begin(), hp_task.end(), -1);
    int64_t ntask = 0, seen = 0;
    std::vector<int32_t> fam_cell((size_t)h.nstore + 1, -1);
    for (int64_t c = 0; c < h.Ntotal; ++c) fam_cell[(size_t)h.pos[ofam(o)][(size_t)c]] = (int32_t)c;
    for (int s = 0; s < h.nhp; ++s)
      for (int64_t t = h.hp_oct[(size_t)s * 8 + o]; t < h.hp_oct[(size_t)s * 8 + o + 1]; ++t, ++ntask)
        hp_task[(size_t)((uint32_t)h.hp_task[(size_t)t * W + 7] & 0x0fffffffu)] = (int32_t)t;
    std::fill(row_at.begin(), row_at.end(), -1);
    if (g.pen_tasks[o] != ntask) fail("task count", o, g.pen_tasks[o]);
    const int64_t dx = osx(o), st[2] = {(int64_t)osy(o) * g.Nxt, (int64_t)osz(o) * g.Nxyt};
    auto swept = [&](int64_t c) { return hp_task[(size_t)c] >= 0; };
    for (int64_t p = g.pen_off[o]; p < g.pen_off[o + 1]; ++p) {
      const Geometry::Pencil& pen = g.pen[(size_t)p];
      const int j = 1 + (int)(pen.id % (uint32_t)g.Ny), k = 1 + (int)(pen.id / (uint32_t)g.Ny);
      if (row_at[pen.id] >= 0) fail("row twice", o, pen.id);
      row_at[pen.id] = (int32_t)p;
      if ((int64_t)pen.cell != g.cell(0, j, k)) fail("row cell", o, pen.cell);
      // storage index of a record's offset (nstore: the zero slot)
      auto index = [&](uint32_t off) -> int64_t {
        if (off % vs || off / vs > pen.len) return -1;
        return off / vs == pen.len ? g.nstore : pen.lo + off / vs;
      };
      bool waits_any[2] = {false, false};
      int64_t before[2] = {-1, -1};
      for (uint32_t q = 0; q < (pen.n & 0x3fffffffu); ++q, ++seen) {
        const uint32_t* r = &g.pen_rec[((size_t)pen.rec + q) * W];
        const int i = (int)(r[1] & 0x3fffu);
        const int64_t c = pen.cell + i;
        if (i < 1 || i > g.Nx || !swept(c)) {
          fail("not a task of the row", o, c);
          continue;
        }
        if ((int)((r[1] >> 14) & 0x3fffu) != 1 + (dx > 0 ? i - 1 : g.Nx - i)) fail("oriented x", o, c);
        if (before[0] >= 0 && (c - before[0]) * dx <= 0) fail("x order", o, c);
        const int32_t* t = &h.hp_task[(size_t)hp_task[(size_t)c] * W];
        const uint32_t flags = (uint32_t)t[7] >> 28;
        if (index(r[0] & 0x0fffffffu) != g.pos[0][(size_t)c]) fail("slot", o, c);
        if (((r[0] >> 28) & 7u) != (flags & 7u)) fail("flags", o, c);
        // x
        for (int d = 1; d <= 2; ++d) {
          const bool reg = r[1] & (d == 1 ? Geometry::kPenX1Reg : Geometry::kPenX2Reg);
          const int64_t n = c - d * dx;
          if (reg != swept(n)) fail("x register", o, c);
          const bool x1 = r[1] & Geometry::kPenX1Reg;
          if (reg || (d == 2 && x1)) {
            // a register: the previous task's result, or what that task read at distance 1
            if (reg && before[d == 2 && x1 ? 1 : 0] != n) fail("x register value", o, c);
            if (!reg && before[0] + dx != c) fail("x shifted value", o, c);
            ++regs;
          } else {
            const uint32_t off = d == 2 ? r[7] & ~7u : r[6];
            const int64_t row = off % 8 ? -1 : index(off / 8);
            const int64_t src = row == g.nstore ? -1 : row >= 0 ? cell_of[(size_t)row] : -2;
            const int64_t want = t[d] == (int32_t)h.nstore ? -1 : fam_cell[(size_t)t[d]];
            if (src != want || (want >= 0 && want != n)) fail("x source", o, c);
          }
        }
        // y, z
        bool special = false;
        for (int ax = 0; ax < 2; ++ax) {
          bool waits = false;
          for (int d = 1; d <= 2; ++d) {
            const int64_t n = c - d * st[ax];
            const uint32_t w = r[2 + 2 * ax + d - 1];
            const bool want_wait = !waits && swept(n);
            waits = waits || swept(n);
            const bool marked = d == 1 ? (r[1] & (ax == 0 ? Geometry::kPenWaitY : Geometry::kPenWaitZ)) != 0
                                       : (r[7] & (ax == 0 ? Geometry::kPenWaitY2 : Geometry::kPenWaitZ2)) != 0;
            if (marked != want_wait) fail("wait mark", o, c);
            if (want_wait) {
              const int64_t id = (int64_t)pen.id - d * (ax == 0 ? osy(o) : osz(o) * g.Ny);
              if (id < 0 || id >= (int64_t)row_at.size() || row_at[(size_t)id] < 0) fail("row order", o, c);
              if (d == 1) waits_any[ax] = true;
              special = special || d == 2;
            }
            int view = 0;
            if ((flags & 8u) && g.lab[(size_t)n] >= 20)
              view = (int)((g.wall_views[(size_t)g.wid[(size_t)n]] >> (8 * o + 4 * ax)) & 15u);
            const uint32_t far = w & 0x3fffffffu;
            if (view) special = true;
            if (view == 9) {
              ++corner;
              if (!(w & Geometry::kPenFar) || !(w & Geometry::kPenFw) ||
                  (int64_t)far != (int64_t)g.wall_corner[(size_t)g.wid[(size_t)n]] * 8 + o)
                fail("corner source", o, c);
              continue;
            }
            switched += view != 0;
            if (view) {
              if (w >> 30 != 2u || (int64_t)far != (int64_t)(view - 1) * (g.nstore + 1) + g.pos[0][(size_t)n])
                fail("source", o, c);
            } else if (w >> 31 || w % 8 || index(w / 8) != g.pos[0][(size_t)n]) {
              fail("source", o, c);
            }
            // the plain slot is the one the hyperplane task names
            const int32_t plain = t[3 + 2 * ax + d - 1];
            if ((plain == (int32_t)h.nstore) != (g.pos[0][(size_t)n] == (int32_t)g.nstore) ||
                (plain != (int32_t)h.nstore && fam_cell[(size_t)plain] != n))
              fail("plain source", o, c);
          }
        }
        if (special != ((r[0] & Geometry::kPenSpecial) != 0)) fail("special mark", o, c);
        before[1] = before[0];
        before[0] = c;
      }
      if (waits_any[0] != (pen.n >> 31 != 0) || waits_any[1] != (((pen.n >> 30) & 1u) != 0)) fail("row waits", o, pen.id);
    }
    if (seen != ntask) fail("tasks seen", o, seen);
  }
  std::printf("rows %zu, register sources %lld, switched reads %lld, corner reads %lld\nbad %lld\n", g.pen.size(),
              (long long)regs, (long long)switched, (long long)corner, (long long)bad);
  return bad ? 1 : 0;
}
