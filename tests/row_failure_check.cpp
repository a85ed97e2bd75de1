// A sweep whose waits give up (the poll limit of the context's own bounded
// waits is set to 0 from the host, so every kernel ends by itself), and the
// iterations after it.
//
//   row_failure_check <raw image> <nx> <ny> <nz> <graph 0|1>
//
// Prints the return codes of: an iteration, three with the limit at 0, two
// more, and "finite F" for the fields at the end.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <vector>

#include "context.h"

int main(int argc, char** argv) {
  if (argc < 6) return 2;
  std::ifstream in(argv[1], std::ios::binary);
  const std::vector<uint8_t> raw((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
  piks_params p{};
  p.nx = std::atoi(argv[2]);
  p.ny = std::atoi(argv[3]);
  p.nz = std::atoi(argv[4]);
  p.fluid_layer = p.wall_ext_order = 2;
  p.nc_fundamental = 4;
  p.half_range = 1;
  p.ref_l = p.kn = p.press_drop = p.accom = 1.0;
  p.chk_converge_step = 10;
  void* h = nullptr;
  if (int rc = piks_create(&p, raw.data(), (int64_t)raw.size(), &h)) {
    std::printf("create %d %s\n", rc, piks_last_error());
    return 1;
  }
  piks::Ctx& c = *static_cast<piks::Ctx*>(h);
  const bool graph = std::atoi(argv[5]) != 0;
  auto step = [&](uint32_t spin, int n) {
    c.pen_spin = spin;
    // a captured iteration holds its limit
    if (graph && c.graph[0]) {
      (void)hipGraphExecDestroy(c.graph[0]);
      c.graph[0] = nullptr;
    }
    c.use_graph = graph;
    std::printf("%d ", piks_iterate(h, n));
    std::fflush(stdout);
  };
  const uint32_t limit = c.pen_spin;
  step(limit, 1);
  step(0, 3);
  step(limit, 1);
  step(limit, 1);
  int32_t kind = -1;
  piks_get_sweep(h, &kind);
  piks_info info;
  piks_get_info(h, &info);
  std::vector<double> v((size_t)info.ntotal);
  piks_get_macro(h, v.data(), nullptr, nullptr, nullptr);
  bool finite = true;
  for (double x : v) finite = finite && std::isfinite(x);
  std::printf("kind %d finite %d\n", kind, (int)finite);
  piks_destroy(h);
  return 0;
}
