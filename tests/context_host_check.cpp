// The host side of a context (ctx_create_host, no GPU), linked against the
// library: prints which sweep the settings chose and what was laid out for it.
//
//   context_host_check <raw image> <nx> <ny> <nz> <layers> <order> <nc> <precision> <sweep>
//
// Output: "rc N" and, if rc is 0, "tiles T rows R raster S vs V nc8 C
// tile_words W row_words P hyper_words H".
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <vector>

#include "context.h"

int main(int argc, char** argv) {
  if (argc < 10) return 2;
  std::ifstream in(argv[1], std::ios::binary);
  const std::vector<uint8_t> raw((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
  piks_params p{};
  p.nx = std::atoi(argv[2]);
  p.ny = std::atoi(argv[3]);
  p.nz = std::atoi(argv[4]);
  p.fluid_layer = std::atoi(argv[5]);
  p.wall_ext_order = std::atoi(argv[6]);
  p.nc_fundamental = std::atoi(argv[7]);
  p.precision = std::atoi(argv[8]);
  p.sweep = std::atoi(argv[9]);
  p.ref_l = p.kn = p.press_drop = p.accom = 1.0;
  p.half_range = 1;
  p.exact_quadrature = p.nc_fundamental == 3;
  p.chk_converge_step = 10;
  piks::Ctx* c = nullptr;
  const int rc = piks::ctx_create_host(&p, raw.data(), (int64_t)raw.size(), &c);
  std::printf("rc %d\n", rc);
  if (rc) return 0;
  std::printf("tiles %d rows %d raster %d vs %d nc8 %d tile_words %zu row_words %zu hyper_words %zu\n", c->sweep_tiles,
              c->pencil, c->g.raster, c->d.vs, c->d.Nc8, c->g.tl_rec.size(), c->g.pen_rec.size(), c->g.hp_task.size());
  delete c;
  return 0;
}
