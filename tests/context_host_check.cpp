// The host side of a context (ctx_create_host, no GPU), linked against the
// library: prints which sweep the settings chose and what was laid out for it.
//
//   context_host_check <raw image> <nx> <ny> <nz> <layers> <order> <nc> <precision> <sweep> [fit]
//
// Output: "rc N" and, if rc is 0, "tiles T rows R raster S vs V nc8 C
// tile_words W row_words P hyper_words H bytes B layout L", with L a digest of
// what the device is given (storage order, records, lists of slots).
// With fit=N, ctx_fit(N bytes) comes before.
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <vector>

#include "context.h"

namespace {

uint64_t digest = 1469598103934665603ull;

template <typename T>
void add(const std::vector<T>& v) {
  const unsigned char* p = reinterpret_cast<const unsigned char*>(v.data());
  for (size_t q = 0; q < v.size() * sizeof(T); ++q) digest = (digest ^ p[q]) * 1099511628211ull;
}

}  // namespace

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
  int rf = 0;
  if (rc == 0 && argc > 10) rf = piks::ctx_fit(*c, (size_t)std::atoll(argv[10]));
  std::printf("rc %d\n", rc ? rc : rf);
  if (rc || rf) return 0;
  const piks::Geometry& g = c->g;
  for (int q = 0; q < 4; ++q) add(g.pos[q]);
  add(g.hp_task);
  add(g.hp_off);
  add(g.hp_oct);
  add(g.hp_lo);
  add(g.hp_len);
  add(g.wall_pos);
  add(c->ns_host);
  add(std::vector<int64_t>{g.nstore, c->d.vs, c->d.ostride, c->d.rs_f, (int64_t)c->n_f, c->n_ns});
  std::printf("tiles %d rows %d raster %d vs %d nc8 %d tile_words %zu row_words %zu hyper_words %zu bytes %zu layout %lld\n",
              c->sweep_tiles, c->pencil, g.raster, c->d.vs, c->d.Nc8, g.tl_rec.size(), g.pen_rec.size(),
              g.hp_task.size(), piks::ctx_device_bytes(*c), (long long)(digest >> 1));
  delete c;
  return 0;
}
