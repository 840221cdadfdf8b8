// parallel_tempering::steps over a model of the C ABI (no device): systems are 64 numbers that a
// sweep scrambles, so every step's energies, masks and draws show in what is printed.
//
//   pt_steps device|host|breaks <steps> [<steps> ...]
//
// one steps() call per count; sa_ladder_exchange_steps always works, always fails for memory, or
// fails for memory after three steps of every second call.  Prints the swap log, energies, minimum,
// rates and final numbers, and on the error stream the most steps that one call asked for.
#include <cinttypes>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "sa/parallel_tempering.hpp"

struct sa_ladder {
  int kind, L, nsys;
  uint64_t t = 0;
  std::vector<uint64_t> v;  // [system][lane]
  int done = 0;
};

namespace {
std::string mode;
int calls = 0, most = 0;
uint64_t mix(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
int E_of(uint64_t v) { return (int)(v % 41) - 20; }
int M_of(uint64_t v) { return (int)((v >> 32) % 41) - 20; }
}  // namespace

extern "C" {
const char *sa_last_error(void) { return "none"; }
const char *sa_status_string(int) { return "status"; }
int sa_ladder_create(int kind, int L, int nsys, sa_ladder **out) {
  *out = new sa_ladder{kind, L, nsys};
  for (int k = 0; k < 64 * nsys; ++k) (*out)->v.push_back(mix((uint64_t)k + 1));
  return SA_OK;
}
int sa_ladder_destroy(sa_ladder *l) { delete l; return SA_OK; }
int64_t sa_ladder_sites(const sa_ladder *l) { return (int64_t)l->L * l->L; }
int sa_ladder_nsys(const sa_ladder *l) { return l->nsys; }
int sa_ladder_sweep(sa_ladder *l, int n) {
  for (int s = 0; s < n; ++s, ++l->t)
    for (uint64_t &x : l->v) x = mix(x + l->t + 0x9E3779B97F4A7C15ULL);
  return SA_OK;
}
int sa_ladder_measure_systems(sa_ladder *l, const int *sys, int n, int32_t *E, int32_t *M) {
  for (int j = 0; j < n; ++j)
    for (int k = 0; k < 64; ++k) {
      E[j * 64 + k] = E_of(l->v[sys[j] * 64 + k]);
      M[j * 64 + k] = M_of(l->v[sys[j] * 64 + k]);
    }
  return SA_OK;
}
int sa_ladder_measure(sa_ladder *l, int32_t *E, int32_t *M) {
  std::vector<int> all;
  for (int j = 0; j < l->nsys; ++j) all.push_back(j);
  return sa_ladder_measure_systems(l, all.data(), l->nsys, E, M);
}
int sa_ladder_swap(sa_ladder *l, int a, int b, uint64_t mask) {
  for (int k = 0; k < 64; ++k)
    if ((mask >> k) & 1) std::swap(l->v[a * 64 + k], l->v[b * 64 + k]);
  return SA_OK;
}
int sa_ladder_exchange_steps(sa_ladder *l, int sweeps, int nsteps, int cold, const int *a, const int *b,
                             const float *min_dE, const double *ha, const double *hb, uint64_t *masks, int32_t *EM) {
  most = std::max(most, nsteps);
  l->done = 0;
  const int limit = mode == "host" ? 0 : mode == "breaks" && ++calls % 2 == 0 ? 3 : nsteps;
  for (int k = 0; k < nsteps; ++k, ++l->done) {
    if (k == limit) return SA_ERR_NOMEM;
    sa_ladder_sweep(l, sweeps);
    const int sys[3] = {cold, a[k], b[k]};
    int32_t *r = EM + (size_t)384 * k;
    for (int q = 0; q < 3; ++q) sa_ladder_measure_systems(l, &sys[q], 1, r + 128 * q, r + 128 * q + 64);
    masks[k] = 0;
    for (int q = 0; q < 64; ++q) {
      const float ea = (float)((double)r[128 + q] + ha[k] * (double)r[192 + q]);
      const float eb = (float)((double)r[256 + q] + hb[k] * (double)r[320 + q]);
      if (-(ea - eb) >= min_dE[k]) masks[k] |= 1ULL << q;
    }
    sa_ladder_swap(l, a[k], b[k], masks[k]);
  }
  return SA_OK;
}
int sa_ladder_exchange_steps_done(const sa_ladder *l) { return l->done; }
int sa_ladder_set_rng(sa_ladder *, int) { return SA_OK; }
int sa_ladder_seed(sa_ladder *, uint64_t) { return SA_OK; }
int sa_ladder_get_seed(const sa_ladder *, uint64_t *s) { *s = 0; return SA_OK; }
int sa_ladder_get_sweep_index(const sa_ladder *l, uint64_t *t) { *t = l->t; return SA_OK; }
int sa_ladder_set_sweep_index(sa_ladder *l, uint64_t t) { l->t = t; return SA_OK; }
int sa_ladder_get_engine(const sa_ladder *, uint64_t *) { return SA_OK; }
int sa_ladder_set_engine(sa_ladder *, const uint64_t *) { return SA_OK; }
int sa_ladder_init_couplings(sa_ladder *) { return SA_OK; }
int sa_ladder_init_spins(sa_ladder *) { return SA_OK; }
int sa_ladder_set_couplings(sa_ladder *, const uint64_t *, const uint64_t *, const uint64_t *) { return SA_OK; }
int sa_ladder_get_couplings(const sa_ladder *, uint64_t *, uint64_t *, uint64_t *) { return SA_OK; }
int sa_ladder_load_J(sa_ladder *, const char *) { return SA_OK; }
int sa_ladder_save_J(const sa_ladder *, const char *) { return SA_OK; }
int sa_ladder_set_spins(sa_ladder *, int, const uint64_t *) { return SA_OK; }
int sa_ladder_get_spins(const sa_ladder *, int, uint64_t *) { return SA_OK; }
int sa_ladder_set_temperature(sa_ladder *, int, double, double, double *) { return SA_OK; }
}

int main(int argc, char **argv) {
  mode = argv[1];
  const std::vector<double> T = {0.6, 0.9, 1.4, 2.0};
  auto lad = std::make_shared<sa::ladder>(SA_KIND_2D, 4, (int)T.size());
  std::vector<std::unique_ptr<sa::hip_sys>> own;
  std::vector<gpu_sys *> sys;
  for (size_t j = 0; j < T.size(); ++j) {
    own.emplace_back(new sa::hip_sys(lad, (int)j, T[j], 0.25));
    sys.push_back(own.back().get());
  }
  std::string name = "pt_steps_%.dat";
  sa::parallel_tempering<gpu_sys> pt(sys, T, 2, name);
  std::vector<sa::swap_record> log;
  pt.set_swap_log(&log);
  for (int q = 2; q < argc; ++q) pt.steps(std::atoi(argv[q]));
  for (auto &r : log) std::printf("step %d %.17g %016" PRIx64 "\n", r.pair, r.u, r.mask);
  for (auto &e : pt.get_E())
    for (float x : e) std::printf("E %.9g\n", x);
  for (float x : pt.get_E_min()) std::printf("min %.9g\n", x);
  for (double x : pt.acceptance()) std::printf("rate %.17g\n", x);
  for (uint64_t x : lad->get()->v) std::printf("v %016" PRIx64 "\n", x);
  std::printf("sweeps %" PRIu64 "\n", lad->get()->t);
  std::fprintf(stderr, "%d\n", most);
  return 0;
}
