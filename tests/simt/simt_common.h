// Shared by the emulation harnesses simt_rows and simt_batch: the input file of
// tests/test_simt_host.py (_write) and a wavefront of 64 host threads.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <string>
#include <thread>
#include <vector>

#include "../../disco-eb_amd/csrc/deb_host.h"

namespace deb {
thread_local std::string g_err;
}

namespace simt {

struct Input {
  FILE *f = nullptr;
  int mode = 0;
  deb_config_t cfg;
  deb_cosmo_t cosmo;
  std::vector<double> tables, q, w, k, tau;
  int32_t desc[14];
  deb::Layout layout;

  template <class T>
  void get(T *p, size_t n) {
    if (n && fread(p, sizeof(T), n, f) != n) {
      fprintf(stderr, "simt: short input\n");
      exit(2);
    }
  }
  template <class T>
  T one() {
    T v;
    get(&v, 1);
    return v;
  }
  std::vector<double> doubles(size_t n) {
    std::vector<double> v(n);
    get(v.data(), n);
    return v;
  }
  explicit Input(const char *path) : f(fopen(path, "rb")) {
    if (!f) exit(2);
    mode = one<int32_t>();
    cfg = one<deb_config_t>();
    cosmo = one<deb_cosmo_t>();
    tables = doubles(one<int64_t>());
    get(desc, 14);
    const int nq = std::max(one<int32_t>(), 1);
    q = doubles(nq);
    w = doubles(nq);
    k = doubles(one<int32_t>());
    tau = doubles(one<int32_t>());
    if (deb::build_layout(cfg, layout)) {
      fprintf(stderr, "simt: %s\n", deb::g_err.c_str());
      exit(2);
    }
  }
  template <int NS>
  void params(deb::Params<NS> &P) const {
    if (deb::fill_params<NS>(P, &cfg, layout, 1, &cosmo, tables.data(), (int64_t)tables.size(), desc, q.data(),
                             w.data(), (int)k.size(), k.data(), (int)tau.size(), tau.data())) {
      fprintf(stderr, "simt: %s\n", deb::g_err.c_str());
      exit(3);
    }
  }
};

// runs body(wave) on 64 threads per wave, each wave with an exchange buffer of its own
template <class F>
void run_waves(int n, F body) {
  std::vector<Wave> waves(n);
  std::vector<std::thread> th;
  for (int w = 0; w < n; ++w)
    for (int l = 0; l < deb::WAVE; ++l)
      th.emplace_back([&, w, l] {
        lane = l;
        parity = 0;
        wave = &waves[w];
        body(w);
      });
  for (auto &t : th) t.join();
}

}  // namespace simt
