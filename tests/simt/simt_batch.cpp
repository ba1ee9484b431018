// CPU emulation harness of the batched solve (integrate_batch): one host thread
// per lane of every wave of a group's workgroup, the workgroup barrier over all
// of them.  Built and run like simt_host (sanitizers).  Test infrastructure only.
//
//   simt_batch rule
//     prints one line "slots batch waves instance lds_bytes" per slot count and
//     group size: which kernel instance runs a group, and the LDS it reserves
//   simt_batch <in.bin> <out.bin>
//     in.bin: written by _write of tests/test_simt_host.py, mode 0, followed by
//       int32 batch; int32 waves (those launched; any number up to 8)
//     out.bin: int32 status[nk]; int32 nsteps[nk]; double y[nk][nout][20]
#include <cstring>
#include <memory>

#include "simt_common.h"

namespace simt {
inline std::barrier<> *group = nullptr;
}
#define __builtin_amdgcn_s_barrier() simt::group->arrive_and_wait()
#define __builtin_amdgcn_wave_barrier() simt::wave->bar.arrive_and_wait()

#include "../../disco-eb_amd/csrc/deb_batch.h"

using namespace deb;

namespace {

constexpr int MAXW = 8;

template <int NS>
void rule() {
  for (int B = 1; B <= 64; ++B) {
    const int waves = batch_waves_of(batch_waves<NS>(), B), nw = batch_instance<NS>(waves);
    const size_t lds = nw * sizeof(BatchWave<NS>) +
                       (nw == 1 ? sizeof(BatchShare<1>) : nw == 2 ? sizeof(BatchShare<2>)
                                : nw == 4 ? sizeof(BatchShare<4>) : sizeof(BatchShare<8>));
    printf("%d %d %d %d %zu\n", NS, B, waves, nw, lds);
  }
}

template <int NS>
int run(simt::Input &in, const char *path) {
  Params<NS> P;
  in.params<NS>(P);
  const int B = in.one<int32_t>(), nw = in.one<int32_t>();
  const int nk = P.nk;
  if (nw < 1 || nw > MAXW || nw > B || nk % B) return 2;
  std::vector<double> y((size_t)nk * P.nout * DEB_NOUT_FIELDS, -12345.0);
  std::vector<int32_t> status(nk, -9), nsteps(nk, -9);
  P.y_out = y.data();
  P.status = status.data();
  P.nsteps = nsteps.data();
  for (int g = 0; g < nk / B; ++g) {
    std::vector<double> ws((size_t)nk * 2 * NS * WAVE, -777.0);
    auto waves = std::make_unique<BatchWave<NS>[]>(nw);  // (an access to a wave that is not launched ends the run)
    std::memset((void *)waves.get(), 0xa5, nw * sizeof(BatchWave<NS>));
    BatchShare<MAXW> share;
    std::memset((void *)&share, 0xa5, sizeof(share));
    std::barrier<> bar(nw * WAVE);
    simt::group = &bar;
    simt::run_waves(nw, [&](int w) { integrate_batch<NS, MAXW>(P, 0, g * B, B, w, nw, waves[w], share, ws.data()); });
  }
  FILE *out = fopen(path, "wb");
  if (!out) return 2;
  fwrite(status.data(), 4, nk, out);
  fwrite(nsteps.data(), 4, nk, out);
  fwrite(y.data(), 8, y.size(), out);
  fclose(out);
  return 0;
}

}  // namespace

int main(int argc, char **argv) {
  if (argc == 2 && std::strcmp(argv[1], "rule") == 0) {
    rule<1>();
    rule<2>();
    rule<3>();
    rule<4>();
    rule<5>();
    rule<6>();
    return 0;
  }
  if (argc != 3) {
    fprintf(stderr, "usage: simt_batch rule | in.bin out.bin\n");
    return 2;
  }
  simt::Input in(argv[1]);
  switch (in.layout.ns) {
    case 1: return run<1>(in, argv[2]);
    case 2: return run<2>(in, argv[2]);
    case 5: return run<5>(in, argv[2]);
    default: fprintf(stderr, "simt_batch: slot count %d not built\n", in.layout.ns); return 2;
  }
}
