// CPU harness of the batched solve's host rule: which kernel instance runs a
// group, and the LDS it reserves.  Test infrastructure only.
//
//   simt_batch rule
//     prints one line "slots batch waves instance lds_bytes" per slot count and group size
#include <cstdio>
#include <cstring>

#include <hip/hip_runtime.h>
#define __builtin_amdgcn_wave_barrier() simt::wave->bar.arrive_and_wait()

#include "../../disco-eb_amd/csrc/deb_batch.h"

using namespace deb;

namespace {

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
  fprintf(stderr, "usage: simt_batch rule\n");
  return 2;
}
