// rr_fold on the CPU, a thread per lane: exit status 0 if every check holds.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../top3d_xl_amd/csrc/t3x_reduce.h"

using namespace t3x;

static int run(int block, double* partials, int nb, double* sc, int* fl, int raiseAfterWave, int* returned) {
  std::atomic<int> early{0}, there{0};
  const RrFold f{partials, nb, sc, fl};
  std::vector<int> got(kBlock, -1);
  model::run_block(
      block, kBlock, [&] { got[threadIdx.x] = rr_fold(f); },
      [&](int w) {
        // waves up to raiseAfterWave start first; then another block raises the flag; then the rest
        if (raiseAfterWave < 0) return;
        if (w <= raiseAfterWave) {
          ++early;
          return;
        }
        while (early < 64 * (raiseAfterWave + 1)) std::this_thread::yield();
        std::this_thread::sleep_for(std::chrono::milliseconds(20));
        if (there++ == 0) __atomic_store_n(&fl[FL_DONE], 1, __ATOMIC_SEQ_CST);
      });
  *returned = got[0];
  for (int g : got)
    if (g != got[0]) return 1;
  return 0;
}

int main() {
  int bad = 0;
  auto check = [&](bool ok, const char* what) {
    if (!ok) std::printf("wrong: %s\n", what), ++bad;
  };
  for (int nb : {1, 63, 300, 1100, 4096}) {
    std::vector<double> p(nb);
    double sum = 0.0;
    for (int i = 0; i < nb; ++i) sum += p[i] = 1.0 + i % 7;
    for (int block : {0, 3}) {
      for (bool meets : {false, true}) {
        double sc[16] = {};
        int fl[8] = {}, r = 0;
        sc[SC_NORMB] = 1.0;
        sc[SC_TOL] = std::sqrt(sum) * (meets ? 2.0 : 0.5);
        fl[FL_ITER] = 4;
        check(run(block, p.data(), nb, sc, fl, -1, &r) == 0 && r == meets, "the block's answer");
        check(fl[FL_DONE] == (block == 0 && meets) && fl[FL_ITER] == (block ? 4 : 5), "what block 0 leaves");
        if (block == 0) check(std::fabs(sc[SC_RR] / sum - 1) < 1e-15 * nb, "the sum");
      }
      double sc[16] = {};
      int fl[8] = {}, r = 0;
      sc[SC_NORMB] = 1.0;
      sc[SC_TOL] = 2.0 * std::sqrt(sum);
      fl[FL_DONE] = 1;  // an iteration after the last one
      fl[FL_ITER] = fl[FL_ITS] = 9;
      p[0] = NAN;
      check(run(block, p.data(), nb, sc, fl, -1, &r) == 0 && r == 1, "a solve that has ended");
      check(fl[FL_ITER] == 9 && fl[FL_ITS] == 9, "its iteration count");
      p[0] = 1.0;
    }
    // another block ends the solve while this one's later waves have yet to start
    for (int after : {0, 2}) {
      double sc[16] = {};
      int fl[8] = {}, r = 0;
      sc[SC_NORMB] = 1.0;
      sc[SC_TOL] = 2.0 * std::sqrt(sum);
      check(run(3, p.data(), nb, sc, fl, after, &r) == 0 && r == 1, "a flag raised inside a block's start");
    }
  }
  return bad != 0;
}
