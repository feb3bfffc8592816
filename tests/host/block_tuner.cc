// Host build of the ensembles' workgroup tuner (mahyco_amd/csrc/block_tuner.hpp)
// for tests/test_block_tuner.py.  Three kernels, four candidates, two steps per
// candidate: kernel 0 runs in every step, kernel 1 only in the second step of a
// candidate (its event still holds the last launch's time in the others), kernel 2
// only in the first step of all.  Reads the candidates' times of kernels 0 and 1 from
// the command line and prints the three picks and the sample counts of kernel 1.
#include <cstdio>
#include <cstdlib>

#include "block_tuner.hpp"

int main(int, char** argv) {
  mhy::BlockTuner<3, 4> t;
  double event[3] = {0.0, 0.0, 0.0};  // time between each kernel's two events
  for (int step = 0; step < 8; ++step) {
    const int c = step / 2;
    t.begin();
    auto launch = [&](int k, double ms) { t.launched(k), event[k] = ms; };
    launch(0, std::atof(argv[1 + c]));
    if (step % 2 == 1) launch(1, std::atof(argv[5 + c]));
    if (step == 0) launch(2, 1.0);
    for (int k = 0; k < 3; ++k)
      if (t.timed[k]) t.add(k, c, event[k]);
  }
  std::printf("%d %d %d\n", t.pick(0), t.pick(1), t.pick(2));
  std::printf("%d %d %d %d\n", t.samples[1][0], t.samples[1][1], t.samples[1][2], t.samples[1][3]);
}
