// Which of a few workgroup counts each kernel of an ensemble step keeps: the
// candidate with the shortest mean time over the launches that were timed with
// it.  A step need not launch every kernel (x-first steps of the fixed options have
// no Lagrange kernel of their own, and the dt reduction runs only where the
// accumulators are empty), so a step's timings are those of the kernels marked since its
// begin(), and candidates are compared by mean, not by sum.  Host code only.
#pragma once

namespace mhy {

template <int KERNELS, int CANDIDATES>
struct BlockTuner {
  bool timed[KERNELS] = {};  // launched in the current step, in a form that candidates change
  double ms[KERNELS][CANDIDATES] = {};
  int samples[KERNELS][CANDIDATES] = {};

  // a tuning step starts
  void begin() {
    for (bool& t : timed) t = false;
  }
  // this step's launch of kernel k
  void launched(int k) { timed[k] = true; }
  // its time with candidate c (once per step)
  void add(int k, int c, double t) {
    ms[k][c] += t;
    ++samples[k][c];
  }
  // the candidate to keep: index 0, the default, where nothing measured faster
  int pick(int k) const {
    auto mean = [&](int c) { return ms[k][c] / samples[k][c]; };
    int best = 0;
    for (int c = 1; c < CANDIDATES; ++c)
      if (samples[k][c] > 0 && samples[k][best] > 0 && mean(c) < mean(best)) best = c;
    return best;
  }
};

}  // namespace mhy
