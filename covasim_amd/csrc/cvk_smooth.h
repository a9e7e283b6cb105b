// The smoothing of r_eff (sim.py:898-952), by all threads of a workgroup.
#pragma once

namespace cvk {

// out = raw convolved `rounds` times with (0.25, 0.5, 0.25), zero beyond the ends (np.convolve 'same'), the days nearer
// than `rounds` to either end keeping raw's value (also where the two ends overlap). T >= 3 days; thread `first` of
// `step` takes days first, first + step, ..; on entry it has written raw at those days and nobody reads tmp. sync: the
// workgroup's barrier. out and tmp are written in turn, each round reading its neighbours' days of the other.
template <class Sync>
__host__ __device__ inline void smooth_days(int T, int rounds, int first, int step, const double* raw, double* out,
                                            double* tmp, const Sync& sync) {
  for (int t = first; t < T; t += step) out[t] = raw[t];
  const double* from = out;
  double* to = tmp;
  for (int r = 0; r < rounds; ++r) {
    sync();
    for (int t = first; t < T; t += step) {
      double acc;
      if (t == 0) acc = from[0] * 0.5 + from[1] * 0.25;
      else if (t == T - 1) acc = from[T - 2] * 0.25 + from[T - 1] * 0.5;
      else acc = from[t - 1] * 0.25 + from[t] * 0.5 + from[t + 1] * 0.25;
      to[t] = acc;
    }
    double* swap = to;
    to = const_cast<double*>(from);
    from = swap;
  }
  sync();  // after an odd count of rounds the last one has read the neighbours' days of out, overwritten now
  for (int t = first; t < T; t += step) {
    if (t < rounds || t >= T - rounds) out[t] = raw[t];
    else if (from != out) out[t] = from[t];
  }
}

}  // namespace cvk
