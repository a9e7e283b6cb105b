// smooth_days of covasim_amd/csrc/cvk_smooth.h on the CPU under the schedules that a workgroup's barriers allow and
// that show a missing one: the threads take turns, each running alone from one barrier to the next, in ascending or
// descending order. stdin: T rounds threads descending, then T values; stdout: the smoothed values.
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#define __host__
#define __device__
#include "cvk_smooth.h"

namespace {
std::mutex m;
std::condition_variable cv;
int n_threads = 0, descending = 0, turn = 0;

int place(int thread) { return descending ? n_threads - 1 - thread : thread; }
void wait_turn(int thread) {
  std::unique_lock<std::mutex> lock(m);
  cv.wait(lock, [&] { return turn % n_threads == place(thread); });
}
void pass_turn() {
  std::lock_guard<std::mutex> lock(m);
  ++turn;
  cv.notify_all();
}
}  // namespace

int main() {
  int T = 0, rounds = 0;
  if (std::scanf("%d %d %d %d", &T, &rounds, &n_threads, &descending) != 4 || T < 3 || n_threads < 1) return 2;
  std::vector<double> raw(T), out(T, -1.0), tmp(T, -2.0);
  for (double& x : raw)
    if (std::scanf("%lf", &x) != 1) return 2;
  std::vector<std::thread> threads;
  for (int k = 0; k < n_threads; ++k)
    threads.emplace_back([&, k] {
      wait_turn(k);
      cvk::smooth_days(T, rounds, k, n_threads, raw.data(), out.data(), tmp.data(), [&] {
        pass_turn();
        wait_turn(k);
      });
      pass_turn();
    });
  for (std::thread& t : threads) t.join();
  for (double x : out) std::printf("%.17g\n", x);
  return 0;
}
