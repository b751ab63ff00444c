// Random interleavings of waves that push and end the flights of a few histories
// while the last primaries start, with the kernel's counting rules (mt_counts.h).
// Prints the pushes to the queue, those that found a count below 1, those the check
// refused, and how many corrupted counts it refused while primaries were left.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "mt_counts.h"

int main(int argc, char** argv) {
  const int runs = argc > 1 ? std::atoi(argv[1]) : 1000;
  std::mt19937 rng(7);
  auto pick = [&](int n) { return int(rng() % unsigned(n)); };
  long long pushes = 0, below = 0, refused = 0, corrupt = 0, caught = 0;
  for (int r = 0; r < runs; ++r) {
    const int n_hist = 1 + pick(4), waves = 2 + pick(3);
    unsigned long long started = 0;
    std::vector<int> count(n_hist, 0);
    std::vector<char> counting(waves, 1);
    std::vector<unsigned long long> seen(waves, 0);  // the counter as each wave read it last
    std::vector<std::vector<int>> held(waves);       // flights of a wave, by history
    std::vector<int> queue;
    for (int step = 0; step < 200; ++step) {
      const int w = pick(waves);
      switch (pick(6)) {
        case 0:  // poll: reads the primaries' counter, then perhaps starts one
          seen[w] = started;
          if (seen[w] >= (unsigned long long)n_hist) counting[w] = 0;
          if (counting[w] && pick(3) == 0 && started < (unsigned long long)n_hist) {
            count[started] = 1;
            held[w].push_back(int(started++));
          }
          break;
        case 1:  // claim an entry; the poll that allowed it may be an old one
          if (!queue.empty()) {
            const int i = pick(int(queue.size()));
            held[w].push_back(queue[i]);
            queue.erase(queue.begin() + i);
          }
          break;
        case 2:  // a flight ends
          if (!held[w].empty()) {
            const int i = pick(int(held[w].size()));
            if (counting[w]) --count[held[w][i]];
            held[w].erase(held[w].begin() + i);
          }
          break;
        default:  // a recoil goes to the queue
          if (!held[w].empty()) {
            const int h = held[w][pick(int(held[w].size()))];
            const int before = counting[w] ? count[h]++ : 1;
            queue.push_back(h);
            ++pushes;
            below += before < 1;
            refused += !mt::count_possible(before, started, n_hist);
            if (started < (unsigned long long)n_hist) {  // had the count been lost
              ++corrupt;
              caught += !mt::count_possible(0, started, n_hist);
            }
          }
      }
    }
  }
  std::printf("pushes %lld\nbelow %lld\nrefused %lld\ncorrupt %lld\ncaught %lld\n", pushes, below, refused, corrupt, caught);
}
