// Runs perm.hpp's compose_swaps on the CPU, one host thread per GPU thread: reads
// "cnt, then cnt pairs (row, ipiv entry)", prints one "dst src" line per move.
#include <pthread.h>

#include <cstdint>
#include <cstdio>
#include <thread>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_readfirstlane(x) (x)
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
static inline int2 make_int2(int x, int y) { return int2{x, y}; }
static inline int min(int a, int b) { return a < b ? a : b; }
struct Idx { int x; };
static thread_local Idx threadIdx;
static pthread_barrier_t barrier;
static void __syncthreads() { pthread_barrier_wait(&barrier); }

#include "../zml_amd/csrc/perm.hpp"

int main() {
  constexpr int NS = 64;   // two waves
  alignas(16) static int2 ev[NS];
  static int node[2 * NS];
  int cnt = 0;
  if (scanf("%d", &cnt) != 1 || cnt < 0 || cnt > NS) return 2;
  for (int k = 0; k < NS; ++k) {
    int i = -1, ip = 0;
    if (k < cnt && scanf("%d %d", &i, &ip) != 2) return 2;
    ev[k] = k < cnt ? zmlhip::swap_entry(i, ip) : make_int2(-1, -1);
  }
  for (int k = 0; k < 2 * NS; ++k) node[k] = 2 * NS - 1 - k;   // whatever an earlier list left
  pthread_barrier_init(&barrier, nullptr, 2 * NS);
  struct Move { bool is; int dst, src; };
  std::vector<Move> moves(2 * NS);
  std::vector<std::thread> threads;
  for (int t = 0; t < 2 * NS; ++t)
    threads.emplace_back([&, t] {
      threadIdx.x = t;
      moves[t].is = zmlhip::compose_swaps<NS>(ev, cnt, node, moves[t].dst, moves[t].src);
    });
  for (auto& t : threads) t.join();
  for (const Move& m : moves)
    if (m.is) printf("%d %d\n", m.dst, m.src);
  return 0;
}
