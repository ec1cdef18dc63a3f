"""The tile queues of map_amd/csrc/spread.hip: their device text (put, the taking of tickets and entries, the end
test) compiled for the host with several work-groups per queue and stalls at every access of a queue's entries,
so that a store that comes a lap late meets the entry after it. The visits themselves are a stand-in that notifies
random tiles. Every tile that is put has to be visited once, by one work-group at a time, and the work-groups end."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "map_amd", "csrc", "spread.hip")

HARNESS = r"""
#include <pthread.h>
#include <sched.h>
#include <time.h>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#define __device__
#define __forceinline__ inline
static thread_local pthread_barrier_t* bar;
static thread_local uint64_t seed;
static unsigned rnd() { seed ^= seed << 13; seed ^= seed >> 7; seed ^= seed << 17; return (unsigned)(seed >> 20); }
static unsigned *q0, *q1;  // the queues' entries
static bool entry(const void* p) { return p >= q0 && p < q1; }
static void stall(const void* p) {
  if (!entry(p)) return;
  const unsigned r = rnd() % 64;
  if (r < 2) { timespec t = {0, 100000}; nanosleep(&t, 0); }
  else if (r < 16) sched_yield();
}
template <class T> T ld_agent(const T* p) { stall(p); T v = __atomic_load_n(p, __ATOMIC_SEQ_CST); stall(p); return v; }
template <class T> void st_agent(T* p, T v) {
  stall(p);
  const T old = __atomic_exchange_n(p, v, __ATOMIC_SEQ_CST);
  if (entry(p) && (old == 0) == (v == 0)) _Exit(v ? 6 : 5);  // an entry stored over another one, or taken twice
}
static bool stalled_cas(unsigned* p, unsigned* seen, unsigned v) {
  stall(p);
  return __atomic_compare_exchange_n(p, seen, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
}
#define __atomic_compare_exchange_n(p, seen, v, weak, s, f) stalled_cas(p, seen, v)
static unsigned add_agent(unsigned* p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
static unsigned add_lds(unsigned* p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
static void or_lds(unsigned* p, unsigned v) { __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST); }
static void wait_stores() {}
static void keep_order() {}
static void nap() { sched_yield(); }
static void anew(int&) {}
static void after_loads(unsigned&) {}
static void sync() { pthread_barrier_wait(bar); }
@BEFORE@
static std::vector<int> busy, visited;
static int budget;
template <class T, int NTH>
void visit(Lds<T>& L, const T*, const uint8_t*, T*, const Work& w, const Geo&, unsigned tile, bool, int t) {
  if (t == 0) {
    if (tile >= (unsigned)(w.ntx * w.nty) || __atomic_exchange_n(&busy[tile], 1, __ATOMIC_SEQ_CST)) _Exit(7);  // one visit of a tile at a time
    visited[tile]++;
    for (unsigned k = rnd() % 4; k > 0 && __atomic_fetch_sub(&budget, 1, __ATOMIC_SEQ_CST) > 0; k--) {
      const unsigned n = rnd() % (unsigned)(w.ntx * w.nty);
      if (n != tile && add_agent(&w.pend[n], 1u) == 0u) put(w, n);
    }
    busy[tile] = 0;
    const unsigned s = L.served;  // as at the end of a visit
    if (add_agent(&w.pend[tile], 0u - s) != s) put(w, tile);
    add_agent(&w.ctl[tile % w.nq * CTL + 2], 1u);
  }
  sync();
}
@AFTER@
int main(int argc, char** argv) {
  constexpr int NTH = @NTH@;
  Work w;
  w.ntx = atoi(argv[1]); w.nty = 1; w.nq = NTH;
  const int groups = atoi(argv[2]), tiles = w.ntx;
  budget = atoi(argv[4]);
  w.cap = (tiles + w.nq - 1) / w.nq;
  busy.assign(tiles, 0); visited = busy;
  std::vector<unsigned> pend(tiles, 1u), queue(w.nq * w.cap, 0u), ctl(w.nq * CTL, 0u);
  w.pend = pend.data(); w.queue = queue.data(); w.ctl = ctl.data();
  q0 = w.queue; q1 = q0 + queue.size();
  std::vector<std::thread> th;
  std::vector<pthread_barrier_t> bars(groups);
  const Geo g{};
  for (int b = 0; b < groups; b++) {
    pthread_barrier_init(&bars[b], 0, NTH);
    Lds<uint8_t>* L = new Lds<uint8_t>();
    for (int t = 0; t < NTH; t++)
      th.emplace_back([=, &bars] {
        bar = &bars[b];
        seed = (uint64_t)atoi(argv[3]) * 0x9e3779b97f4a7c15ull + b * 977 + t * 13 + 1;
        visits<uint8_t, NTH>(*L, nullptr, nullptr, nullptr, w, g, (unsigned)b, t);
      });
  }
  for (auto& x : th) x.join();
  for (unsigned v : queue) if (v) return 2;
  for (unsigned v : pend) if (v) return 3;
  unsigned puts = 0, done = 0, sum = 0;
  for (unsigned q = 0; q < w.nq; q++) { puts += ctl[q * CTL + 1]; done += ctl[q * CTL + 2]; }
  for (int v : visited) sum += v;
  return done == tiles + puts && sum == done ? 0 : 4;
}
"""


@pytest.mark.parametrize("queues,shapes", [(1, ((2, 2), (3, 3), (4, 4), (8, 5))), (2, ((4, 4), (5, 4), (8, 8)))])
def test_entries_are_taken_once(queues, shapes, tmp_path):
    text = open(SOURCE).read()
    text = text[text.index("// ---- visits"):text.index("// ---- end of the visits")]
    visit, after = text.index("template <class T, int NTH>\n__device__ void visit("), text.index("// No visit is going on")
    src, exe = tmp_path / "q.cpp", tmp_path / "q"
    src.write_text(HARNESS.replace("@BEFORE@", text[:visit]).replace("@AFTER@", text[after:]).replace("@NTH@", str(queues)))
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-w", str(src), "-o", str(exe), "-lpthread"], check=True)
    for tiles, groups in shapes:
        for seed in range(1, 4):
            r = subprocess.run([str(exe), str(tiles), str(groups), str(seed), "20000"], timeout=60)
            assert r.returncode == 0, (tiles, groups, seed, r.returncode)
