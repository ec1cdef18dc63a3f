"""The tile visits of map_amd/csrc/spread.hip: their device text compiled for the host (g++, AddressSanitizer), a
thread per GPU thread and several work-groups at once, against the oracle; and the kernels on the GPU at the
edges of tiles and blocks."""
import os
import subprocess

import numpy as np
import pytest

from map_amd import workloads as W
from parity import assert_exact

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "map_amd", "csrc", "spread.hip")

HARNESS = r"""
#include <pthread.h>
#include <sched.h>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#define __device__
#define __forceinline__ inline
static thread_local pthread_barrier_t* bar;
template <class T> T ld_agent(const T* p) { return __atomic_load_n(p, __ATOMIC_SEQ_CST); }
static float ld_agent(const float* p) { uint32_t u = __atomic_load_n((const uint32_t*)p, __ATOMIC_SEQ_CST); float f; __builtin_memcpy(&f, &u, 4); return f; }
template <class T> void st_agent(T* p, T v) { __atomic_store_n(p, v, __ATOMIC_SEQ_CST); }
static void st_agent(float* p, float v) { uint32_t u; __builtin_memcpy(&u, &v, 4); __atomic_store_n((uint32_t*)p, u, __ATOMIC_SEQ_CST); }
static unsigned add_agent(unsigned* p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
static unsigned add_lds(unsigned* p, unsigned v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
static void or_lds(unsigned* p, unsigned v) { __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST); }
static void wait_stores() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }
static void keep_order() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }
static void nap() { sched_yield(); }
static void anew(int&) {}
static void after_loads(unsigned&) {}
static void sync() { pthread_barrier_wait(bar); }
@SECTION@
typedef @T@ T;
int main(int argc, char** argv) {
  Geo g;
  g.DS0 = atoi(argv[1]); g.DS1 = atoi(argv[2]); g.BS0 = atoi(argv[3]); g.BS1 = atoi(argv[4]);
  g.NB0 = (g.DS0 + g.BS0 - 1) / g.BS0; g.NB1 = (g.DS1 + g.BS1 - 1) / g.BS1;
  const size_t n = (size_t)g.BS0 * g.BS1 * g.NB0 * g.NB1;
  T *in = new T[n], *out = new T[n];
  uint8_t* dir = new uint8_t[n];
  if (fread(in, sizeof(T), n, stdin) != n || fread(dir, 1, n, stdin) != n) return 1;
  Work w;
  w.ntx = (g.DS0 + TS - 1) / TS; w.nty = (g.DS1 + TS - 1) / TS;
  const unsigned tiles = (unsigned)(w.ntx * w.nty);
  constexpr int NTH = 128, WGS = 2;
  w.nq = tiles < WGS ? 1 : WGS;
  w.cap = (tiles + w.nq - 1) / w.nq;
  std::vector<uint64_t> words(tiles * TS * TS / 4);
  std::vector<unsigned> done(tiles * 2 * TS, 0u), pend(tiles, 1u), queue(w.nq * w.cap, 0u), ctl(w.nq * CTL, 0u);
  w.words = words.data(); w.done = done.data(); w.pend = pend.data(); w.queue = queue.data(); w.ctl = ctl.data();
  std::vector<std::thread> th;
  pthread_barrier_t bars[WGS];
  Lds<T>* L[WGS];
  for (int b = 0; b < WGS; b++) {
    pthread_barrier_init(&bars[b], 0, NTH);
    L[b] = new Lds<T>();
    for (int t = 0; t < NTH; t++) th.emplace_back([=, &bars] { bar = &bars[b]; visits<T, NTH>(*L[b], in, dir, out, w, g, (unsigned)b, t); });
  }
  for (auto& x : th) x.join();
  for (unsigned v : queue) if (v) return 2;
  for (unsigned v : pend) if (v) return 3;
  unsigned puts = 0, visited = 0;
  for (unsigned q = 0; q < w.nq; q++) { puts += ctl[q * CTL + 1]; visited += ctl[q * CTL + 2]; }
  if (visited != tiles + puts) return 4;
  for (int y = 0; y < g.DS1; y++)
    for (int x = 0; x < g.DS0; x++)  // as the last kernel does
      if (!(done[(size_t)y * 2 * w.ntx + x / 32] >> (x % 32) & 1u)) out[rowt(g, y) + colt(g, x)] = T(0);
  fwrite(out, sizeof(T), n, stdout);
}
"""


def cases(w, h, seed):
    """Random codes (invalid ones, cycles and cells that flow out of the raster among them), directions of a
    rough surface, one path through the whole raster along its rows, and everything flowing one way."""
    rng = np.random.default_rng(seed)
    z = rng.random((h, w)) + np.hypot(*np.mgrid[0:h, 0:w]) * 0.5
    snake = np.full((h, w), 1, np.uint8)
    snake[1::2] = 16
    snake[0::2, -1] = 4
    snake[1::2, 0] = 4
    return {"random": rng.choice(np.array([0, 1, 2, 4, 8, 16, 32, 64, 128, 3, 255], np.uint8), (h, w)),
            "surface": W.d8_directions(z), "snake": snake, "east": np.full((h, w), 1, np.uint8),
            "north west": np.full((h, w), 32, np.uint8)}


def values(dt, w, h):
    rng = np.random.default_rng(9)
    return (rng.random((h, w)) * 3).astype(dt) if np.issubdtype(dt, np.floating) else rng.integers(0, 200, (h, w)).astype(dt)


@pytest.mark.parametrize("dt,ctype", [(np.float32, "float"), (np.uint8, "uint8_t"), (np.int64, "int64_t")])
def test_visits_match_the_oracle(O, dt, ctype, tmp_path):
    from map_amd import binfile
    text = open(SOURCE).read()
    section = text[text.index("// ---- visits"):text.index("// ---- end of the visits")]
    src, exe = tmp_path / "h.cpp", tmp_path / "h"
    src.write_text(HARNESS.replace("@SECTION@", section).replace("@T@", ctype))
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-w", "-fsanitize=address,undefined", str(src), "-o", str(exe), "-lpthread"], check=True)
    for w, h, bs in ((1, 1, (32, 32)), (64, 64, (64, 64)), (65, 129, (32, 16)), (150, 70, (128, 64))):
        for name, d in cases(w, h, w).items():
            v = values(dt, w, h)
            data = binfile.to_blocks(v, bs).tobytes() + binfile.to_blocks(d, bs, 1).tobytes()  # codes in the padding, too
            r = subprocess.run([str(exe)] + [str(x) for x in (w, h) + bs], input=data, stdout=subprocess.PIPE, timeout=100,
                               env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
            assert r.returncode == 0, (name, w, h, r.returncode)
            got = binfile.from_blocks(np.frombuffer(r.stdout, dt), (w, h), bs)
            want = O.spread_scan(O.from_array(v, bs), O.from_array(d, bs)).val
            assert_exact(got, want, "%s %dx%d %s" % (name, w, h, ctype))


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,bs", [(1, 1, (32, 32)), (64, 64, (64, 64)), (65, 63, (32, 16)), (129, 200, (128, 64)), (1000, 777, (256, 96))])
def test_visits_on_the_gpu(G, O, w, h, bs):
    for dt in (np.float32, np.float64, np.uint8, np.int16, np.int64):
        for name, d in cases(w, h, w).items():
            if name == "snake" and w * h > 30000:
                continue  # the oracle takes a front of cells at a time: minutes for a path of this length
            print("case visits", w, h, bs, np.dtype(dt).name, name, flush=True)
            v = values(dt, w, h)
            got = G.to_array(G.spread_scan(G.from_array(v, bs), G.from_array(d, bs)))
            assert_exact(got, O.spread_scan(O.from_array(v, bs), O.from_array(d, bs)).val, "%s %dx%d" % (name, w, h))
