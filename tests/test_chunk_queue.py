"""The chunk queue of the generated kernels (device/mapx_dev.hiph, work distribution): its device text compiled for
the host, a work-group a thread-0 at a time in random order. A take takes effect when its result is used, the last
one of a work-group, whose result nobody uses, as late as it can: launch after launch every chunk has to be dealt
out once and the queue to be left at zero. On the GPU, statistics of a batch against its rasters alone."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "map_amd", "csrc", "device", "mapx_dev.hiph")

HARNESS = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <vector>
#define __device__
#define __forceinline__ inline
typedef unsigned int u32;
struct Dim { unsigned x; };
static Dim gridDim, blockIdx, threadIdx{0};
static std::map<unsigned, u32*> late;  // per work-group: the counter of a take that has not landed
static void land() {
  auto it = late.find(blockIdx.x);
  if (it != late.end()) { ++*it->second; late.erase(it); }
}
static u32* finished;
static u32 atomicAdd(u32* p, u32 v) {
  if (p == finished) { u32 d = *p; *p += v; return d; }  // its result is used at once
  land();  // the take before: its result has just been used
  u32 d = *p;
  for (auto& l : late) d += l.second == p;
  late[blockIdx.x] = p;
  return d;
}
static void atomicExch(u32* p, u32 v) { *p = v; }
static void __syncthreads() {}
static int readfirstlane(int v) { return v; }
#define __builtin_amdgcn_readfirstlane readfirstlane
static void landed() { land(); }
@SECTION@
int main(int argc, char** argv) {
  const int grid = atoi(argv[1]), n = atoi(argv[2]);
  std::vector<u32> q(9 * kQueueLine, 0u);
  finished = &q[8 * kQueueLine];
  gridDim.x = grid;
  std::mt19937 rng(grid + n);
  for (int launch = 0; launch < 3; launch++) {
    std::vector<Sched> sc(grid);
    std::vector<int> slot(grid), at(grid, -2), seen(n, 0), run;
    for (int g = 0; g < grid; g++) {
      sc[g].q = q.data(); sc[g].n = n; sc[g].s = &slot[g];
      run.push_back(g);
    }
    while (!run.empty()) {
      const size_t i = rng() % run.size();
      const int g = run[i];
      blockIdx.x = g;
      const int c = at[g] == -2 ? sched_first(sc[g]) : sched_next(sc[g], at[g]);
      if (c <= at[g]) return 1;  // chunk numbers increase
      at[g] = c;
      if (c < n) { seen[c]++; continue; }
      sched_done(sc[g]);
      run[i] = run.back();
      run.pop_back();
    }
    for (auto& l : late) ++*l.second;  // the launch has ended
    late.clear();
    for (int c : seen) if (c != 1) return 2;
    for (u32 v : q) if (v) return 3;
  }
  return 0;
}
"""


def test_queue_deals_every_chunk_once_launch_after_launch(tmp_path):
    text = open(HEADER).read()
    part = text[text.index("// ---- work distribution"):]
    part = part[:part.index("// ---- ", 8)]
    src, exe = tmp_path / "s.cpp", tmp_path / "s"
    src.write_text(HARNESS.replace("@SECTION@", part))
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", str(src), "-o", str(exe)], check=True)
    for grid in (8, 16, 256):
        for n in (1, 7, 8, 9, 100, 4095, 4096, 4099, 20000):
            assert subprocess.run([str(exe), str(grid), str(n)], timeout=60).returncode == 0, (grid, n)


@pytest.mark.gpu
@pytest.mark.parametrize("n,side", [(6, 2000), (9, 300)])  # more than 4096 chunks (dealt out in runs of eight), and fewer
def test_batches_match_single_rasters(G, n, side):
    """Statistics of whole numbers (every sum exact) of rasters that go in one launch with the queue, evaluated twice."""
    rng = np.random.Generator(np.random.PCG64(n))
    outs, want = [], []
    for i in range(n):
        print("case batch", n, side, i, flush=True)
        h, w = side - 3 * i, side + 5 * i
        v = rng.integers(-100, 101, (h, w)).astype(np.float32)
        z = ((np.arange(w)[None] // 31 + np.arange(h)[:, None] // 17) % 16).astype(np.int32)
        R, Z = G.from_array(v, (512, 512)), G.from_array(z, (512, 512))
        alone = G.zstats(R + 0.0, Z, 16)
        G.eval(alone)
        want.append((alone.table(), np.bincount(z.ravel()), np.bincount(z.ravel(), v.ravel())))
        outs.append(G.zstats(R, Z, 16))
    for again in range(2):
        G.eval(*outs)
        for s, (t, count, total) in zip(outs, want):
            got = s.table()
            assert np.array_equal(got["count"], count) and np.array_equal(got["sum"], total)
            for k in ("sum", "min", "max", "count"):
                assert np.array_equal(got[k], t[k])
