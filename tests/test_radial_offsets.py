"""Bands along y keep a lane's row as a 32-bit byte offset from the wavefront's lowest row
(map_amd/csrc/radial.hip, mode LINES). The file's host code is compiled with g++ and its launches are caught: on
every geometry, blocks of 4 GiB and more among them, each wavefront of such a band has to span less than 2^32 bytes;
and blocks whose offsets fit keep the mode."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "map_amd", "csrc", "radial.hip")

HIP = r"""
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(n)
#define __restrict__
struct dim3 { unsigned x; dim3(unsigned v) : x(v) {} };
static dim3 threadIdx(0), blockIdx(0);
typedef int hipError_t;
typedef void* hipStream_t;
const int hipSuccess = 0;
static int hipGetLastError() { return 0; }
static const char* hipGetErrorString(int) { return ""; }
static float __int_as_float(int v) { float f; memcpy(&f, &v, 4); return f; }
static int __float_as_int(float f) { int v; memcpy(&v, &f, 4); return v; }
static double __hiloint2double(int, int) { return 0; }
static int __double2hiint(double) { return 0; }
static int __double2loint(double) { return 0; }
#define __builtin_amdgcn_readlane(v, l) (v)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_update_dpp(o, v, c, r, b, z) (v)
#define asm(...)
#define hipLaunchKernelGGL(kernel, grid, block, shared, stream, in, out, P) caught(P, (int)sizeof(*(in)))
struct Catch { template <class P> void operator()(const P& p, int bytes); };
static Catch caught;
"""

MAIN = r"""
static long long lines = 0, bad = 0;
template <class PP> void Catch::operator()(const PP& P, int bytes) {
  using namespace mapx::radial;
  for (int o = 0; o < 8; o++) {
    const Oct& O = P.oct[o];
    const int waves = P.first[o + 1] - P.first[o];
    if (O.mode != LINES || waves <= 0) continue;
    lines++;
    for (int w = 0; w < waves; w++) {  // rows (w - 1) * OWN .. of the wavefront, clamped as in the kernel
      int64_t lo = INT64_MAX, hi = INT64_MIN;
      for (int r = (w - 1) * OWN; r < (w + 1) * OWN; r++) {
        const int rc = r < 0 ? 0 : (r > O.L1 ? O.L1 : r);
        const int64_t t = colt(P, P.s0 + rc * O.sx);
        lo = t < lo ? t : lo;
        hi = t > hi ? t : hi;
      }
      bad += (hi - lo) * bytes >= (int64_t)1 << 32;
    }
  }
}
int main(int argc, char** argv) {
  int a[8];
  for (int i = 0; i < 8; i++) a[i] = atoi(argv[i + 1]);
  const int nb0 = (a[2] + a[0] - 1) / a[0], nb1 = (a[3] + a[1] - 1) / a[1];
  mapx::radial::run(nullptr, nullptr, a[6], 2, a[0], a[1], nb0, nb1, a[2], a[3], a[4], a[5], nullptr);
  printf("%lld %lld\n", lines, bad);
}
"""


@pytest.mark.parametrize("bs,ds,s,size,used", [
    ((32768, 32832), (40000, 300), (32700, 150), 4, False),   # more than 4 GiB from a block column to the next
    ((32768, 16448), (40000, 300), (32760, 299), 8, False),
    ((32768, 32768), (40000, 300), (32700, 150), 4, True),    # 4 GiB less a row
    ((64, 1 << 24), (400, 200), (70, 100), 4, False),         # two and three block columns in a wavefront
    ((16, 1 << 24), (100, 200), (8, 100), 4, False),
    ((32768, 32768), (32768, 300), (100, 150), 4, True),      # one block column: consecutive cells
    ((16384, 32768), (20000, 300), (16380, 150), 4, True),    # 2 GiB
    ((1024, 1024), (3000, 2100), (1500, 900), 4, True),
    ((32, 32), (300, 200), (150, 100), 8, True)])
def test_row_offsets_fit_32_bits(bs, ds, s, size, used, tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src, exe = tmp_path / "r.cpp", tmp_path / "r"
    text = open(SOURCE).read().replace("#pragma clang fp contract(off)", "")
    src.write_text(text + MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-I" + str(tmp_path), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)] + [str(v) for v in bs + ds + s] + [str(size), "0"], stdout=subprocess.PIPE, check=True).stdout.split()
    assert int(out[1]) == 0, "a wavefront's rows span 2^32 bytes or more"
    if size == 8 or bs[1] % 64 == 0:
        assert (int(out[0]) > 0) == used
