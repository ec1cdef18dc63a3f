"""Bit chains (device/mapx_dev.hiph, codegen's bit_rule, the runtime's chains): a 3x3 rule on 0/1 rasters
applied generation after generation on a bit-packed copy, against the oracle and the per-group path.

On the CPU the device text of one generation runs with the 64 lanes of a wavefront in one value (g++), strip
by strip and launch by launch as the step kernel does, for every rule the generator accepts here."""
import json
import os
import subprocess

import numpy as np
import pytest

from map_amd import workloads as W
from parity import assert_exact

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "map_amd", "csrc", "device", "mapx_dev.hiph")


def majority(M, s, n):
    for _ in range(n):
        s = M.astype(M.convolve(s, [[1, 1, 1]] * 3) > 4, M.U8)
    return s


def shifted(M, s, n):
    """Two windows, a neighbour and a conditional; the mask is one row of a column."""
    for _ in range(n):
        a = M.convolve(s, [[0, 1, 0], [1, 0, 1], [0, 1, 0]])
        b = M.convolve(s, [[1], [0], [1]])
        s = M.astype(M.con((a == 2) ^ (b == 1), s([1, -1]), s == 0), M.U8)
    return s


RULES = {"life": W.life, "majority": majority, "shifted": shifted}

HARNESS = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#define __device__
#define __forceinline__ inline
typedef unsigned int u32;
struct V64 {
  u32 a[64];
  V64() {}
  V64(u32 v) { for (u32& x : a) x = v; }
};
#define OP(o) static V64 operator o(const V64& p, const V64& q) { V64 r; for (int i = 0; i < 64; i++) r.a[i] = p.a[i] o q.a[i]; return r; }
OP(&) OP(|) OP(^)
static V64 operator~(const V64& p) { V64 r; for (int i = 0; i < 64; i++) r.a[i] = ~p.a[i]; return r; }
static V64 operator<<(const V64& p, int n) { V64 r; for (int i = 0; i < 64; i++) r.a[i] = p.a[i] << n; return r; }
static V64 operator>>(const V64& p, int n) { V64 r; for (int i = 0; i < 64; i++) r.a[i] = p.a[i] >> n; return r; }
static V64 lane_prev(const V64& p) { V64 r(0u); for (int i = 1; i < 64; i++) r.a[i] = p.a[i - 1]; return r; }
static V64 lane_next(const V64& p) { V64 r(0u); for (int i = 0; i < 63; i++) r.a[i] = p.a[i + 1]; return r; }
namespace mx {
@SECTION@
}
@RULE@
int main(int argc, char** argv) {
  const int W = atoi(argv[1]), H = atoi(argv[2]), BS0 = atoi(argv[3]), BS1 = atoi(argv[4]), total = atoi(argv[5]);
  constexpr int R = @R@, K = 8, NR = R + 2 * K;
  const int WD = (W + 31) / 32, nsx = (WD + 61) / 62;
  std::vector<u32> in((size_t)WD * H, 0u), out(in);
  for (int y = 0; y < H; y++)
    for (int x = 0; x < W; x++) in[(size_t)y * WD + x / 32] |= (u32)(getchar() & 1) << (x % 32);
  for (int done = 0; done < total; done += K) {
    const int gens = total - done < K ? total - done : K;
    for (int sy = 0; sy * R < H; sy++)
      for (int sx = 0; sx < nsx; sx++) {
        const int y0 = sy * R - K;
        V64 v[NR];
        mx::BitEdge<V64> e;
        e.H = H;
        for (int l = 0; l < 64; l++) {
          const int col = sx * 62 - 1 + l, cl = col < 0 ? 0 : (col >= WD ? WD - 1 : col), cb = cl % (BS0 / 32);
          for (int i = 0; i < NR; i++) {
            const int y = y0 + i, yc = y < 0 ? 0 : (y >= H ? H - 1 : y);
            v[i].a[l] = in[(size_t)yc * WD + cl];
          }
          e.x0.a[l] = col == 0;
          e.x1.a[l] = col == WD - 1 ? 1u << ((W - 1) & 31) : 0u;
          e.b0.a[l] = cb == 0;
          e.b1.a[l] = col == WD - 1 ? e.x1.a[l] : (cb == BS0 / 32 - 1 ? 0x80000000u : 0u);
        }
        const bool edge = sx == 0 || sx * 62 + 62 >= WD - 1 || y0 <= 0 || y0 + NR >= H;
        mx::BitSeams<NR> seams = {};
        for (int i = 0; i < NR; i++) {
          seams.up[i / 32] |= (u32)mx::bit_seam(y0 + i, H, BS1, false) << (i % 32);
          seams.down[i / 32] |= (u32)mx::bit_seam(y0 + i, H, BS1, true) << (i % 32);
        }
        for (int t = 0; t < gens; t++) {
          if (edge) mx::bit_generation<V64, Rule, NR, true>(v, e, y0, seams);
          else mx::bit_generation<V64, Rule, NR, false>(v, e, y0, seams);
        }
        for (int l = 1; l <= 62; l++)
          for (int i = 0; i < R; i++)
            if (sx * 62 - 1 + l < WD && y0 + K + i < H) out[(size_t)(y0 + K + i) * WD + sx * 62 - 1 + l] = v[K + i].a[l];
      }
    in.swap(out);
  }
  for (int y = 0; y < H; y++)
    for (int x = 0; x < W; x++) putchar((int)(in[(size_t)y * WD + x / 32] >> (x % 32) & 1u));
}
"""


def bit_rule(M, script):
    p = M.plan(script(M, M.from_array(np.zeros((40, 40), np.uint8), (32, 32)), 3))
    rules = {g["bit_rule"] for g in p["groups"] if "bit_rule" in g}
    assert len(rules) <= 1, rules
    return rules.pop() if rules else None


@pytest.mark.parametrize("name", sorted(RULES))
def test_generation_matches_the_oracle(M, O, name, tmp_path):
    text = open(HEADER).read()
    section = text[text.index("template <class V> struct BitRow"):text.index("// Geometry of a bit chain")]
    rule = bit_rule(M, RULES[name])
    assert rule, name
    rule = rule[rule.index("struct Rule"):rule.index("}  // namespace")]
    for rows in (4, 16, 80):
        src, exe = tmp_path / "h.cpp", tmp_path / "h"
        src.write_text(HARNESS.replace("@SECTION@", section).replace("@RULE@", rule).replace("@R@", str(rows)))
        subprocess.run(["g++", "-O0", "-std=c++17", "-w", str(src), "-o", str(exe)], check=True)
        # one dword and less, ragged columns and rows, blocks of one row, seams, several strips each way
        for w, h, bs, gens in ((5, 3, (32, 4), 9), (32, 32, (32, 32), 3), (70, 90, (32, 1), 11), (131, 77, (64, 16), 17),
                               (300, 150, (96, 64), 8), (2100, 40, (1024, 32), 10), (4001, 35, (512, 16), 9)):
            a = (np.random.default_rng(w + h).random((h, w)) < 0.4).astype(np.uint8)
            r = subprocess.run([str(exe)] + [str(v) for v in (w, h, bs[0], bs[1], gens)], input=a.tobytes(), stdout=subprocess.PIPE,
                               check=True)
            want = RULES[name](O, O.from_array(a, bs), gens).val
            assert_exact(np.frombuffer(r.stdout, np.uint8).reshape(h, w), want, "%s %dx%d blocks %s, %d rows" % (name, w, h, bs, rows))


@pytest.mark.parametrize("name,script", [
    ("a value above 1", lambda M, s, n: M.convolve(s, W.LIFE_MASK) + s),
    ("a weight above 1", lambda M, s, n: M.astype(M.convolve(s, [[1, 2, 1]]) > 2, M.U8)),
    ("a wide window", lambda M, s, n: M.astype(M.convolve(s, [[1] * 5]) > 2, M.U8)),
    ("a float", lambda M, s, n: M.astype(M.convolve(s, W.LIFE_MASK) * 0.5 > 1.0, M.U8)),
    ("division by a sum", lambda M, s, n: M.astype(M.convolve(s, W.LIFE_MASK) / (s + 0) == 2, M.U8)),
    ("a local group", lambda M, s, n: M.astype(s == 0, M.U8))])
def test_groups_that_are_no_bit_rule(M, name, script):
    assert bit_rule(M, script) is None, name


def per_group(G, make):
    """The same script with the tile shape forced, which keeps to one kernel per group."""
    for k, v in (("tile_tx", 512), ("tile_ty", 16), ("tile_vx", 8)):
        G.set_option(k, v)
    try:
        return G.to_array(make())
    finally:
        for k in ("tile_tx", "tile_ty", "tile_vx"):
            G.set_option(k, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("w,h,bs,gens", [(5, 3, (32, 4), 9), (320, 256, (64, 64), 8), (1000, 517, (128, 64), 21), (2100, 300, (1024, 32), 16),
                                         (9000, 8300, (1024, 512), 10)])
def test_chains_match_the_groups(G, O, w, h, bs, gens, graph):
    print("case bit chain", w, h, bs, gens, graph, flush=True)
    a = (np.random.default_rng(w).random((h, w)) < 0.35).astype(np.uint8)
    G.set_option("graph", graph)
    try:
        for name, rule in sorted(RULES.items()):
            S = G.from_array(a, bs)
            l0 = G.stats()["launches"]
            got = G.to_array(rule(G, S, gens))
            assert G.stats()["launches"] - l0 == 2 + -(-gens // 8), name  # pack, steps, unpack
            S2 = G.from_array(a, bs)  # another node: nothing of the first evaluation is held
            assert_exact(got, per_group(G, lambda: rule(G, S2, gens)), name)
            if w * h < 1 << 20:
                assert_exact(got, rule(O, O.from_array(a, bs), gens).val, name + " (oracle)")
    finally:
        G.set_option("graph", 0)


@pytest.mark.gpu
def test_chains_fall_back_and_split(G, O):
    """Values above 1 anywhere (also beside cells the raster does not have) run the groups; a raster the
    caller keeps in the middle is there afterwards; chains of several boards run in one evaluation."""
    bs, gens = (64, 32), 12
    rng = np.random.default_rng(3)
    a = (rng.random((90, 150)) < 0.35).astype(np.uint8)
    for where in ((0, 0), (89, 149), (40, 70)):
        b = a.copy()
        b[where] = 2
        print("case fall back", where, flush=True)
        assert_exact(G.to_array(W.life(G, G.from_array(b, bs), gens)), O.life(b, bs, gens), "value 2 at %s" % (where,))
    mid = W.life(G, G.from_array(a, bs), 5)
    end = W.life(G, mid, 7)
    other = W.life(G, G.from_array(1 - a, bs), gens)
    G.eval(end, other)
    assert_exact(G.to_array(end), O.life(a, bs, gens), "end")
    assert_exact(G.to_array(other), O.life(1 - a, bs, gens), "other board")
    l0 = G.stats()["launches"]
    assert_exact(G.to_array(mid), O.life(a, bs, 5), "kept in the middle")
    assert G.stats()["launches"] == l0  # it was held
    # a chain whose input and output are rasters of the same evaluation
    c = W.life(G, G.astype(G.from_array(a * 3, bs) > 2, G.U8), gens)
    assert_exact(G.to_array(G.convolve(c, [[1, 2, 1]])), O.convolve(O.from_array(O.life(a, bs, gens), bs), [[1, 2, 1]]).val, "inside")
