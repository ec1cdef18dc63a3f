// Spreading scan (the reference's SpreadScan with SUM: runtime/dag/SpreadScan.cpp,
// runtime/skeleton/SpreadingSkeleton.cpp:288-388, runtime/task/SpreadingTask.cpp).
// Each cell c holds a D8 direction code dir[c] (1 E, 2 SE, 4 S, 8 SW, 16 W,
// 32 NW, 64 N, 128 NE; y grows south); its downstream cell is c + off(dir[c])
// when the code is one of the eight and the cell lies inside the raster. The
// total that flows through c is
//   T(c) = in(c) + sum of T(u) over the upstream neighbours u of c
// (the neighbours whose downstream cell is c, in the order y outer, x inner),
// in the raster's C type, and the result is out(c) = T(c) when c has a
// downstream cell: the amount that leaves c. A cell without one keeps the
// neutral value 0, as in the reference, whose iterations move the amounts
// downstream until nothing changes and add to each cell what leaves it.
//
// The reference iterates over the whole raster until it is stable (one
// step per cell of the longest flow path). Here every cell is computed once, by
// visits to 64x64 tiles: a work-group takes a tile whose upstream tiles have
// finished cells since its last visit, loads what its unfinished cells need into
// LDS, and walks from every cell whose upstream totals are all known, cell by
// cell downstream, until it leaves the tile or meets a cell that still waits for
// another one (the last walk to arrive goes on). Then it stores the new totals,
// publishes the tile's finished cells, and notifies the tiles they flow into,
// which go into a queue unless they are there already. The first visit of every
// tile is in the queue from the start.
//
// What bounds it: the latency of the walks' steps. A step is one round trip to
// LDS and the sums, 570 cycles, instead of the round trips to the coherence
// point (3 us a step) of walks over the whole raster, and the other totals of a
// cell come with it. A tile of a smooth DEM is visited 6 to 9 times (FIFO order
// batches the notifications while the queue is long), each time with some 10
// walks of up to 48 cells; the LDS of a tile lets 5 work-groups run per CU. The
// loads and stores of a visit, a tile of values and its words, take as long as
// the walks. 16384^2 cells F32: 16.8 ms (walks over the whole raster after a
// pass over 32x32 tiles: 38 ms); 2048^2: 0.91 ms (2.4 ms). Measured slower: a
// loop per walk (70 ms), one queue for all tiles (64 ms), tiles put off while
// they have one notification only (fewer visits, but as much time for the
// putting off).
//
// Each cell is computed exactly once and every sum follows the fixed neighbour
// order, so the result does not depend on the schedule. Every notification
// stands for a cell that has just finished, so the visits end. Cells on a
// direction cycle never have all their upstream totals; the last kernel gives
// them the 0 (the reference's iteration does not end for them).
#include "spread.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

#pragma clang fp contract(off)

namespace mapx {
namespace spread {

constexpr int NT = 256;

// Totals, finished bits and the queue move between work-groups (on any XCD)
// through the device's coherence point: relaxed agent-scope loads, stores and
// atomics, which pass the XCD-local L2. The order comes from the waits: a
// visit's totals have arrived before its finished bits are stored, and those
// before the notification; a reader loads the notification word, then the bits,
// then the totals, each after the one before has returned. A release / acquire
// pair at agent scope would write back or invalidate a whole L2 per visit.
template <class T> __device__ __forceinline__ T ld_agent(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void st_agent(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned add_agent(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned add_lds(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void or_lds(unsigned* p, unsigned v) {
  __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// every store of the wavefront has arrived
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// LDS operations of a wavefront run in order; the compiler keeps them so
__device__ __forceinline__ void keep_order() { asm volatile("" ::: "memory"); }
// `v` is used only after what comes before, so that loads behind it are issued before its wait
__device__ __forceinline__ void after_loads(unsigned& v) { asm volatile("" : "+v"(v) : : "memory"); }
__device__ __forceinline__ void nap() { __builtin_amdgcn_s_sleep(8); }
__device__ __forceinline__ void sync() { __syncthreads(); }
// keeps what depends on the thread's number alone from being hoisted out of the loop over
// the visits: the places of its 16 cells took 335 registers, one work-group per CU
__device__ __forceinline__ void anew(int& t) { asm volatile("" : "+v"(t)); }

// ---- visits (the text up to the next such line is also compiled for the host by its test) ----

struct Geo {
  int BS0, BS1, NB0, NB1, DS0, DS1;
};

// The block-tiled element index of cell (x, y) splits into a row term and a column
// term: ((by*NB0 + bx)*BS1 + ly)*BS0 + lx = rowt(y) + colt(x), with by, ly = y / BS1,
// y % BS1 and bx, lx = x / BS0, x % BS0.
__device__ __forceinline__ unsigned rowt(const Geo& g, int y) {
  const int by = y / g.BS1;
  return ((unsigned)by * g.NB0 * g.BS1 + (unsigned)(y - by * g.BS1)) * g.BS0;
}
__device__ __forceinline__ unsigned colt(const Geo& g, int x) {
  const int bx = x / g.BS0;
  return (unsigned)bx * g.BS1 * g.BS0 + (unsigned)(x - bx * g.BS0);
}

constexpr int TS = 64;              // tile side
constexpr int RH = TS + 2;          // side with the ring of neighbouring cells
constexpr int RS = RH;              // a row of the ring arrays
constexpr int NR = RH * RS + 2;     // their size: rows start at an odd place, so that cell pairs of the tile are dwords
constexpr int NRING = 4 * TS + 4;
__device__ __forceinline__ int place(int lx, int ly) { return (ly + 1) * RS + lx + 2; }  // -1..TS each

// What the work-groups share, in one scratch allocation.
struct Work {
  uint64_t* words;  // per tile: its cells' words (Lds::word), four a piece
  unsigned* done;   // finished cells: nty*TS rows of 2*ntx dwords
  unsigned* pend;   // per tile: notifications not yet answered (1 at the start: the first visit)
  // Tile k waits in queue k % nq, whose work-groups are those b with b % nq the same: one
  // queue's counters, hit by every visit, took longer than the visits (64 ms against 24 for
  // 16384^2 cells at the time; loads behind them on that memory channel waited as well).
  unsigned* queue;  // nq times cap entries: tile + 1, 0 free
  unsigned* ctl;    // per queue CTL words: visits taken, entries put, visits done
  unsigned nq, cap;
  int ntx, nty;
};
constexpr unsigned CTL = 64;       // 256 bytes a queue
constexpr unsigned MAX_QUEUES = 64;
__device__ __forceinline__ unsigned tiles_of(const Work& w, unsigned q) {  // of queue q
  return ((unsigned)w.ntx * (unsigned)w.nty - q + w.nq - 1u) / w.nq;
}

// Directions in the order of the bits 0..7: E SE S SW W NW N NE (code 1 << d).
__device__ __forceinline__ int dir_dx(int d) { return (d <= 1 || d == 7) - (d >= 3 && d <= 5); }
__device__ __forceinline__ int dir_dy(int d) { return (d >= 1 && d <= 3) - (d >= 5 && d <= 7); }
// 0..7, or 8 for a code that is none of the eight
__device__ __forceinline__ int dir_of(unsigned code) {
  return code != 0u && (code & (code - 1u)) == 0u ? 31 - __builtin_clz(code) : 8;
}
// Place of an upstream neighbour that flows along d in the order y outer, x inner:
// it lies at (-dx, -dy), so SE is first (above left), then S, SW, E, W, NE, N, NW.
__device__ __forceinline__ int up_place(int d) { return (int)((0x56742103u >> (4 * d)) & 15u); }
// Offset of that neighbour, and of the downstream cell along d, in the ring arrays.
__device__ __forceinline__ int up_off(int p) {
  const int q = p < 4 ? p : p + 1;
  return (q / 3 - 1) * RS + q % 3 - 1;
}
__device__ __forceinline__ int down_off(unsigned d) {
  // +1, RS+1, RS, RS-1, -1, -RS-1, -RS, -RS+1 as bytes
  static_assert(RS == 66, "the table below");
  return (int)(int8_t)(uint8_t)(0xbfbebdff41424301ull >> (8u * d));
}

// A cell's word, 16 bits: 0..7 its upstream neighbours by place, 8..11 how many of them are
// unfinished (15: the cell itself is finished), 12..15 its direction 0..7 inside the tile, or
// SINK (no downstream cell inside the raster) or where it leaves the tile: W, E, N, S or
// across the corner it lies in.
constexpr unsigned FINISHED = 0xf00u;
constexpr unsigned SINK = 8u, TO_W = 9u, TO_E = 10u, TO_N = 11u, TO_S = 12u, TO_CORNER = 13u;
// Bit (dy+1)*3 + dx+1 of the neighbouring tile that the cell at place `at` flows to.
__device__ __forceinline__ unsigned tile_bit(unsigned d, int at) {
  if (d < TO_CORNER) return d == TO_W ? 1u << 3 : d == TO_E ? 1u << 5 : d == TO_N ? 1u << 1 : 1u << 7;
  const int lx = (at - 2) % RS, ly = (at - 2) / RS - 1;
  return 1u << ((ly ? 6 : 0) + (lx ? 2 : 0));
}

template <class T>
struct Lds {
  T tot[NR];                // totals of finished cells, input values of the others
  union {                   // two words a dword, for the counts' atomics
    unsigned word2[NR / 2];
    uint16_t word[NR];
  };
  unsigned fin[RH][4];      // finished bits of the tile's rows and the ring's at the start: the dwords left, 0, 1, right
  unsigned fresh[TS * 2];   // cells finished by this visit
  unsigned unf[2];          // rows of the tile with an unfinished cell
  unsigned rt[RH], ct[RH];
  uint16_t list[4 * TS];    // places of the cells to start from
  unsigned nlist;
  unsigned notify;          // neighbours to notify, bit (dy+1)*3 + dx+1
  unsigned ticket, tile, served, sum;
};

// An entry's place is shared: a work-group can wait there with a ticket of a later lap, and an
// entry put late can meet the next lap's. So it goes into a free place, and out of its place, by
// compare-and-exchange: no entry is stored over another one or taken twice. Which of the
// work-groups that wait at a place gets which of its entries does not matter. The place of put n is
// free in the end: a queue holds a tile once, at most cap in all, so when put n has its number the
// ticket of put n - cap, and with it a work-group that empties the place, has been taken. (The
// builtin is the one that both compilers of this text know; its system scope adds nothing to
// agent scope here, and it is relaxed.)
__device__ __forceinline__ bool swap_entry(unsigned* slot, unsigned seen, unsigned v) {
  return __atomic_compare_exchange_n(slot, &seen, v, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED);
}
__device__ __forceinline__ void put(const Work& w, unsigned tile) {
  const unsigned q = tile % w.nq;
  unsigned* slot = w.queue + q * w.cap + add_agent(&w.ctl[q * CTL + 1], 1u) % w.cap;
  while (!swap_entry(slot, 0u, tile + 1u)) nap();
}

// Ring cell k of a tile: -1..TS in x and y.
__device__ __forceinline__ void ring_cell(int k, int& lx, int& ly) {
  if (k < RH) { lx = k - 1; ly = -1; }
  else if (k < 2 * RH) { lx = k - RH - 1; ly = TS; }
  else if (k < 2 * RH + TS) { lx = -1; ly = k - 2 * RH; }
  else { lx = TS; ly = k - 2 * RH - TS; }
}
// Edge cell k (of 4 * TS - 4).
__device__ __forceinline__ void edge_cell(int k, int& lx, int& ly) {
  lx = k < TS ? k : k < 2 * TS ? k - TS : k < 3 * TS - 2 ? 0 : TS - 1;
  ly = k < TS ? 0 : k < 2 * TS ? TS - 1 : k < 3 * TS - 2 ? k - 2 * TS + 1 : k - 3 * TS + 3;
}
template <class T> __device__ __forceinline__ bool finished(const Lds<T>& L, int lx, int ly) {  // at the start
  const int b = 32 + lx;
  return (L.fin[ly + 1][b >> 5] >> (b & 31)) & 1u;
}
// Which of a cell's eight neighbours were finished at the start, by place.
template <class T> __device__ __forceinline__ unsigned neighbours(const Lds<T>& L, int lx, int ly) {
  const int b = 31 + lx, k = b >> 5, sh = b & 31;
  unsigned r[3];
#pragma unroll
  for (int q = 0; q < 3; q++) r[q] = (unsigned)((((uint64_t)L.fin[ly + q][k + 1] << 32) | L.fin[ly + q][k]) >> sh) & 7u;
  return r[0] | (r[1] & 1u) << 3 | (r[1] & 4u) << 2 | r[2] << 5;
}

// bits ? v : a zero that leaves every sum as it is (-0 for floating types)
__device__ __forceinline__ unsigned only32(unsigned m, unsigned v, unsigned z) { return (v & m) | (z & ~m); }
template <class T> __device__ __forceinline__ T only(unsigned m, T v) { return (T)(v & (T)(int)m); }
template <> __device__ __forceinline__ float only<float>(unsigned m, float v) {
  unsigned u;
  __builtin_memcpy(&u, &v, 4);
  u = only32(m, u, 0x80000000u);
  __builtin_memcpy(&v, &u, 4);
  return v;
}
template <> __device__ __forceinline__ double only<double>(unsigned m, double v) {
  unsigned u[2];
  __builtin_memcpy(u, &v, 8);
  u[0] &= m;
  u[1] = only32(m, u[1], 0x80000000u);
  __builtin_memcpy(&v, u, 8);
  return v;
}

// The words of a tile's cells from the directions (its own and the ring's), on the first visit.
template <class T, int NTH>
__device__ void make_words(Lds<T>& L, const uint8_t* __restrict__ dir, const Geo& g, int x0, int y0, int t) {
#pragma unroll 4
  for (int i = t; i < TS * TS; i += NTH) {
    const int lx = i % TS, ly = i / TS;
    unsigned word = SINK << 12 | FINISHED;  // outside the raster
    if (x0 + lx < g.DS0 && y0 + ly < g.DS1) {
      unsigned d = (unsigned)dir_of(dir[L.rt[ly + 1] + L.ct[lx + 1]]);
      if (d < 8u) {
        const int nx = lx + dir_dx((int)d), ny = ly + dir_dy((int)d), x = x0 + nx, y = y0 + ny;
        const bool ox = nx < 0 || nx >= TS, oy = ny < 0 || ny >= TS;
        if (x < 0 || y < 0 || x >= g.DS0 || y >= g.DS1) d = SINK;
        else if (ox && oy) d = TO_CORNER;
        else if (ox) d = nx < 0 ? TO_W : TO_E;
        else if (oy) d = ny < 0 ? TO_N : TO_S;
      }
      word = d << 12;
    }
    L.word[place(lx, ly)] = (uint16_t)word;
  }
  sync();
  auto flows = [&](int lx, int ly, int d, bool done) {  // cell (lx, ly) of the tile or the ring flows along d
    const int cx = lx + dir_dx(d), cy = ly + dir_dy(d);
    if (cx < 0 || cx >= TS || cy < 0 || cy >= TS) return;
    const int c = place(cx, cy);
    add_lds(&L.word2[c >> 1], ((1u << up_place(d)) + (done ? 0u : 256u)) << (16 * (c & 1)));
  };
#pragma unroll 4
  for (int i = t; i < TS * TS; i += NTH) {
    const int lx = i % TS, ly = i / TS, d = (int)(L.word[place(lx, ly)] >> 12);
    if (d < 8) flows(lx, ly, d, false);
  }
  for (int k = t; k < NRING; k += NTH) {
    int lx, ly;
    ring_cell(k, lx, ly);
    const int x = x0 + lx, y = y0 + ly;
    if (x < 0 || y < 0 || x >= g.DS0 || y >= g.DS1) continue;
    const int d = dir_of(dir[L.rt[ly + 1] + L.ct[lx + 1]]);
    if (d < 8) flows(lx, ly, d, finished(L, lx, ly));
  }
  sync();
}

template <class T, int NTH>
__device__ void visit(Lds<T>& L, const T* __restrict__ in, const uint8_t* __restrict__ dir, T* out, const Work& w, const Geo& g,
                      unsigned tile, bool first, int t) {
  static_assert(NTH >= 2 * TS && NTH <= 4 * TS && NTH % TS == 0, "a dword of finished bits, an edge cell per thread");
  constexpr int ROWS = TS * TS / NTH, WPT = TS * TS / 4 / NTH;  // rows and pieces of words per thread
  const int tx = (int)(tile % (unsigned)w.ntx), ty = (int)(tile / (unsigned)w.ntx), x0 = tx * TS, y0 = ty * TS;
  const int DW = 2 * w.ntx;
  uint64_t* words = w.words + (size_t)tile * (TS * TS / 4);
  if (t == 0) L.notify = L.nlist = 0u;
  if (t < 2) L.unf[t] = 0u;
  if (t < 2 * TS) L.fresh[t] = 0u;
  for (int i = t; i < 2 * RH; i += NTH) {
    const int c = i % RH - 1;
    if (i < RH) L.rt[i] = y0 + c >= 0 && y0 + c < g.DS1 ? rowt(g, y0 + c) : 0u;
    else L.ct[i - RH] = x0 + c >= 0 && x0 + c < g.DS0 ? colt(g, x0 + c) : 0u;
  }
  sync();
  uint64_t word4[WPT];
  if (!first) {
#pragma unroll
    for (int j = 0; j < WPT; j++) word4[j] = ld_agent(&words[j * NTH + t]);
  }
  for (int i = t; i < RH * 4; i += NTH) {
    const int r = i >> 2, q = i & 3, y = y0 + r - 1, c = 2 * tx - 1 + q;
    unsigned f = 0u;
    if (y >= 0 && y < w.nty * TS && c >= 0 && c < DW) f = ld_agent(&w.done[(unsigned)y * (unsigned)DW + (unsigned)c]);
    if (q == 1 || q == 2) {  // cells outside the raster count as finished: nothing to do for them
      const int left = g.DS0 - (x0 + (q - 1) * 32);
      if (left < 32) f |= left <= 0 ? ~0u : ~0u << left;
      if (y >= g.DS1) f = ~0u;
      if (f != ~0u && r >= 1 && r <= TS) or_lds(&L.unf[(r - 1) >> 5], 1u << ((r - 1) & 31));
    }
    L.fin[r][q] = f;
  }
  if (!first) {
#pragma unroll
    for (int j = 0; j < WPT; j++) {
      const int k = j * NTH + t, c = place((k & 15) * 4, k >> 4) >> 1;
      L.word2[c] = (unsigned)word4[j];
      L.word2[c + 1] = (unsigned)(word4[j] >> 32);
    }
  }
  sync();
  // Values, every load in flight before the first is used: the rows with an unfinished cell
  // and those next to them, the finished cells of the ring.
  const int lx = t % TS, ly0 = t / TS;
  const uint64_t unf = (uint64_t)L.unf[1] << 32 | L.unf[0], need = unf | unf << 1 | unf >> 1;
  const unsigned ct = L.ct[lx + 1];
  const bool inx = x0 + lx < g.DS0;
  T val[ROWS];
#pragma unroll
  for (int j = 0; j < ROWS; j++) {
    const int ly = ly0 + j * (NTH / TS);
    val[j] = T(0);
    if ((need >> ly & 1u) && inx && y0 + ly < g.DS1) {
      const unsigned e = L.rt[ly + 1] + ct;
      val[j] = first ? in[e] : ld_agent(&out[e]);
    }
  }
  for (int k = t; k < NRING; k += NTH) {
    int rx, ry;
    ring_cell(k, rx, ry);
    const int x = x0 + rx, y = y0 + ry;
    if (x >= 0 && y >= 0 && x < g.DS0 && y < g.DS1 && finished(L, rx, ry)) L.tot[place(rx, ry)] = ld_agent(&out[L.rt[ry + 1] + L.ct[rx + 1]]);
  }
#pragma unroll
  for (int j = 0; j < ROWS; j++) L.tot[place(lx, ly0 + j * (NTH / TS))] = val[j];
  // The cells to start from: on the first visit those without an unfinished upstream cell;
  // later those of the tile's edge that the ring's newly finished cells complete (an inner
  // cell becomes ready by a walk).
  unsigned go = 0u;
  if (first) {
    make_words<T, NTH>(L, dir, g, x0, y0, t);
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
      const int ly = ly0 + j * (NTH / TS);  // a row's and a column's cells go to TS different threads
      if ((L.word[place((t - ly) & (TS - 1), ly)] & 0xf00u) == 0u) go |= 1u << j;
    }
  } else {
    for (int k = t; k < 4 * TS - 4; k += NTH) {
      int ex, ey;
      edge_cell(k, ex, ey);
      const int c = place(ex, ey);
      const unsigned word = L.word[c];
      if ((word & 0xf00u) == FINISHED) continue;
      unsigned left = 0u;
      for (unsigned u = word & 0xffu & ~neighbours(L, ex, ey); u; u &= u - 1u) left++;
      L.word[c] = (uint16_t)((word & 0xf0ffu) | left << 8);
      if (left == 0u) L.list[add_lds(&L.nlist, 1u)] = (uint16_t)c;
    }
  }
  sync();
  const bool idle = !first && L.nlist == 0u;
  // Walks. One loop for all of a thread's: it goes to its next cell to start from as soon as a
  // walk ends (a loop per walk would run as long as the longest of the wavefront's each time).
  // Few starts, of a later visit, stay in the first wavefronts.
  bool on = first ? go != 0u : (unsigned)t < L.nlist;
  auto next_start = [&]() {
    const int ly = ly0 + (NTH / TS) * (31 - __builtin_clz(go & (0u - go)));
    go &= go - 1u;
    return place((t - ly) & (TS - 1), ly);
  };
  int at = place(0, 0);
  if (on) at = first ? next_start() : (int)L.list[t];
  unsigned c = L.word[at], told = 0u;
  T up[8], acc = L.tot[at];
#pragma unroll
  for (int p = 0; p < 8; p++) up[p] = L.tot[at + up_off(p)];
  while (on) {
#pragma unroll
    for (int p = 0; p < 8; p++) acc = (T)(acc + only<T>(0u - (c >> p & 1u), up[p]));
    L.tot[at] = acc;
    L.word[at] = (uint16_t)(c | FINISHED);
    const unsigned d = c >> 12;
    bool go_on = d < SINK;
    if (go_on) {
      // The count of the next cell falls after the total is in LDS, and its values are read
      // after that, one round trip for all: when this was the last of its upstream cells,
      // the totals of the others were there before their own decrements.
      at += down_off(d);
      const int sh = 16 * (at & 1);
      keep_order();
      c = add_lds(&L.word2[at >> 1], 0u - (256u << sh));
      keep_order();
      acc = L.tot[at];
#pragma unroll
      for (int p = 0; p < 8; p++) up[p] = L.tot[at + up_off(p)];
      after_loads(c);
      c = c >> sh & 0xffffu;
      go_on = (c & 0xf00u) == 0x100u;
    } else if (d > SINK) {
      told |= tile_bit(d, at);
    }
    if (!go_on) {
      on = go != 0u;
      if (on) {
        at = next_start();
        c = L.word[at];
        acc = L.tot[at];
#pragma unroll
        for (int p = 0; p < 8; p++) up[p] = L.tot[at + up_off(p)];
      }
    }
  }
  if (told) or_lds(&L.notify, told);
  sync();
  // the new totals (a cell without a downstream cell keeps 0), all cells on the first visit; the changed words
#pragma unroll 4
  for (int j = 0; j < ROWS && !idle; j++) {
    const int ly = ly0 + j * (NTH / TS);
    if (!(unf >> ly & 1u) || !inx || y0 + ly >= g.DS1) continue;
    const unsigned word = L.word[place(lx, ly)];
    const bool f = (word & 0xf00u) == FINISHED && !finished(L, lx, ly);
    if (f) or_lds(&L.fresh[2 * ly + (lx >> 5)], 1u << (lx & 31));
    if (f || first) st_agent(&out[L.rt[ly + 1] + ct], f && word >> 12 == SINK ? T(0) : L.tot[place(lx, ly)]);
  }
#pragma unroll
  for (int j = 0; j < WPT; j++) {
    const int k = j * NTH + t, c2 = place((k & 15) * 4, k >> 4) >> 1;
    const uint64_t now = (uint64_t)L.word2[c2 + 1] << 32 | L.word2[c2];
    if (first || now != word4[j]) st_agent(&words[k], now);
  }
  wait_stores();
  sync();
  if (t < 2 * TS && L.fresh[t])
    st_agent(&w.done[(unsigned)(y0 + (t >> 1)) * (unsigned)DW + (unsigned)(2 * tx + (t & 1))], L.fin[(t >> 1) + 1][1 + (t & 1)] | L.fresh[t]);
  wait_stores();
  sync();
  if (t < 9 && (L.notify >> t & 1u)) {
    const unsigned n = (unsigned)((ty + t / 3 - 1) * w.ntx + tx + t % 3 - 1);
    if (add_agent(&w.pend[n], 1u) == 0u) put(w, n);
  }
  wait_stores();
  sync();
  if (t == 0) {
    const unsigned s = L.served;
    if (add_agent(&w.pend[tile], 0u - s) != s) put(w, tile);  // notified during the visit
    wait_stores();  // what this visit put is counted before the visit is counted as done
    add_agent(&w.ctl[tile % w.nq * CTL + 2], 1u);
  }
}

// No visit is going on or waiting: as many are done as there were to start with and were put.
// Both only grow, and the done ones are read first, so equal sums were equal at a moment
// between the two readings. (By the threads t < MAX_QUEUES of a work-group.)
template <class T>
__device__ bool all_done(Lds<T>& L, const Work& w, int t) {
  sync();
  if (t == 0) L.sum = (unsigned)w.ntx * (unsigned)w.nty;
  sync();
  if ((unsigned)t < w.nq) add_lds(&L.sum, 0u - ld_agent(&w.ctl[(unsigned)t * CTL + 2]));
  sync();
  if ((unsigned)t < w.nq) add_lds(&L.sum, ld_agent(&w.ctl[(unsigned)t * CTL + 1]));
  sync();
  return L.sum == 0u;
}

template <class T, int NTH>
__device__ void visits(Lds<T>& L, const T* __restrict__ in, const uint8_t* __restrict__ dir, T* out, const Work& w, const Geo& g, unsigned group,
                       int t) {
  const unsigned q = group % w.nq, ntiles = tiles_of(w, q);
  for (;;) {
    sync();
    if (t == 0) L.ticket = add_agent(&w.ctl[q * CTL], 1u);
    sync();
    const unsigned k = L.ticket;
    const bool first = k < ntiles;  // the first visits are the first tickets
    unsigned* slot = w.queue + q * w.cap + (first ? 0u : (k - ntiles) % w.cap);
    for (;;) {
      if (t == 0) {
        unsigned v = first ? k * w.nq + q + 1u : 0u;
        for (int r = 0; !first && v == 0u && r < 16; r++) {
          v = ld_agent(slot);
          if (v && !swap_entry(slot, v, 0u)) v = 0u;
          if (!v) nap();
        }
        L.tile = v;
        // read before the finished bits: what is notified later is another visit's
        if (v) L.served = ld_agent(&w.pend[v - 1u]);
      }
      sync();
      if (L.tile) break;
      if (all_done(L, w, t)) return;
    }
    const unsigned tile = L.tile - 1u;
    sync();
    anew(t);
    visit<T, NTH>(L, in, dir, out, w, g, tile, first, t);
  }
}

// ---- end of the visits ----

template <class T>
__global__ void __launch_bounds__(NT, sizeof(T) == 8 ? 3 : 5) k_visit(const T* __restrict__ in, const uint8_t* __restrict__ dir, T* out, Work w, Geo g) {
  __shared__ Lds<T> L;
  visits<T, NT>(L, in, dir, out, w, g, blockIdx.x, (int)threadIdx.x);
}

// Clears the finished bits and the queue, and queues every tile's first visit.
__global__ void __launch_bounds__(NT) k_start(Work w) {
  const unsigned e = blockIdx.x * NT + threadIdx.x, tiles = (unsigned)w.ntx * (unsigned)w.nty;
  if (e < tiles * (unsigned)(TS * 2)) w.done[e] = 0u;
  if (e < tiles) w.pend[e] = 1u;
  if (e < w.nq * w.cap) w.queue[e] = 0u;
  if (e < w.nq * CTL) w.ctl[e] = 0u;
}

// Cells that no visit finished lie on or below a direction cycle: 0.
template <class T> __global__ void __launch_bounds__(NT) k_cycles(T* out, Work w, Geo g) {
  const unsigned e = blockIdx.x * NT + threadIdx.x, DW = 2u * (unsigned)w.ntx;
  const int y = (int)(e / DW), x = (int)(e % DW) * 32;
  if (y >= g.DS1 || x >= g.DS0) return;
  unsigned left = ~w.done[e];
  if (g.DS0 - x < 32) left &= ~(~0u << (g.DS0 - x));
  for (; left; left &= left - 1u) {
    const int b = 31 - __builtin_clz(left & (0u - left));
    out[rowt(g, y) + colt(g, x + b)] = T(0);
  }
}

static void check(hipError_t e, const char* w) {
  if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}

template <class T>
static void launch(void* out, const void* in, const void* dir, void* scratch, const Geo& g, hipStream_t s) {
  Work w;
  w.ntx = (g.DS0 + TS - 1) / TS;
  w.nty = (g.DS1 + TS - 1) / TS;
  const unsigned tiles = (unsigned)w.ntx * (unsigned)w.nty;
  int dev = 0, cus = 0, per_cu = 0;
  check(hipGetDevice(&dev), "hipGetDevice");
  check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
  check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(&k_visit<T>), NT, 0),
        "hipOccupancyMaxActiveBlocksPerMultiprocessor");
  const unsigned fit = (unsigned)((cus > 0 ? cus : 1) * (per_cu > 0 ? per_cu : 1)), groups = tiles < fit ? tiles : fit;
  w.nq = groups < MAX_QUEUES ? groups : MAX_QUEUES;  // every queue has work-groups
  w.cap = (tiles + w.nq - 1) / w.nq;
  w.words = (uint64_t*)scratch;
  w.done = (unsigned*)(w.words + (size_t)tiles * (TS * TS / 4));
  w.ctl = w.done + (size_t)tiles * (TS * 2);
  w.pend = w.ctl + MAX_QUEUES * CTL;
  w.queue = w.pend + tiles;
  if ((size_t)((char*)(w.queue + (size_t)w.nq * w.cap) - (char*)scratch) > scratch_bytes(g.DS0, g.DS1))
    throw std::runtime_error("spread: the scratch is too small");
  // (at least nq * cap <= tiles + nq entries and nq * CTL counters to clear)
  const unsigned grid = (unsigned)(((size_t)tiles * (TS * 2) + MAX_QUEUES * CTL + NT - 1) / NT);
  hipLaunchKernelGGL(k_start, dim3(grid), dim3(NT), 0, s, w);
  check(hipGetLastError(), "spread start launch");
  hipLaunchKernelGGL((k_visit<T>), dim3(groups), dim3(NT), 0, s, (const T*)in, (const uint8_t*)dir, (T*)out, w, g);
  check(hipGetLastError(), "spread visit launch");
  hipLaunchKernelGGL((k_cycles<T>), dim3(grid), dim3(NT), 0, s, (T*)out, w, g);
  check(hipGetLastError(), "spread cycle launch");
}

int run(void* out, const void* in, const void* dir, void* scratch, int dt, int BS0, int BS1, int NB0, int NB1, int DS0,
        int DS1, void* stream) {
  if (BS0 <= 0 || BS1 <= 0 || NB0 <= 0 || NB1 <= 0 || DS0 <= 0 || DS1 <= 0 || DS0 > NB0 * BS0 || DS1 > NB1 * BS1)
    throw std::runtime_error("spread: bad raster geometry");
  const Geo g{BS0, BS1, NB0, NB1, DS0, DS1};
  const uint64_t n = (uint64_t)BS0 * BS1 * NB0 * NB1;
  // element indices are 32-bit
  if (n >= (1ull << 32)) throw std::runtime_error("spread: rasters of 2^32 or more cells are not supported");
  hipStream_t s = (hipStream_t)stream;
  switch (dt) {  // DataTypeEnum: F32 1, F64 2, U8 4, U16 5, U32 6, U64 7, S8 8, S16 9, S32 10, S64 11
    case 1: launch<float>(out, in, dir, scratch, g, s); break;
    case 2: launch<double>(out, in, dir, scratch, g, s); break;
    case 4: launch<uint8_t>(out, in, dir, scratch, g, s); break;
    case 5: launch<uint16_t>(out, in, dir, scratch, g, s); break;
    case 6: launch<uint32_t>(out, in, dir, scratch, g, s); break;
    case 7: launch<uint64_t>(out, in, dir, scratch, g, s); break;
    case 8: launch<int8_t>(out, in, dir, scratch, g, s); break;
    case 9: launch<int16_t>(out, in, dir, scratch, g, s); break;
    case 10: launch<int32_t>(out, in, dir, scratch, g, s); break;
    case 11: launch<int64_t>(out, in, dir, scratch, g, s); break;
    default: throw std::runtime_error("spread: unsupported data type");
  }
  return 3;
}

}  // namespace spread
}  // namespace mapx
