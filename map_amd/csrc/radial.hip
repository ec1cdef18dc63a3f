// Radial scan (the reference's RadialScan / RadiatingSkeleton,
// runtime/skeleton/RadiatingSkeleton.cpp:47-325, runtime/skeleton/util.cpp:543-616,
// runtime/task/RadiatingTask.cpp:133-271): for an observer cell s, every cell
// p gets R(p) = OP(base(p), in(p)) (in(p) skipped when not finite), where the
// plane around s is cut into 8 octants (first direction F, second S; the
// cells with d0 = (p-s).F >= d1 = (p-s).S >= 0) and
//   base(s) = neutral; base = R(p-F) on the F axis (d1 = 0); base = R(p-F-S)
//   on the diagonal (d1 = d0); else the ray's crossing of column d0-1,
//   a*w + b*(1-w), a = R(p-F), b = R(p-F-S), w = d1/d0*(d0-1) - (d1-1).
// Cells on an axis or a diagonal belong to two octants and get the same
// value from both.
//
// Column d0 of an octant depends only on column d0-1, so a launch advances
// every octant by one band of K columns. A wavefront owns 64 rows, one per lane
// (`b` below), and also runs the 64 rows before them (`a`: row r at column c
// needs rows r and r-1 at column c-1, so after K <= 64 columns the owned rows are
// exact); wavefronts never wait on each other, and a column needs no LDS and no
// barrier: the neighbouring row is one lane up. The band's inputs are loaded
// before the columns, its results stored after them to `out` (block-tiled, like
// every raster), from which the next band reads its starting column.
//
// What bounds it: the latencies of a launch, which with about one wavefront per
// SIMD nothing overlaps. Of a band's 18.5 us (16384^2 cells) the chain of columns
// is 5.7: 2 rows x 20 instructions a column, some 210 cycles of dependent ones. The
// other 12.9 are the launch itself, the loads before the first column and the stores
// after the last (measured with the columns left out). (One launch for all bands, with
// wavefronts that wait for the row before theirs, took as long: each hand-over costs
// what 16 columns do.)
// The division of the interpolation weight, d1/d0, is by a number that all rows
// of a column share: q = d1 * (1/d0), then q + (d1 - q d0) * (1/d0) with fused
// multiply-adds is the correctly rounded quotient (Markstein, IBM Journal of
// Research and Development 34, 1990); for F32 it was compared with the division
// for every d1 < d0 <= 65536, and larger rasters divide. Bands are aligned in the raster, so
// that one lies in a single row or column of blocks: along y its columns are a constant stride
// apart, and along x, where the rows are a block row apart, a row's K cells move as vectors.
// (Cell by cell, with a step through the blocks for each, the addresses took more instructions
// than the columns; that path is left for block sides that K does not divide and for blocks of
// gigabytes.)
// 16384^2 F32 from the centre: 2.4 ms, 18.7 us a band (a work-group of 256 rows exchanging
// columns through LDS with a barrier, cells moved one by one: 4.8 ms; a branch around the
// operation for inputs that are not finite, and the diagonal's selection in every band:
// 20 us a band).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

// every product and sum rounds on its own, as the generated kernels do (-ffp-contract=off)
#pragma clang fp contract(off)

namespace mapx {
namespace radial {

constexpr int NT = 256;        // threads per work-group (its wavefronts are on their own)
constexpr int OWN = 64;        // rows a wavefront owns
constexpr int QUICK_MAX = 65536;  // columns up to which the F32 quotient was compared

// How a band's cells are addressed: one after the other (any blocks); a band that lies in one
// row of blocks, its columns one block row apart (along y); or one column of blocks, its
// columns consecutive cells (along x, towards larger or smaller x).
enum Mode : int { CELLS = 0, LINES = 1, UP = 2, DOWN = 3 };

struct Oct {
  int fx, fy, sx, sy;  // unit vectors of the first and second directions
  int L0, L1;          // last column (along F) and last row (along S) inside the raster
  int mode;
  // this launch's band: position p (0..K-1) is column cb + p, for p0 <= p < p1
  int cb, p0, p1;
};

struct Params {
  int BS0, BS1, NB0, NB1;
  int s0, s1;          // observer cell
  Oct oct[8];
  int first[9];        // first wavefront of each octant in this launch; first[8] = total
};

// The block-tiled element index of cell (x, y) is rowt(y) + colt(x).
__device__ __forceinline__ int64_t rowt(const Params& P, int y) {
  const int by = y / P.BS1;
  return ((int64_t)by * P.NB0 * P.BS1 + (y - by * P.BS1)) * P.BS0;
}
__device__ __forceinline__ int64_t colt(const Params& P, int x) {
  const int bx = x / P.BS0;
  return (int64_t)bx * P.BS1 * P.BS0 + (x - bx * P.BS0);
}

// The term of a coordinate that steps along F.
struct Along {
  int64_t off, stride, jump;  // jump: from a block's last index to the next block's first, in steps of +1
  int i, B, f;
  __device__ __forceinline__ void init(const Params& P, bool x, int u, int dir) {
    B = x ? P.BS0 : P.BS1;
    i = u % B;
    f = dir;
    off = x ? colt(P, u) : rowt(P, u);
    stride = x ? 1 : P.BS0;
    jump = (x ? (int64_t)P.BS1 * P.BS0 : (int64_t)P.NB0 * P.BS1 * P.BS0) - (int64_t)(B - 1) * stride;
  }
  __device__ __forceinline__ void step() {
    i += f;
    int64_t d = f * stride;
    if (i == B) { i = 0; d = jump; }
    else if (i < 0) { i = B - 1; d = -jump; }
    off += d;
  }
};

enum Op { SUM = 0, PROD = 1, MAX = 2, MIN = 3 };

template <class T, int OP> __device__ __forceinline__ T neutral() {
  if (OP == SUM) return (T)0;
  if (OP == PROD) return (T)1;
  if (OP == MAX) return -__builtin_huge_val();
  return __builtin_huge_val();
}
// max and min as the instruction: for fmaxf / fminf the compiler quiets both operands first,
// which a NaN made by arithmetic is already (a signalling x is not finite and not combined)
__device__ __forceinline__ float vmax(float a, float b) { float r; asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }
__device__ __forceinline__ float vmin(float a, float b) { float r; asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }
template <int OP> __device__ __forceinline__ float combine(float b, float x) {
  if (OP == SUM) return b + x;
  if (OP == PROD) return b * x;
  if (OP == MAX) return vmax(b, x);
  return vmin(b, x);
}
template <int OP> __device__ __forceinline__ double combine(double b, double x) {
  if (OP == SUM) return b + x;
  if (OP == PROD) return b * x;
  if (OP == MAX) return fmax(b, x);
  return fmin(b, x);
}

// Lane i's value in every lane; the value of the lane before, in lane 0 `first` or 0.
__device__ __forceinline__ int lane_read(int v, int i) { return __builtin_amdgcn_readlane(v, i); }
__device__ __forceinline__ int lane_prev(int v, int first) { return __builtin_amdgcn_update_dpp(first, v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ int lane_prev(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_read(float v, int i) { return __int_as_float(lane_read(__float_as_int(v), i)); }
__device__ __forceinline__ float lane_prev(float v, float first) {
  return __int_as_float(lane_prev(__float_as_int(v), __float_as_int(first)));
}
__device__ __forceinline__ float lane_prev(float v) { return __int_as_float(lane_prev(__float_as_int(v))); }
__device__ __forceinline__ double lane_read(double v, int i) {
  return __hiloint2double(lane_read(__double2hiint(v), i), lane_read(__double2loint(v), i));
}
__device__ __forceinline__ double lane_prev(double v, double first) {
  return __hiloint2double(lane_prev(__double2hiint(v), __double2hiint(first)),
                          lane_prev(__double2loint(v), __double2loint(first)));
}
__device__ __forceinline__ double lane_prev(double v) {
  return __hiloint2double(lane_prev(__double2hiint(v)), lane_prev(__double2loint(v)));
}
__device__ __forceinline__ int64_t lane_read(int64_t v, int i) {
  const unsigned lo = (unsigned)lane_read((int)(unsigned)v, i), hi = (unsigned)lane_read((int)(v >> 32), i);
  return (int64_t)((uint64_t)hi << 32 | lo);
}

template <class T> struct alignas(16) Vec {
  T v[16 / sizeof(T)];
};

// One row of a column: r, and (T)r, (T)(r - 1).
template <class T> struct Row {
  int r;
  T f, m1;
  __device__ __forceinline__ explicit Row(int row) : r(row), f((T)row), m1((T)(row - 1)) {}
};

// R of row r at column c: cf = (T)c, y = 1 / cf, a = R of row r, nb = R of row r - 1 at column c - 1.
// (DIAG: the row may be on the diagonal.)
template <class T, int OP, bool QUICK, bool DIAG>
__device__ __forceinline__ T radial_step(const Row<T>& row, int c, T cf, T y, T a, T nb, T x) {
  // linear_interpolation's weight (runtime/skeleton/util.cpp:564; its float literals are exact here)
  T q;
  if constexpr (QUICK) {
    q = row.f * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, cf, row.f), y, q);
  } else {
    q = row.f / cf;
  }
  const T w = q * (cf - (T)1) - row.m1;
  const T mix = a * w + nb * ((T)1 - w);  // a*w + b*(1-w)
  T base = DIAG && row.r == c ? nb : mix;
  base = row.r == 0 ? a : base;
  const T both = combine<OP>(base, x);  // not under the condition: the instruction would get a branch
  return __builtin_isfinite(x) ? both : base;
}

// The columns of a band, position by position (FULL: all of them are in it; DIAG: some row
// may be on the diagonal). va, vb: the rows'
// inputs; the owned row's results replace vb.
template <class T, int OP, int K, bool QUICK, bool FULL, bool DIAG>
__device__ __forceinline__ void columns(const Oct& O, const Row<T>& ra, const Row<T>& rb, T pa, T pb, const T (&va)[K], T (&vb)[K]) {
  // lane p: column cb + p and its reciprocal
  const T cl = (T)(O.cb + (int)(threadIdx.x & 63)), yl = (T)1 / cl;
#pragma unroll
  for (int p = 0; p < K; p++) {
    if (!FULL && (p < O.p0 || p >= O.p1)) continue;  // uniform
    const T cf = lane_read(cl, p), y = lane_read(yl, p);
    const T na = lane_prev(pa), nb = lane_prev(pb, lane_read(pa, 63));
    pa = radial_step<T, OP, QUICK, DIAG>(ra, O.cb + p, cf, y, pa, na, va[p]);
    pb = radial_step<T, OP, QUICK, DIAG>(rb, O.cb + p, cf, y, pb, nb, vb[p]);
    vb[p] = pb;
  }
}

template <class T, int OP, int K, bool QUICK>
__global__ void __launch_bounds__(NT) k_radial(const T* __restrict__ in, T* __restrict__ out, Params P) {
  static_assert(K <= OWN, "the rows before the owned ones cover the band");
  constexpr int V = 16 / sizeof(T);  // cells of a vector
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (NT / 64) + (threadIdx.x >> 6)));
  if (g >= P.first[8]) return;
  int o = 0;
  while (o < 7 && g >= P.first[o + 1]) o++;
  const Oct O = P.oct[o];
  const int r0 = (g - P.first[o] - 1) * OWN;
  const Row<T> ra(r0 + lane), rb(r0 + OWN + lane);
  const bool along_x = O.fx != 0;
  // Terms of the two rows, clamped into the octant's rows so that every address below is a
  // raster cell: all loads are issued unconditionally. Cells outside the octant are unused.
  auto term = [&](int r) {
    const int rc = r < 0 ? 0 : (r > O.L1 ? O.L1 : r);
    return along_x ? rowt(P, P.s1 + rc * O.sy) : colt(P, P.s0 + rc * O.sx);
  };
  const int64_t ta = term(ra.r), tb = term(rb.r);
  const int cfirst = O.cb + O.p0, uf = along_x ? P.s0 : P.s1, df = along_x ? O.fx : O.fy;
  const bool full = O.p0 == 0 && O.p1 == K;

  // the previous column's values (in front of the first column the neutral value stands in)
  T pa = neutral<T, OP>(), pb = pa;
  if (cfirst > 0) {
    Along q;
    q.init(P, along_x, uf + (cfirst - 1) * df, df);
    pa = out[q.off + ta];
    pb = out[q.off + tb];
  }
  // LINES: position p is at line + p * dline, a lane's rows at byte offsets da, db from there
  const int64_t ends[2] = {lane_read(ta, 0), lane_read(tb, 63)}, t0 = ends[0] < ends[1] ? ends[0] : ends[1];
  const unsigned da = (unsigned)((ta - t0) * sizeof(T)), db = (unsigned)((tb - t0) * sizeof(T));
  const int64_t line = (O.mode == LINES ? rowt(P, uf + O.cb * df) : 0) + t0, dline = (int64_t)df * P.BS0;
  const int xa = P.s0 + (O.mode == DOWN ? -(O.cb + K - 1) : O.cb);  // UP, DOWN: the band's smallest x
  T va[K], vb[K];
  if (O.mode == LINES) {
    const char* l = (const char*)(in + line);
#pragma unroll
    for (int p = 0; p < K; p++) {
      va[p] = *(const T*)(l + da);
      vb[p] = *(const T*)(l + db);
      l += dline * (int64_t)sizeof(T);
    }
  } else if (O.mode == CELLS) {
    Along q;
    q.init(P, along_x, uf + cfirst * df, df);
#pragma unroll
    for (int p = 0; p < K; p++) {
      va[p] = in[q.off + ta];
      vb[p] = in[q.off + tb];
      if (p >= O.p0 && p + 1 < O.p1) q.step();  // uniform: positions outside the band repeat its ends
    }
  } else {
    const int64_t x = colt(P, xa);
    Vec<T> a[K / V], b[K / V];
#pragma unroll
    for (int q = 0; q < K / V; q++) {
      a[q] = *(const Vec<T>*)(in + x + ta + q * V);
      b[q] = *(const Vec<T>*)(in + x + tb + q * V);
    }
    if (O.mode == UP) {
#pragma unroll
      for (int p = 0; p < K; p++) { va[p] = a[p / V].v[p % V]; vb[p] = b[p / V].v[p % V]; }
    } else {
#pragma unroll
      for (int p = 0; p < K; p++) { va[p] = a[(K - 1 - p) / V].v[(K - 1 - p) % V]; vb[p] = b[(K - 1 - p) / V].v[(K - 1 - p) % V]; }
    }
  }
  if (full && r0 + 2 * OWN - 1 < O.cb) columns<T, OP, K, QUICK, true, false>(O, ra, rb, pa, pb, va, vb);
  else if (full) columns<T, OP, K, QUICK, true, true>(O, ra, rb, pa, pb, va, vb);
  else columns<T, OP, K, QUICK, false, true>(O, ra, rb, pa, pb, va, vb);
  // the owned rows' results of the band
  if (rb.r > O.L1) return;
  const bool whole = full && r0 + 2 * OWN - 1 <= O.cb;  // uniform: no cell of the band outside the octant
  if (O.mode == LINES) {
    char* l = (char*)(out + line);
    if (whole) {
#pragma unroll
      for (int p = 0; p < K; p++) {
        *(T*)(l + db) = vb[p];
        l += dline * (int64_t)sizeof(T);
      }
    } else {
#pragma unroll
      for (int p = 0; p < K; p++) {
        if (p >= O.p0 && p < O.p1 && rb.r <= O.cb + p) *(T*)(l + db) = vb[p];
        l += dline * (int64_t)sizeof(T);
      }
    }
  } else if (O.mode == CELLS) {
    Along q;
    q.init(P, along_x, uf + cfirst * df, df);
#pragma unroll
    for (int p = 0; p < K; p++) {
      if (p < O.p0 || p >= O.p1) continue;  // uniform
      if (rb.r <= O.cb + p) out[q.off + tb] = vb[p];
      q.step();
    }
  } else {
    T* x = out + colt(P, xa) + tb;
    const bool up = O.mode == UP;
    if (whole && up) {
#pragma unroll
      for (int q = 0; q < K / V; q++) {
        Vec<T> w;
#pragma unroll
        for (int e = 0; e < V; e++) w.v[e] = vb[q * V + e];
        *(Vec<T>*)(x + q * V) = w;
      }
    } else if (whole) {
#pragma unroll
      for (int q = 0; q < K / V; q++) {
        Vec<T> w;
#pragma unroll
        for (int e = 0; e < V; e++) w.v[e] = vb[K - 1 - q * V - e];
        *(Vec<T>*)(x + q * V) = w;
      }
    } else {
#pragma unroll
      for (int p = 0; p < K; p++)
        if (p >= O.p0 && p < O.p1 && rb.r <= O.cb + p) x[up ? p : K - 1 - p] = vb[p];
    }
  }
}

static void check(hipError_t e, const char* w) {
  if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}

// Octants in the reference's order (RadialCase, runtime/Direction.hpp:68):
// NORTH_EAST, EAST_NORTH, EAST_SOUTH, SOUTH_EAST, SOUTH_WEST, WEST_SOUTH,
// WEST_NORTH, NORTH_WEST; x grows east, y grows south.
static const int kDirs[8][4] = {{0, -1, 1, 0}, {1, 0, 0, -1}, {1, 0, 0, 1}, {0, 1, 1, 0},
                                {0, 1, -1, 0}, {-1, 0, 0, 1}, {-1, 0, 0, -1}, {0, -1, -1, 0}};

static int reach(int s, int ds, int u0, int u1) {  // cells from s to the edge along (u0, u1) on its axis
  const int u = u0 ? u0 : u1;
  return u > 0 ? ds - 1 - s : s;
}

// Whether a wavefront's 2 * OWN rows along x lie within 2^32 bytes: LINES keeps their places as 32-bit
// offsets (a 64-bit address per row, cell and lane would be two more instructions each). They cross
// into another block column at most once in BS0 cells, a block's cells further on.
static bool lines_fit(int BS0, int BS1, int NB0, int dt_bytes) {
  const int rows = 2 * OWN - 1, crossed = (BS0 - 1 + rows) / BS0, most = crossed < NB0 - 1 ? crossed : NB0 - 1;
  return (uint64_t)((int64_t)most * BS0 * (BS1 - 1) + rows) * (uint64_t)dt_bytes < (1ull << 32);
}

// dt_bytes 4: float, 8: double; op: 0 sum, 1 prod, 2 max, 3 min. Returns the launch count.
int run(void* out, const void* in, int dt_bytes, int op, int BS0, int BS1, int NB0, int NB1, int DS0, int DS1, int s0,
        int s1, void* stream) {
  if (s0 < 0 || s1 < 0 || s0 >= DS0 || s1 >= DS1) throw std::runtime_error("radial: start cell outside the raster");
  if (op < 0 || op > 3) throw std::runtime_error("radial: bad reduction");
  Params P{};
  P.BS0 = BS0; P.BS1 = BS1; P.NB0 = NB0; P.NB1 = NB1; P.s0 = s0; P.s1 = s1;
  int maxL0 = 0;
  for (int o = 0; o < 8; o++) {
    Oct& O = P.oct[o];
    O.fx = kDirs[o][0]; O.fy = kDirs[o][1]; O.sx = kDirs[o][2]; O.sy = kDirs[o][3];
    O.L0 = O.fx ? reach(s0, DS0, O.fx, 0) : reach(s1, DS1, 0, O.fy);
    O.L1 = O.sx ? reach(s0, DS0, O.sx, 0) : reach(s1, DS1, 0, O.sy);
    maxL0 = O.L0 > maxL0 ? O.L0 : maxL0;
  }
  if (dt_bytes != 4 && dt_bytes != 8) throw std::runtime_error("radial: F32 or F64 rasters only");
  const int K = dt_bytes == 8 ? 32 : 64;
  // bands aligned in x or y lie in one column or row of blocks, and vectors along x are aligned
  for (int o = 0; o < 8; o++) {
    Oct& O = P.oct[o];
    O.mode = O.fx ? (BS0 % K ? CELLS : O.fx > 0 ? UP : DOWN) : (BS1 % K || !lines_fit(BS0, BS1, NB0, dt_bytes) ? CELLS : LINES);
  }
  const bool quick = dt_bytes == 4 && maxL0 <= QUICK_MAX;
  hipStream_t s = (hipStream_t)stream;
  int launches = 0;
  for (int b = 0;; b++) {
    int total = 0;
    bool any = false;
    for (int o = 0; o < 8; o++) {
      P.first[o] = total;
      Oct& O = P.oct[o];
      const int f = O.fx + O.fy, u = O.fx ? s0 : s1, ua = (u / K + f * b) * K;  // smallest x or y of an aligned band
      O.cb = O.mode == CELLS ? K * b : f > 0 ? ua - u : u - (ua + K - 1);
      O.p0 = O.cb < 0 ? -O.cb : 0;
      O.p1 = O.L0 - O.cb + 1 < K ? O.L0 - O.cb + 1 : K;
      if (O.cb > O.L0) continue;
      any = true;
      const int last = O.cb + O.p1 - 1, rmax = last < O.L1 ? last : O.L1;
      total += rmax / OWN + 1;
    }
    P.first[8] = total;
    if (!any) break;
    const unsigned grid = (unsigned)((total + NT / 64 - 1) / (NT / 64));
#define MAPX_RADIAL(T, OPV, KV, Q) \
  hipLaunchKernelGGL((k_radial<T, OPV, KV, Q>), dim3(grid), dim3(NT), 0, s, (const T*)in, (T*)out, P)
#define MAPX_RADIAL_OPS(T, KV, Q)                   \
  if (op == SUM) MAPX_RADIAL(T, SUM, KV, Q);        \
  else if (op == PROD) MAPX_RADIAL(T, PROD, KV, Q); \
  else if (op == MAX) MAPX_RADIAL(T, MAX, KV, Q);   \
  else MAPX_RADIAL(T, MIN, KV, Q)
    if (dt_bytes == 8) { MAPX_RADIAL_OPS(double, 32, false); }
    else if (quick) { MAPX_RADIAL_OPS(float, 64, true); }
    else { MAPX_RADIAL_OPS(float, 64, false); }
#undef MAPX_RADIAL_OPS
#undef MAPX_RADIAL
    check(hipGetLastError(), "k_radial launch");
    launches++;
  }
  return launches;
}

}  // namespace radial
}  // namespace mapx
