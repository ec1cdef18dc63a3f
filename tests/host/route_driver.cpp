// Which kernels the runtime compiles and launches, and what memory it takes for them, on the
// device double (dev_double.cpp, compiled into this file behind hooks on its compilation, launch
// and allocation entries) through the C ABI. One scenario per run: route_driver NAME.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "dev.hpp"

#define function function_double
#define launch launch_double
#define malloc_device malloc_device_double
#define spread spread_double
#include "dev_double.cpp"
#undef spread
#undef malloc_device
#undef function
#undef launch

#include "../../include/mapx.h"

namespace {
struct Launched {
  std::string name;
  unsigned grid, grid_y;
};
std::vector<std::string> compiled;  // kernels asked for, in order
std::map<std::string, std::string> sources;
std::vector<Launched> launched;
size_t largest = 0;  // device allocation
std::function<void(const Launched&, void**, const size_t*, int)> on_launch;
}  // namespace

namespace mapx {
namespace dev {
void* malloc_device(size_t bytes) {
  largest = std::max(largest, bytes);
  return malloc_device_double(bytes);
}
Function function(const std::string& source, const std::string& name) {
  compiled.push_back(name);
  sources[name] = source;
  return function_double(source, name);
}
void launch(const Function& f, unsigned grid, unsigned block, void** params, const size_t* sizes, int n, unsigned grid_y) {
  launched.push_back({f.name, grid, grid_y});
  if (on_launch) on_launch(launched.back(), params, sizes, n);
  launch_double(f, grid, block, params, sizes, n, grid_y);
}
}  // namespace dev
namespace spread {
// cell words and finished bits, a notification word and a queue entry per 64x64 tile; counters
size_t needs(int w, int h) { return (size_t)((w + 63) / 64) * ((h + 63) / 64) * (8192 + 512 + 8) + 64 * 256 + 64 * 4; }
int run(void*, const void*, const void*, void* scratch, int, int, int, int, int, int DS0, int DS1, void*) {
  const std::vector<char> z(needs(DS0, DS1));
  dev::h2d(scratch, z.data(), z.size());
  return 3;
}
}  // namespace spread
}  // namespace mapx

namespace {

enum { F32 = 1, U8 = 4, S32 = 10, ROWBLK = 3, DEV_GPU = 4, SUM = 1, GT = 9 };

[[noreturn]] void fail(const std::string& what) {
  std::fprintf(stderr, "route driver: %s (%s)\n", what.c_str(), ma_lastError());
  std::exit(2);
}
void expect(bool ok, const std::string& what) {
  if (!ok) fail(what);
}
bool ends(const std::string& s, const std::string& tail) {
  return s.size() >= tail.size() && s.compare(s.size() - tail.size(), tail.size(), tail) == 0;
}
bool has(const std::string& s, const std::string& part) { return s.find(part) != std::string::npos; }
int kernels(const std::vector<std::string>& v, const std::string& part) {
  int n = 0;
  for (auto& s : v) n += has(s, part);
  return n;
}
int launches(const std::string& part) {
  int n = 0;
  for (auto& l : launched) n += has(l.name, part);
  return n;
}

// A held node, as a program holds one.
struct R {
  ma_node_t* n = nullptr;
  R() {}
  explicit R(ma_node_t* p) : n(p) {
    expect(n != nullptr, "factory");
    ma_increaseRef(n);
  }
  R(const R& o) : n(o.n) { if (n) ma_increaseRef(n); }
  R& operator=(const R& o) {
    if (o.n) ma_increaseRef(o.n);
    if (n) ma_decreaseRef(n);
    n = o.n;
    return *this;
  }
  ~R() { if (n) ma_decreaseRef(n); }
};
ma_dim2_t dim(int a, int b) { ma_dim2_t d; d.arr[0] = a; d.arr[1] = b; d.n = 2; return d; }
ma_dim2_t none() { ma_dim2_t d; d.arr[0] = 0; d.arr[1] = 0; d.n = 0; return d; }
ma_variant_t s32(int v) { ma_variant_t x; std::memset(&x, 0, sizeof x); x.u.s32 = v; x.dtype = S32; return x; }
R input(int w, int h, int bs, int dt, int size) {
  const size_t n = (size_t)((w + bs - 1) / bs) * ((h + bs - 1) / bs) * bs * bs * size;
  std::vector<char> a(n, 0);
  return R(ma_input(a.data(), n, dim(w, h), dt, dim(bs, bs)));
}
R conv(const R& a, const std::vector<int>& w) {
  std::vector<ma_variant_t> v;
  for (int x : w) v.push_back(s32(x));
  return R(ma_convolution(a.n, v.data(), (int)v.size(), dim(3, 3)));
}
// n generations of a 0/1 rule: more than `over` of the nine cells
R rule(R s, int n, int over = 4, int weight = 1) {
  for (int g = 0; g < n; g++) {
    R k(ma_constant(s32(over), none(), S32, ROWBLK, none()));
    R many(ma_binary(conv(s, std::vector<int>(9, weight)).n, k.n, GT));
    s = R(ma_cast(many.n, U8));
  }
  return s;
}
void eval(const std::vector<R>& v) {
  std::vector<ma_node_t*> p;
  for (const R& r : v) p.push_back(r.n);
  ma_eval(p.data(), (int)p.size());
  if (std::strlen(ma_lastError())) fail("eval");
}

// The module of a chain of 0/1 rules is compiled when a chain runs, for the shape it runs with.
void scenario_compile() {
  eval({rule(input(300, 200, 64, U8, 1), 3)});  // too short to pay
  expect(kernels(compiled, "bit_") == 0, "kernels compiled for a chain that does not pay");
  expect(launches("_pack") == 0, "a chain that does not pay ran");
  ma_setOption("form", 0);
  eval({rule(input(300, 200, 64, U8, 1), 40)});
  ma_setOption("form", 1);
  ma_setOption("tile_tx", 256); ma_setOption("tile_ty", 16); ma_setOption("tile_vx", 4);
  eval({rule(input(300, 200, 64, U8, 1), 40)});
  ma_setOption("tile_tx", 0); ma_setOption("tile_ty", 0); ma_setOption("tile_vx", 0);
  expect(kernels(compiled, "bit_") == 0, "kernels compiled for chains that run by groups");
  eval({rule(input(300, 200, 64, U8, 1), 40, 4, 2)});
  expect(kernels(compiled, "bit_") == 0, "kernels compiled for groups that are no bit rule");
  eval({rule(input(300, 200, 64, U8, 1), 40)});
  expect(launches("_pack") == 1 && launches("_step") == 5 && launches("_unpack") == 1, "a chain of 40 generations");
  expect(kernels(compiled, "_step") == 1, "more than one shape compiled");
  const size_t n = compiled.size();
  eval({rule(input(310, 190, 64, U8, 1), 40)});  // the same rule and shape on another raster
  expect(compiled.size() == n && launches("_pack") == 2, "compiled again for another raster");
  eval({rule(input(4000, 4000, 512, U8, 1), 24)});
  expect(kernels(compiled, "_step") == 2 && launches("_pack") == 3, "the shape of a large raster");
  for (auto& s : sources)
    if (has(s.first, "_step")) {
      size_t steps = 0;
      for (size_t p = 0; (p = s.second.find("mx::bit_step<", p)) != std::string::npos; p++) steps++;
      expect(steps == 1, "a module holds more than one step kernel");
    }
}

void serve(const std::vector<R>& v) {
  std::vector<ma_node_t*> p;
  for (const R& r : v) p.push_back(r.n);
  if (ma_serveSubmit(p.data(), (int)p.size()) < 0) fail("serveSubmit");
  for (int i = 0; i < 1000; i++) {
    if (ma_serveStep(0) < 0) fail("serveStep");
    long long id;
    double a, b, c;
    if (ma_serveTake(&id, &a, &b, &c, 1) == 1) return;
  }
  fail("a request that does not complete");
}

// A plan made for a request of the server has its chains when it is evaluated later.
void scenario_served_plan() {
  R s = rule(input(300, 200, 64, U8, 1), 40);
  if (ma_serveOpen(64LL << 20, 8) != 0) fail("serveOpen");
  serve({s});
  if (ma_serveClose() != 0) fail("serveClose");
  expect(launches("_pack") == 0, "the served form runs by groups");
  ma_release(s.n);
  eval({s});
  expect(launches("_pack") == 1 && launches("_step") == 5, "the plan of a served request has no chain");
}

// Per-zone statistics: the partial records of chunks (24 bytes a zone) stay below what the cells take.
R statistics(int w, int h, int nz, bool windows) {
  R a = input(w, h, 256, F32, 4), z = input(w, h, 256, S32, 4);
  eval({a, z});
  return R(ma_zonalStats(windows ? conv(a, {1, 2, 1, 2, 4, 2, 1, 2, 1}).n : a.n, z.n, nz));
}
void scenario_zone_records() {
  ma_setOption("focal_zonal", 1);
  int chunks = 0;
  on_launch = [&](const Launched& l, void** params, const size_t*, int n) {
    if (n == 8 && has(l.name, "krn_") && !ends(l.name, "_fin")) chunks = *(int*)params[5];
  };
  struct { int w, h, nz, windows, least, most; } one[] = {
      {4096, 4096, 16, 1, 2048, 2048}, {4096, 4096, 3000, 1, 256, 256}, {2048, 2048, 3000, 1, 256, 256},
      {2048, 2048, 256, 1, 1024, 1024}, {4096, 4096, 256, 0, 512, 512}, {512, 512, 3000, 0, 64, 64}, {100, 60, 3000, 1, 1, 15}};
  for (auto& c : one) {
    eval({statistics(c.w, c.h, c.nz, c.windows != 0)});
    expect(chunks >= c.least && chunks <= c.most, std::to_string(chunks) + " chunks of " + std::to_string(c.w) + " x " +
           std::to_string(c.h) + " cells, " + std::to_string(c.nz) + " zones");
  }
  // a batch whose records are more than 512 MB goes in several launches
  largest = 0;
  launched.clear();
  std::vector<R> v;
  for (int i = 0; i < 160; i++) v.push_back(statistics(512 - i % 16, 512 - i / 16, 3000, false));
  eval(v);
  expect(largest <= (size_t)512 << 20, "one allocation of " + std::to_string(largest >> 20) + " MB");
  expect((int)launched.size() <= 2 * 2 * 3, "the batch in too many launches");
  on_launch = nullptr;
}
// Where the device is too small for these records, coarser chunks are taken.
void scenario_zone_records_small_device() {
  ma_setOption("focal_zonal", 1);
  setenv("MAPX_DOUBLE_HBM", std::to_string(20 << 20).c_str(), 1);
  eval({statistics(1024, 1024, 3000, true)});
  std::vector<R> v;
  for (int i = 0; i < 6; i++) v.push_back(statistics(256 - i, 256, 3000, false));
  setenv("MAPX_DOUBLE_HBM", std::to_string(16 << 20).c_str(), 1);
  eval(v);
  unsetenv("MAPX_DOUBLE_HBM");
}

// A served flow accumulation is admitted with the memory it takes: its raster and the scan's scratch.
void scenario_served_flow() {
  for (auto& c : std::vector<std::pair<int, int>>{{40, 30}, {700, 500}}) {
    const int w = c.first, h = c.second, bs = 32;
    R rain = input(w, h, bs, F32, 4), dir = input(w, h, bs, U8, 1);
    eval({rain, dir});
    if (ma_serveOpen(64LL << 20, 8) != 0) fail("serveOpen");
    R acc(ma_spreadScan(rain.n, dir.n, SUM));
    serve({acc});
    const char* p = std::strstr(ma_serveStats(), "\"peak_inflight_bytes\": ");
    expect(p != nullptr, "serveStats");
    const size_t got = std::strtoull(p + 23, nullptr, 10);
    const size_t need = (size_t)((w + bs - 1) / bs) * ((h + bs - 1) / bs) * bs * bs * 4 + mapx::spread::needs(w, h);
    expect(got == need, "admitted with " + std::to_string(got) + " bytes, takes " + std::to_string(need));
    if (ma_serveClose() != 0) fail("serveClose");
  }
}

// Rasters that hold more than 0 and 1: the pack kernels of `bad` say so.
void report(const std::vector<bool>& bad) {
  auto n = std::make_shared<size_t>(0);
  launched.clear();
  on_launch = [=](const Launched& l, void** params, const size_t*, int) {
    if (!ends(l.name, "_pack")) return;
    if (*n < bad.size() && bad[*n]) **(unsigned**)params[3] = 1;  // its word in pinned memory
    ++*n;
  };
}
void scenario_no_bits() {
  R in = input(300, 200, 64, U8, 1), s = rule(in, 40);
  auto groups = [] { return (int)launched.size() - launches("bit_"); };
  report({true});
  eval({s});
  expect(launches("_pack") == 2 && groups() == 1, "the generations after the first one are a chain");
  ma_release(s.n);
  report({});
  eval({s});
  expect(launches("_pack") == 1 && groups() == 1, "the second evaluation looks at the same raster again");
  R t = rule(in, 41, 3);
  report({true, true, true});
  eval({t});
  expect(launches("_pack") == 2 && groups() == 41, "rasters that are never 0/1 run by groups");
  ma_release(t.n);
  report({});
  eval({t});
  expect(launches("_pack") == 0 && groups() == 41, "rasters that are never 0/1 are tried again");
  on_launch = nullptr;
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> all = {{"compile", scenario_compile}, {"served plan", scenario_served_plan}, {"no bits", scenario_no_bits},
                                                      {"served flow", scenario_served_flow},
                                                      {"zone records", scenario_zone_records},
                                                      {"zone records, small device", scenario_zone_records_small_device}};
  if (argc != 2 || !all.count(argv[1])) return 3;
  ma_setupDevices("", DEV_GPU, "");
  all.at(argv[1])();
  std::printf("route driver: ok\n");
  return 0;
}
