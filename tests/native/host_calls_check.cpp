// Host side of the C entry points on a stand-in for the HIP runtime
// (fake_hip.hpp): what they launch, keep, free and report.
// Usage: host_calls_check CHECK
#include <cstdio>
#include <thread>

#include "../../include/top3d_hip.h"
#include "fake_hip.hpp"

#define REQUIRE(c)                                                     \
  do {                                                                 \
    if (!(c)) {                                                        \
      std::printf("FAIL line %d: %s\n", __LINE__, #c);                 \
      return 1;                                                        \
    }                                                                  \
  } while (0)

using fake::Launch;

static bool named(const Launch &l, const char *part) {
  return l.name.find(part) != std::string::npos;
}

struct Grid {
  gridContext gc{};
  gpuGrid gpu{};
  int nl;
  Grid(int nx, int ny, int nz, int nl_) : nl(nl_) {
    setupGC(&gc, nl, nx, ny, nz);
    gpu.num_targets = 1;
    gridContextToGPUGrid(&gc, &gpu, nl, 0);
  }
  ~Grid() {
    freeGPUGrid(&gpu, nl);
    freeGC(&gc, nl);
  }
  size_t nelem() const { return (gc.wrapx - 1) * (gc.wrapy - 1) * (gc.wrapz - 1); }
  size_t ndof(int l) const {
    int a, b, c, d;
    uint_fast32_t n;
    computePadding(&gc, l, &a, &b, &c, &d, &n);
    return n;
  }
};

struct Device {  // an array on the device
  double *p = nullptr;
  explicit Device(size_t n) { hipMalloc((void **)&p, sizeof(double) * n); }
  ~Device() { hipFree(p); }
};

// A call's sums of filter weights stay its own while another call on the same
// grid, with another radius, runs between its two launches.
static int filter_sums() {
  Grid g(16, 8, 8, 3);
  Device in(g.nelem()), out(g.nelem()), out2(g.nelem());
  for (const double other : {2.9, 4.5}) {
    const void *sums = nullptr, *inner = nullptr, *used = nullptr;
    bool nested = false, alive = true;
    fake::on_launch = [&](const Launch &l) {
      if (named(l, "k_filter_sums")) {
        const void *hs = *(void **)l.args[5];
        if (nested) {
          inner = hs;
          return;
        }
        sums = hs;
        nested = true;
        top3d_density_filter(&g.gc, other, 0, TOP3D_HALO_ZERO, in.p, out2.p);
        nested = false;
        alive = fake::is_device(sums);
      } else if (named(l, "k_filter_tile") && !nested) {
        used = *(void **)l.args[6];
      }
    };
    const int rc = top3d_density_filter(&g.gc, 2.5, 0, TOP3D_HALO_ZERO, in.p, out.p);
    fake::on_launch = nullptr;
    REQUIRE(rc == TOP3D_OK);
    REQUIRE(sums && inner && used == sums);
    REQUIRE(alive && inner != sums);
  }
  return 0;
}

// Without memory for the sums of weights the filter runs as the loop over the
// window, which needs none; its transpose, whose loop needs an array, reports the
// error and leaves the output alone.
static int filter_without_memory() {
  Grid g(16, 8, 8, 3);
  Device in(g.nelem()), out(g.nelem());
  std::vector<std::string> launched;
  fake::on_launch = [&](const Launch &l) { launched.push_back(l.name); };
  auto starved = [&](auto call) {
    launched.clear();
    top3d_clear_error();
    fake::fail_malloc = 1;
    const int rc = call();
    fake::fail_malloc = 0;
    return rc;
  };
  const double r = 2.5;
  REQUIRE(starved([&] {
            return top3d_density_filter(&g.gc, r, 0, TOP3D_HALO_KEEP, in.p, out.p);
          }) == TOP3D_OK);
  REQUIRE(launched.size() == 1 && launched[0].find("k_filterILi0E") != std::string::npos);
  REQUIRE(top3d_last_error() == TOP3D_OK && hipGetLastError() == 0);
  REQUIRE(starved([&] {
            applyDensityFilter(g.gc, r, in.p, out.p);
            return top3d_last_error();
          }) == TOP3D_OK && launched.size() == 1);
  REQUIRE(starved([&] {
            return top3d_density_filter(&g.gc, r, 1, TOP3D_HALO_KEEP, in.p, out.p);
          }) == TOP3D_ERR_HIP && launched.empty());
  // (the first two arrays of the gradient are the grid's: kept from this call)
  REQUIRE(top3d_compliance_backward(&g.gpu, 1.5, in.p, out.p, 1.0, out.p) == TOP3D_OK);
  REQUIRE(starved([&] {
            return top3d_compliance_backward(&g.gpu, r, in.p, out.p, 1.0, out.p);
          }) == TOP3D_ERR_HIP);
  for (const std::string &n : launched) REQUIRE(n.find("k_filter") == std::string::npos);
  // the gradient in place: with its result array, but none for the sums
  top3d_clear_error();
  applyDensityFilterGradient(g.gc, 1.5, in.p);
  REQUIRE(starved([&] {
            applyDensityFilterGradient(g.gc, r, in.p);
            return top3d_last_error();
          }) == TOP3D_ERR_HIP && launched.empty());
  fake::on_launch = nullptr;
  return 0;
}

// A change that could not be computed for want of memory does not read as none,
// and leaves no staging arrays behind.
static int change_without_memory() {
  Grid g(8, 4, 4, 3);
  const int n = (int)g.nelem();
  std::vector<double> x(n, 0.5), xnew(n, 0.5);
  const size_t before = fake::held();
  REQUIRE(compute_change(x.data(), xnew.data(), n) == 0.0f);  // (its block is kept)
  REQUIRE(fake::held() == before + 1);
  bool launched = false;
  freeGPUGrid(&g.gpu, g.nl);  // the kept block goes with the last grid
  freeGC(&g.gc, g.nl);
  const size_t none = fake::held();
  // the third allocation fails, after the staging of the two host arrays
  fake::on_launch = [&](const Launch &) { launched = true; };
  top3d_clear_error();
  fake::fail_malloc = 3;
  const float change = compute_change(x.data(), xnew.data(), n);
  fake::fail_malloc = 0;
  fake::on_launch = nullptr;
  REQUIRE(!launched && top3d_last_error() == TOP3D_ERR_HIP);
  REQUIRE(fake::held() == none);
  REQUIRE(change > 1.0f);
  return 0;
}

struct Held {
  size_t blocks = fake::held();
  int events = fake::events, streams = fake::streams;
  bool operator==(const Held &o) const {
    return blocks == o.blocks && events == o.events && streams == o.streams;
  }
};

// Grids with their solvers, coarse factors and inverses give back all that they
// allocated, also where an allocation failed half way.
static int given_back() {
  top3d_synchronize();  // (the library's stream is made once)
  const Held none;
  auto lives = [&](bool solve) {
    Grid g(16, 8, 8, 3);
    SolverDataBuffer data{};
    allocateSolverData(g.gc, 3, &data);
    if (solve && data.r) {
      Device x(g.nelem()), F(g.ndof(0)), U(g.ndof(0));
      int it;
      float res;
      solveStateMG_halo(&g.gpu, x.p, 4, 3, 1e-5, &data, &it, &res, F.p, U.p);
    }
    if (data.r) freeSolverData(&data, 3);
    CSRMatrix M{};
    allocateSubspaceMatrix(g.gc, 2, &M);
    CoarseSolverData coarse{};
    initializeCholmod(g.gc, 2, &coarse, M);
    finishCholmod(g.gc, 2, &coarse, M, 0);
    freeSubspaceMatrix(&M);
  };
  lives(true);
  REQUIRE(Held() == none);
  for (int n = 1; n < 200; n += 7) {
    fake::fail_malloc = n;
    lives(false);
    fake::fail_malloc = 0;
    if (!(Held() == none)) std::printf("allocation %d failing\n", n);
    REQUIRE(Held() == none);
  }
  {
    Device A(100 * 100);
    const Held before;
    top3d_dense_spd_inverse(A.p, 100, 20);
    REQUIRE(Held() == before);
  }
  return 0;
}

// A thread that goes from one device to another launches the level-1 sweep in
// the shape of the device it is on, as a thread that has seen no other does.
static int shapes_by_device() {
  Grid g(128, 64, 64, 3);
  Device x(g.nelem()), invD(g.ndof(1)), u(g.ndof(1)), b(g.ndof(1)), tmp(g.ndof(1));
  Dim3 grid{};
  fake::on_launch = [&](const Launch &l) {
    if (named(l, "k_level1_sweep")) grid = l.grid;
  };
  auto sweep = [&](int device, int cus) {
    fake::device = device;
    fake::cus = cus;
    smoothDampedJacobiSubspace_halo(g.gpu.target, x.p, 1, 1, 0.6, invD.p, u.p, b.p, tmp.p);
    return grid;
  };
  const Dim3 first = sweep(0, 256), here = sweep(1, 32);
  Dim3 fresh{};
  std::thread([&] { fresh = sweep(1, 32); }).join();
  fake::on_launch = nullptr;
  fake::device = 0;
  REQUIRE(first.x != fresh.x || first.y != fresh.y);
  REQUIRE(here.x == fresh.x && here.y == fresh.y);
  return 0;
}

// The events of the live sweep timing enclose launches of the plain fine sweep
// (mode 3 of k_fine_march) only, and the mean is over those.
static int sweep_timing() {
  for (const int mixed : {0, 1}) {
    Grid g(16, 8, 8, 3);
    SolverDataBuffer data{};
    allocateSolverData(g.gc, 3, &data);
    top3d_set_precision(&data, mixed ? TOP3D_MIXED : TOP3D_FP64);
    top3d_set_max_iter(&data, 1);
    Device x(g.nelem()), F(g.ndof(0)), U(g.ndof(0));
    std::vector<std::string> order;  // launches, "" for a recorded event
    std::map<void *, int> at;
    fake::on_launch = [&](const Launch &l) { order.push_back(l.name); };
    fake::on_record = [&](void *e) {
      at[e] = (int)order.size();
      order.push_back("");
    };
    int enclosed = 0;
    bool plain = true;
    fake::elapsed = [&](void *a, void *b) {  // 1 ms per launch between them
      for (int i = at[a] + 1; i < at[b]; i++) {
        enclosed++;
        plain = plain && order[i].find("k_fine_march") != std::string::npos &&
                order[i].find("Li3E") != std::string::npos;
      }
      return (float)(at[b] - at[a] - 1);
    };
    int it, count = 0;
    float res;
    double ms = 0.0;
    top3d_sweep_timing(&data, 1, nullptr, nullptr, nullptr);
    solveStateMG_halo(&g.gpu, x.p, 4, 3, 1e-5, &data, &it, &res, F.p, U.p);
    top3d_sweep_timing(&data, 0, &ms, &count, nullptr);
    fake::on_launch = nullptr;
    fake::on_record = nullptr;
    fake::elapsed = nullptr;
    freeSolverData(&data, 3);
    REQUIRE(count == 7);                       // of one V(4,4)-cycle
    REQUIRE(plain && enclosed == (mixed ? 5 : 6));  // one or two in launches with more work
    REQUIRE(ms == 1.0);
  }
  return 0;
}

int main(int argc, char **argv) {
  const std::map<std::string, int (*)()> checks = {
      {"filter_sums", filter_sums}, {"filter_without_memory", filter_without_memory},
      {"change_without_memory", change_without_memory},
      {"given_back", given_back}, {"shapes_by_device", shapes_by_device},
      {"sweep_timing", sweep_timing}};
  auto it = argc > 1 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  const int rc = it->second();
  if (rc == 0) std::printf("OK\n");
  return rc;
}
