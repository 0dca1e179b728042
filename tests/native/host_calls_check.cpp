// Host side of the C entry points on a stand-in for the HIP runtime
// (fake_hip.hpp): what they launch, keep, free and report.
// Usage: host_calls_check CHECK
#include <cstdio>

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

int main(int argc, char **argv) {
  const std::map<std::string, int (*)()> checks = {{"filter_sums", filter_sums}};
  auto it = argc > 1 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  const int rc = it->second();
  if (rc == 0) std::printf("OK\n");
  return rc;
}
