// The library's host side without a GPU: this program defines the HIP calls that an operator makes (they take
// precedence over the runtime's), allocates host memory for them and launches nothing. It prints what it is
// told to do by its arguments and, in between, each call that matters to a caller:
//   create DEGREE NX NY NZ PRECISION | device D | refuse BYTES (allocations of at least that many fail)
//   tangent (of a material without transition, bound to a temperature) | mapping
//   vmult | vmult_f32 | vmult_noalloc          prints "alloc DEVICE BYTES", "launch BLOCKS" and "rc CODE"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "../../include/mpdg_heat.h"

namespace {
int device = 0;
size_t refused = ~(size_t)0;
struct Dim3 {
  unsigned x, y, z;
};
Dim3 grid{}, block{};
size_t shared = 0;
void *stream = nullptr;
constexpr int kSuccess = 0, kOutOfMemory = 2;
}  // namespace

extern "C" {
int hipGetDevice(int *d) {
  *d = device;
  return kSuccess;
}
int hipMalloc(void **p, size_t bytes) {
  if (bytes >= refused) return kOutOfMemory;
  std::printf("alloc %d %zu\n", device, bytes);
  *p = std::malloc(bytes);
  return *p ? kSuccess : kOutOfMemory;
}
int hipFree(void *p) {
  std::free(p);
  return kSuccess;
}
int hipMemset(void *p, int v, size_t bytes) {
  std::memset(p, v, bytes);
  return kSuccess;
}
int hipGetLastError() { return kSuccess; }
int hipDeviceSynchronize() { return kSuccess; }
int hipFuncSetAttribute(const void *, int, int) { return kSuccess; }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t s, void *st) {
  grid = g;
  block = b;
  shared = s;
  stream = st;
  return kSuccess;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *s, void **st) {
  *g = grid;
  *b = block;
  *s = shared;
  *st = stream;
  return kSuccess;
}
int hipLaunchKernel(const void *, Dim3 g, Dim3, void **, size_t, void *) {
  std::printf("launch %u\n", g.x * g.y * g.z);
  return kSuccess;
}
}

int main(int argc, char **argv) {
  mpdg_heat_op *op = nullptr;
  double unused[1] = {0.0};  // vectors are never read or written
  for (int i = 1; i < argc; ++i) {
    const std::string what = argv[i];
    auto number = [&]() -> long { return ++i < argc ? std::atol(argv[i]) : 0; };
    std::printf("%s\n", what.c_str());
    if (what == "device") {
      device = (int)number();
    } else if (what == "refuse") {
      refused = (size_t)number();
    } else if (what == "create") {
      mpdg_heat_desc d{};
      d.degree = (int)number();
      for (int &n : d.n_cells) n = (int)number();
      d.precision = (int)number();
      d.extent[0] = d.extent[1] = d.extent[2] = d.rho_cp = 1.0;
      std::printf("rc %d\n", mpdg_heat_op_create(&d, &op));
    } else if (what == "tangent") {
      mpdg_heat_material m{};
      m.density[0] = m.specific_heat[0] = m.conductivity[0] = 1.0;
      const double velocity[3] = {0.0, 0.0, 0.0};
      (void)mpdg_heat_op_reset_time_increment(op, 1.0);
      int rc = mpdg_heat_op_set_tangent(op, &m, 0, velocity);
      if (rc == MPDG_OK) rc = mpdg_heat_op_bind_temperature(op, unused, unused, nullptr);
      std::printf("rc %d\n", rc);
    } else if (what == "mapping") {
      std::printf("rc %d\n", mpdg_heat_op_set_mapping(op, unused));
    } else if (what == "vmult") {
      std::printf("rc %d\n", mpdg_heat_op_vmult(op, unused, unused, nullptr));
    } else if (what == "vmult_f32") {
      float *v = reinterpret_cast<float *>(unused);
      std::printf("rc %d\n", mpdg_heat_op_vmult_f32(op, v, v, nullptr));
    } else if (what == "vmult_noalloc") {
      std::printf("rc %d\n", mpdg_heat_op_vmult_noalloc(op, unused, unused, nullptr));
    } else {
      std::fprintf(stderr, "what is %s?\n", what.c_str());
      return 1;
    }
  }
  return mpdg_heat_op_destroy(op);
}
