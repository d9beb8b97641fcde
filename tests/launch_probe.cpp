// Which kernels one lambda evaluation launches, without a GPU: the HIP entry
// points that register and launch kernels are defined here, in front of the
// runtime's, and only write the names down.  Prints a line per shape:
// "<patch> <frames> <bits> <rows given> <status> <kernels>".
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>
#include <vector>

#include "../pgure-svt_amd/csrc/kernels.hpp"

static std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
static std::vector<std::string> launched;

extern "C" {
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*,
                           int*) {
  names()[host] = device;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = dim3(1);
  *b = dim3(1);
  *lds = 0;
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
  launched.push_back(names()[f]);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
}

int main() {
  const uint32_t shapes[][2] = {{2, 3}, {3, 9}, {4, 3}, {4, 15}, {6, 15}, {8, 15}};
  for (const auto& q : shapes)
    for (int bits = 32; bits <= 64; bits += 32)
      for (int rows = 0; rows < 2; ++rows) {
        pgsvt::Shape sh{};
        sh.nr = sh.nc = 32;
        sh.bs = q[0];
        sh.nw = q[1];
        sh.m = sh.bs * sh.bs;
        sh.fs = sh.nr * sh.nc;
        sh.vol = sh.fs * sh.nw;
        sh.n1 = sh.nr - sh.bs + 1;
        sh.p_all = sh.p_sel = sh.n1 * sh.n1;
        sh.fstride = pgsvt::factor_stride(sh.nw, sh.m);
        sh.fp64 = bits == 64;
        launched.clear();
        char dummy[8];
        const hipError_t e =
            pgsvt::launch_evaluation(sh, dummy, dummy, nullptr, nullptr, 1, 3, 3, 0, nullptr, dummy,
                                     rows ? dummy : nullptr, nullptr, nullptr, nullptr, nullptr);
        std::printf("%u %u %d %d %d", q[0], q[1], bits, rows, (int)e);
        for (const auto& n : launched) std::printf(" %s", n.c_str());
        std::printf("\n");
      }
  return 0;
}
