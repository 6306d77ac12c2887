// The order of loads and waits in the T64 GEMMs (gemm_n.hip, gemm_w.hip), checked on the host: every lane of every wave
// of a block runs the kernel's own source (test_dma_order.py rewrites its asm statements as calls) with loads that land
// as late as the waits allow (hip_runtime.h here), over two tiles of few and of several steps. Each MFMA's operands must
// have landed and be of its own 64-group, and so must the row scales (a NaN would reach C).
#include <stdio.h>

#include <vector>

#include "gemm_n.hip"
#include "gemm_w.hip"

namespace ifd {
alignas(16) uint8_t lds[160 * 1024];
}
using namespace ifd;

template <class Kernel, class Args>
static void run(const char* name, int MT, int units, int waves, int groups, Kernel k, Args a, std::vector<float>& C) {
  emu::units = units, emu::unread = units / 3 * 3, emu::bad = 0;  // three register sets
  gridDim.x = 1, blockIdx.x = 0;
  long nan = 0;
  for (int t = 0; t < 64 * waves; t++) {
    memset(lds, 0, sizeof(lds));
    threadIdx.x = t;
    emu::mfma = 0, emu::first = groups == 1 ? 0 : t / 128, emu::step = groups;
    k(a);
    emu::wait(0);
    for (float& v : C) nan += v != v, v = 0.f;
    if (emu::mfma != 2L * units * emu::per_unit) emu::bad++;
  }
  printf("%s MT=%d units=%d: %ld operands, %ld scales\n", name, MT, units, emu::bad, nan);
}

template <int MT, int FORM>
static void n_case() {
  for (int R = 1; R <= 9; R++) {
    const int N = 256, K = 256 * R, M = 32 * MT - 3;
    std::vector<float> C((size_t)M * N);
    GemmNArgs a{(const uint16_t*)0x1000, K, nullptr, 0, N, K, C.data(), N, M, 2, nullptr, 0, 1, nullptr, N / 64, 2, 0, 0};
    emu::act = a.A, emu::per_unit = (FORM ? 12 : 8) * MT;
    run(FORM == 2 ? "n2" : FORM ? "n1" : "n0", MT, R, 8, 4, k_gemm_n<MT, 4, FORM, 3, 2>, a, C);
  }
}

template <int MT>
static void w_case() {
  for (int G = 4; G <= 12; G++) {
    const int N = 512, K = 64 * G, M = 32 * MT - 3;
    std::vector<float> C((size_t)M * N);
    GemmWArgs a{(const uint16_t*)0x1000, K, nullptr, 0, N, K, C.data(), N, M, 2, nullptr, 1, 2, N / 64, 2, 0, 0};
    emu::act = a.A, emu::per_unit = 8 * MT;
    run("w", MT, G, 4, 1, k_gemm_w<MT, kWF32>, a, C);
  }
}

int main(int, char** argv) {
  if (argv[1][0] == 'n') {
    n_case<1, 0>(), n_case<2, 0>(), n_case<3, 0>(), n_case<4, 0>();
    n_case<1, 1>(), n_case<2, 1>(), n_case<1, 2>(), n_case<2, 2>();
  } else {
    w_case<4>(), w_case<5>(), w_case<6>(), w_case<7>(), w_case<8>();
  }
}
