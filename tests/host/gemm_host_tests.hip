// Host-side checks of the projection launchers (gemm.hpp): decisions and refusals that are made
// before any launch, so they need no GPU. Operands are placeholders: the program refuses to run
// where a device is visible. Usage: <program> <case>; prints PASS or the reason.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "gemm.hpp"

using namespace hllm_rocm;

namespace {

constexpr int kCus = 256;

GemmArgs projection(int rows, int n, uint64_t k, int epilogue, bool deferred) {
  GemmArgs a{};
  a.M = rows;
  a.N = n;
  a.Kp = pad32(k);
  a.w_rows_padded = (uint64_t)(n + 255) / 256 * 256;
  a.x_rows_padded = gemm_padded_rows((uint64_t)rows);
  a.workspace_floats = 32ull << 20;
  a.epilogue = epilogue;
  a.defer_reduce = deferred ? 1 : 0;
  return a;
}

// The message of the failure that `call` raises before (or instead of) its launch.
template <typename F>
std::string failure(F&& call) {
  try {
    call();
  } catch (const Failure& e) {
    return e.what();
  }
  return "";
}

// A split residual projection without a consumer for its partials is refused by every launcher
// (the reduce kernel stores its sums, it does not add them to the residual stream).
bool split_residual_is_refused() {
  const GemmArgs a = projection(96, 1024, 4096, kEpiResidual, false);
  for (int config : {0, 9, 12, 15, 16, 18}) {
    const std::string message = failure([&] { launch_gemm_config(nullptr, a, kF16, a.M, kCus, config, 4); });
    if (message.find("splits K only for a consumer") == std::string::npos) {
      std::printf("config %d: '%s'\n", config, message.c_str());
      return false;
    }
  }
  return true;
}

// q/k/v and gate+up of one row fold their RMSNorm.
bool folds(bool expect_qkv, bool expect_gate_up) {
  const bool qkv = gemm_folds_norm(projection(1, 4096, 1024, kEpiStore, true), kF16, 1, 1024, kCus);
  const bool gate_up = gemm_folds_norm(projection(1, 6144, 1024, kEpiSwiglu, false), kF16, 1, 1024, kCus);
  if (qkv != expect_qkv || gate_up != expect_gate_up) std::printf("q/k/v folds: %d, gate+up: %d\n", qkv, gate_up);
  return qkv == expect_qkv && gate_up == expect_gate_up;
}
bool norms_fold() { return folds(true, true); }
// Under a decode launch shape other than the folded kernel's (set in the environment by the caller)
// q/k/v keeps its separate norm.
bool another_decode_shape_keeps_the_norm() { return folds(false, true); }

// A pass decides once whether its norms fold; a configuration forced by another thread before the
// launch does not fail it. (Without a GPU the launch itself fails, with the runtime's message.)
bool forced_configuration_keeps_the_decision() {
  const float row = 0.0f;
  for (GemmArgs a : {projection(1, 4096, 1024, kEpiStore, true), projection(1, 6144, 1024, kEpiSwiglu, false)}) {
    if (!gemm_folds_norm(a, kF16, 1, 1024, kCus)) return false;
    a.norm.h = &row;
    a.norm.hidden = 1024;
    set_forced_gemm_config(12);
    const std::string message = failure([&] { launch_gemm(nullptr, a, kF16, 1, kCus); });
    set_forced_gemm_config(-1);
    if (message.find("cannot fold") != std::string::npos) {
      std::printf("'%s'\n", message.c_str());
      return false;
    }
  }
  return true;
}

struct Case {
  const char* name;
  bool (*run)();
};
const Case kCases[] = {{"split_residual_is_refused", split_residual_is_refused},
                       {"norms_fold", norms_fold},
                       {"another_decode_shape_keeps_the_norm", another_decode_shape_keeps_the_norm},
                       {"forced_configuration_keeps_the_decision", forced_configuration_keeps_the_decision}};

}  // namespace

int main(int argc, char** argv) {
  int devices = 0;
  if (hipGetDeviceCount(&devices) == hipSuccess && devices > 0) {
    std::printf("%d devices visible: run with HIP_VISIBLE_DEVICES=-1\n", devices);
    return 3;
  }
  for (const Case& c : kCases) {
    if (argc > 1 && std::strcmp(argv[1], c.name) != 0) continue;
    const bool ok = c.run();
    std::printf("%s %s\n", ok ? "PASS" : "FAIL", c.name);
    return ok ? 0 : 1;
  }
  return 2;
}
