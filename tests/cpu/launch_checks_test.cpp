// Host checks of launches whose kernels rely on them. Every call here must be
// refused before anything reaches a device, so no device is needed.
#include <cstdio>
#include <cstring>
#include <functional>

#include "vx_internal.h"

using namespace vx;

static uint32_t* word(uintptr_t at) { return reinterpret_cast<uint32_t*>(at); }

// Layers of 2^3 and 2^2 values as a prover lays them out, levels from `lo` up.
static FriTailArgs tail(uint32_t lo) {
  FriTailArgs a{};
  for (auto& p : a.in) p = word(0x1000);
  a.ch = reinterpret_cast<Channel*>(word(0x2000));
  a.n_layers = 2;
  for (uint32_t li = 0; li < 2; li++) {
    FriTailLayer& T = a.layer[li];
    T.log_n = 3 - li;
    T.lo = lo;
    for (auto& p : T.out) p = word(0x3000);
    T.tw = word(0x4000);
    T.tree = word(0x5000);
    uint32_t w = 0;
    for (uint32_t l = lo; l <= T.log_n; l++) {
      T.off[l] = w;
      w += 8u << (T.log_n - l);
    }
    T.root_out = word(0x6000);
    T.alpha = word(0x7000 + 16 * li);
    T.next_alpha = li == 0 ? word(0x7010) : nullptr;
  }
  return a;
}

static bool refused(const std::function<void()>& f) {
  try {
    f();
  } catch (const Error& e) {
    std::printf("%s\n", e.what());
    return e.code == ERR_ARG;
  }
  return false;
}

int main(int argc, char** argv) {
  const char* what = argc > 1 ? argv[1] : "";
  FriTailArgs a = tail(!std::strcmp(what, "tail_level_0") ? 0 : 1);
  bool ok = false;
  if (!std::strcmp(what, "tail_level_0")) {  // the merge stores from level 1 up
    ok = refused([&] { fri_tail(a, nullptr); });
  } else if (!std::strcmp(what, "tail_other_challenge")) {  // layer 1 folds by what layer 0 draws
    a.layer[1].alpha = word(0x7020);
    ok = refused([&] { fri_tail(a, nullptr); });
  } else if (!std::strcmp(what, "tail_no_challenge")) {
    a.layer[0].next_alpha = nullptr;
    ok = refused([&] { fri_tail(a, nullptr); });
  } else if (!std::strcmp(what, "proof_destination")) {  // stored 16 bytes at a time
    ok = refused([&] { set_inputs(word(0x1000), word(0x2000), 3, 1, 1, word(0x3008), nullptr); });
  } else if (!std::strcmp(what, "inputs_pointer_slot")) {
    ok = refused([&] { set_inputs(word(0x1004), word(0x2000), 3, 1, 1, word(0x3010), nullptr); });
  }
  std::printf("%s %s\n", ok ? "PASS" : "FAIL", what);
  return ok ? 0 : 1;
}
