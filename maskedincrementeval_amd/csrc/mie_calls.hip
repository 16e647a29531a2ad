// Recorded call sequences (mie_run_calls): the entry points by number, and their arguments from 8-byte words.
// Host code only.  What it replaces is the host's side of every call of a step -- in Python 15-25 us each (shape checks,
// pointers, ctypes conversion), more than most kernels of a small frame take; from words a call costs its own checks and
// the launch.
#include "mie_common.h"

#include <string.h>

#include <utility>

namespace {

template <typename A> struct Word;          // one argument out of its word, and its signature letter
template <> struct Word<int> {
  static constexpr char kind = 'i';
  static int get(uint64_t v) { return (int)(int64_t)v; }
};
template <> struct Word<long long> {
  static constexpr char kind = 'l';
  static long long get(uint64_t v) { return (long long)v; }
};
template <> struct Word<float> {
  static constexpr char kind = 'f';
  static float get(uint64_t v) {
    const uint32_t b = (uint32_t)v;
    float f;
    memcpy(&f, &b, sizeof f);
    return f;
  }
};
template <> struct Word<double> {
  static constexpr char kind = 'd';
  static double get(uint64_t v) {
    double d;
    memcpy(&d, &v, sizeof d);
    return d;
  }
};
template <typename T> struct Word<T*> {
  static constexpr char kind = 'w';
  static T* get(uint64_t v) { return reinterpret_cast<T*>((uintptr_t)v); }
};
template <typename T> struct Word<const T*> {
  static constexpr char kind = 'r';
  static const T* get(uint64_t v) { return reinterpret_cast<const T*>((uintptr_t)v); }
};
template <> struct Word<const mie_tileset*> {
  static constexpr char kind = 't';
  static const mie_tileset* get(uint64_t v) { return reinterpret_cast<const mie_tileset*>((uintptr_t)v); }
};

constexpr int kMaxArgs = 40;

template <auto Fn> struct Entry;
template <typename... A, int (*Fn)(A...)> struct Entry<Fn> {
  static constexpr int n = (int)sizeof...(A) - 1;          // the stream comes last
  static_assert(n <= kMaxArgs, "argument count");
  template <size_t... I>
  static int run(const uint64_t* w, void* stream, std::index_sequence<I...>) {
    const uint64_t s = (uint64_t)(uintptr_t)stream;
    return Fn(Word<A>::get(I == (size_t)n ? s : w[I])...);
  }
  static int call(const uint64_t* w, void* stream) { return run(w, stream, std::make_index_sequence<sizeof...(A)>{}); }
  static const char* sig() {
    struct Cut {
      char s[kMaxArgs + 2] = {Word<A>::kind..., 0};
      Cut() { s[n] = 0; }
    };
    static const Cut cut;
    return cut.s;
  }
};

struct Row {
  const char* name;
  int n;
  int (*call)(const uint64_t*, void*);
  const char* (*sig)();
};
#define ROW(f) {#f, Entry<&f>::n, &Entry<&f>::call, &Entry<&f>::sig}
const Row kRows[] = {
    ROW(mie_mask_from_delta), ROW(mie_build_mask_tiles), ROW(mie_build_mask_tiles_thresholded), ROW(mie_build_mask_plan),
    ROW(mie_build_mask_plan_wgs), ROW(mie_conv_masked), ROW(mie_conv_masked_ws), ROW(mie_conv_masked_noalloc),
    ROW(mie_conv_refresh), ROW(mie_act_incr), ROW(mie_kfence_incr), ROW(mie_mul_incr), ROW(mie_add_incr),
    ROW(mie_maxpool_incr), ROW(mie_accumulate), ROW(mie_upsample2x_incr), ROW(mie_upsample2x_pair_incr),
    ROW(mie_convlstm_gates_incr), ROW(mie_convgru_gates_incr), ROW(mie_conv_gates_masked), ROW(mie_conv_gates_masked_ws),
    ROW(mie_convlstm_gates_refresh), ROW(mie_convgru_gates_refresh), ROW(mie_mul_dense), ROW(mie_scale_incr),
    ROW(mie_avgpool_incr), ROW(mie_linear_incr), ROW(mie_upconv_masked), ROW(mie_upconv_masked_ws),
    ROW(mie_upconv_pred_masked), ROW(mie_upconv2x_pred_masked), ROW(mie_tconv_masked), ROW(mie_tconv_refresh), ROW(mie_tconv2x_masked),
    ROW(mie_tconv2x_refresh), ROW(mie_upconv2x_masked), ROW(mie_upconv2x_refresh), ROW(mie_events_to_frame), ROW(mie_events_to_frame_bf16),
    ROW(mie_conv_gru_masked), ROW(mie_tconv2x_lead_masked),
};
#undef ROW
constexpr int kRowCount = (int)(sizeof(kRows) / sizeof(kRows[0]));

}  // namespace

extern "C" int mie_call_index(const char* name) {
  for (int i = 0; name != nullptr && i < kRowCount; ++i)
    if (strcmp(kRows[i].name, name) == 0) return i;
  mie_set_error("mie_call_index: no entry point %s in call sequences", name ? name : "NULL");
  return MIE_ERR_UNSUPPORTED;
}

extern "C" const char* mie_call_signature(int entry) {
  return entry >= 0 && entry < kRowCount ? kRows[entry].sig() : nullptr;
}

extern "C" int mie_run_calls(const mie_call* calls, int n_calls, const uint64_t* inputs, int n_inputs, void* stream) {
  MIE_REQUIRE(n_calls >= 0 && (calls != nullptr || n_calls == 0), MIE_ERR_INVALID_ARG, "mie_run_calls: calls is NULL");
  MIE_REQUIRE(n_inputs >= 0 && (inputs != nullptr || n_inputs == 0), MIE_ERR_INVALID_ARG, "mie_run_calls: inputs is NULL");
  for (int i = 0; i < n_calls; ++i) {
    const mie_call& c = calls[i];
    MIE_REQUIRE(c.entry >= 0 && c.entry < kRowCount && c.n_args == kRows[c.entry].n && c.args != nullptr,
                MIE_ERR_INVALID_ARG, "mie_run_calls: call %d names no entry point or has the wrong number of arguments", i);
    const uint64_t* words = c.args;
    uint64_t local[kMaxArgs];
    if (c.n_patches > 0) {
      memcpy(local, c.args, sizeof(uint64_t) * (size_t)c.n_args);
      for (int p = 0; p < c.n_patches; ++p) {
        const int slot = c.patches[2 * p], in = c.patches[2 * p + 1];
        MIE_REQUIRE(slot >= 0 && slot < c.n_args && in >= 0 && in < n_inputs, MIE_ERR_INVALID_ARG,
                    "mie_run_calls: call %d patches argument %d from input %d", i, slot, in);
        local[slot] = inputs[in];
      }
      words = local;
    }
    const int rc = kRows[c.entry].call(words, stream);
    if (rc != MIE_OK) return rc;
  }
  return MIE_OK;
}
