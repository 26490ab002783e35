// tunables.h -- named integer knobs of the gfx950 dispatch heuristics
// (decode/prefill crossover, split-K factors).  Defaults are the values
// measured best on MI355X; llk_set_tunable() overrides them at run time.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdint>

namespace llk {

// The knobs and their defaults (described in tunables.cpp).  A launch plan reads
// 10 to 30 of them, so they are read by index: by name they were most of a
// plan's time (SwiGLU 300 x 1000 x 1100 1.8 us, now 0.7).
#define LLK_KNOBS(X) \
  X(decode_max_m, 64) \
  X(decode_splits, 0) \
  X(decode_target_wgs, 256) \
  X(decode_min_kb, 2) \
  X(decode_group_width, 0) \
  X(decode_tile, 1) \
  X(midm_max_m, 128) \
  X(tile_splits, 0) \
  X(tile_wgs_per_wave, 256) \
  X(tile_min_kb, 4) \
  X(tile_tail_split, 1) \
  X(tile_wide, 1) \
  X(flex_tile, 1) \
  X(kernel_fn_rowmajor, 1) \
  X(max_workspaces, 16)

enum class Knob : int {
#define LLK_KNOB(name, value) name,
  LLK_KNOBS(LLK_KNOB)
#undef LLK_KNOB
};

extern std::atomic<int64_t> g_knob_values[];

// The current value of a knob.
inline int64_t tunable(Knob k) {
  return g_knob_values[(int)k].load(std::memory_order_relaxed);
}
// Sets a knob; returns false for an unknown name.
bool setTunable(const char* name, int64_t value);
// Reads a knob into *value; returns false for an unknown name.
bool getTunable(const char* name, int64_t* value);

}  // namespace llk
