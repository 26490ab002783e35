// tunables.cpp -- storage for the knobs declared in tunables.h.
#include "tunables.h"

#include <cstring>

namespace llk {

// decode_max_m:      largest M (<= 64) routed to the small-M bandwidth kernel.
// decode_splits:     force its cross-workgroup k-split count (0 = cost model).
// decode_target_wgs: workgroups per round in the small-M cost model (1 per CU).
// decode_min_kb:     fewest 64-k steps per split.
// decode_group_width: force the 32-column groups per small-M workgroup (1, 2
//                    or 4; 0 = cost model, 2 or 1); a forced width runs the
//                    small-M kernel of that width.
// decode_tile:       1 = M <= 64 with K a multiple of 64 and 16-byte aligned
//                    X rows runs on the decode tile kernel (LDS-DMA ring);
//                    0 = always the small-M kernel (and no mid-M form).
// midm_max_m:        largest M (<= 256) above 64 that runs on the decode
//                    tile kernel's 128- and 256-row forms (K a multiple of
//                    64, 16-byte aligned X rows) instead of the tile
//                    kernels; 64 or less = never.  128 by default: the
//                    256-row form re-reads 32 KiB of X per 64-k step beside
//                    16 KiB of weights and loses to the tile kernels (config
//                    5 MLP at M = 200 / 255: 146 / 156 us against 140 / 143).
// tile_splits:       force the tile kernel's k-split count (0 = cost model).
// tile_wgs_per_wave: workgroups the tile kernel runs at once (1 per CU).
// tile_min_kb:       fewest 64-k steps per tile-kernel split.
// tile_tail_split:   1 = the tile kernel may run the columns of its last,
//                    partial wave as a separate k-split launch; 0 = never.
// tile_wide:         fused SwiGLU with bf16 output: 1 = the cost model may
//                    take the wide tile kernel (16 B columns per matrix, B = 7
//                    or 11) where its whole waves beat the 128-column tile;
//                    0 = never; 7 or 11 = that width whenever it applies.
// flex_tile:         1 = the cost model may take the flex tile kernel (above
//                    64 rows, and below for K < 64), and up to 64 rows the
//                    small-M kernel unsplit in place of a k split, as long as
//                    no other knob of the kernels compared has been set; 0 = neither; 222, 224 or 244 = that tile (64 x
//                    64, 64 x 128 or 128 x 128 MFMA rows), tile_splits its k
//                    splits.
// kernel_fn_rowmajor: 1 = the KernelFn entries read device weights with
//                    aligned rows straight into the kernels' row-major forms
//                    (the decode tile kernel's up to 128 rows, the tile
//                    kernel's above: SwiGLU and the accumulating matmul);
//                    0 = they pack the weights on every call.
// max_workspaces:    library-owned workspaces kept per device (one per
//                    stream, or per thread on the per-thread default
//                    stream); beyond it the least recently used idle one is
//                    freed once its last call has finished.
std::atomic<int64_t> g_knob_values[] = {
#define LLK_KNOB(name, value) {value},
    LLK_KNOBS(LLK_KNOB)
#undef LLK_KNOB
};

namespace {

constexpr const char* kNames[] = {
#define LLK_KNOB(name, value) #name,
    LLK_KNOBS(LLK_KNOB)
#undef LLK_KNOB
};

std::atomic<int64_t>* find(const char* name) {
  for (size_t i = 0; i < sizeof(kNames) / sizeof(*kNames); ++i)
    if (std::strcmp(kNames[i], name) == 0) return &g_knob_values[i];
  return nullptr;
}

}  // namespace

bool setTunable(const char* name, int64_t value) {
  std::atomic<int64_t>* const v = find(name);
  if (v) v->store(value, std::memory_order_relaxed);
  return v != nullptr;
}

bool getTunable(const char* name, int64_t* value) {
  std::atomic<int64_t>* const v = find(name);
  if (v) *value = v->load(std::memory_order_relaxed);
  return v != nullptr;
}

}  // namespace llk
