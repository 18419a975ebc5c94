// One-launch H x v by column panels.
#pragma once
#include "chains.hpp"
#include "hxv2.hpp"

namespace edl {

// Whether panels of C columns of `elem` bytes run on this view (columns
// within LDS, up-spin table packed).
bool cols_ok(const TwoPassView& V, int C, size_t elem);
// out = H q in the view's layout, panels of cfg.one_C columns a block of
// cfg.one_threads.
template <typename T>
void launch_cols(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, const T* q, T* out,
                 const TwoPassCfg& cfg, hipStream_t st);

}  // namespace edl
