// One-launch H x v by column panels, and Lanczos steps of two launches on it.
#pragma once
#include "chains.hpp"
#include "hxv2.hpp"

namespace edl {

// Whether panels of C columns of `elem` bytes run on this view (columns
// within LDS, up-spin table packed).
bool cols_ok(const TwoPassView& V, int C, size_t elem);
// Blocks of a launch, the size of LzChain::part_dw of a chain on it.
int cols_grid(const TwoPassView& V, const TwoPassCfg& cfg);
// Operator mode (L = null): out = H qa in the view's layout.  Chain mode: the
// second launch of a step, see launch_chain_b.  cfg.one_C, one_threads.
template <typename T>
void launch_cols(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, T* qa, T* qb, T* out,
                 const LzChain* L, const TwoPassCfg& cfg, hipStream_t st);
// First launch of a chain step: alpha_k of the step before from the partials
// the column launch left, and its phase B (r = t - alpha_k v over t, block
// partials of |r|^2, q_k to the stored basis, replay term).  The launches pass
// the scalars on in two places, L.sc (column launch to this one) and L.sc2
// (back), and every block adds the partials up itself, in block order, so that
// a step needs no reduction launches.  After the last column launch, and before the
// host reads the chain, launch_chain_alpha completes alpha_k.
int chain_b_grid(const TwoPassView& V);
template <typename T>
void launch_chain_b(const TwoPassView& V, T* qa, T* qb, const LzChain& L, hipStream_t st);
void launch_chain_alpha(const LzChain& L, hipStream_t st);

}  // namespace edl
