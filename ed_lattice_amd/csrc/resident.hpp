// Lanczos chains of small sectors, each run whole by one block.
#pragma once
#include "chains.hpp"
#include "hxv2.hpp"
#include "seeds.hpp"

namespace edl {

// One chain of a resident launch.  It starts from the seed of a ground state
// (gs set), from a given vector (src set), or goes on from the state an
// earlier launch left in q0, q1 and *sc (neither set).
struct ResChain {
  TwoPassView V;          // sector tables (ld = DimUp)
  const void* lut_up;     // coefficient tables of the chain's scalar type
  const void* lut_dw;
  const double* src;      // start vector, natural layout, fp64
  const double* gs;       // state the seed acts on
  int gs_dimup;
  SeedSpec seed;
  void* q0;               // stored vectors (natural layout), q_k in q[k & 1]; null: not kept
  void* q1;
  LzScalars* sc;
  double* alpha;          // [nmax], zeroed by the launch that starts the chain
  double* beta;           // [nmax]
  void* basis;            // [nmax][dim] q_k stored as they are made, or null
  double* bscale;         // [nmax] their norms
  double* x;              // fp64 accumulator x += ccoef_k q_k / s_k (replay), or null
  const double* ccoef;
  int nmax;
  double brk_tol;         // relative breakdown threshold on beta
};

// Whether chains on `s` can run resident (whether they do: also by size, see the
// callers): packed hop tables, no non-local
// block, at most kResMaxRows elements a thread, vector and tables within LDS.
bool res_ok(const Sector& s, size_t elem);
// Up to `steps` further Lanczos steps of every chain (device array), one
// block per chain.  All chains' sectors satisfy res_ok; max_dim, lds: the
// largest of their dimensions and of res_lds_bytes.
template <typename T>
void launch_resident(const ResChain* d_chains, int n, int64_t max_dim, size_t lds, bool one, const InterParams& I,
                     int steps, hipStream_t st);
size_t res_lds_bytes(const Sector& s, size_t elem);

}  // namespace edl
