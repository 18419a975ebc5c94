// One-launch H x v: a block stages C whole columns in LDS, gathers their up
// hops there and their down hops from the neighbour columns in global memory
// (consecutive rows: whole cache lines, the hop list uniform over a wave and
// held in scalar registers).  No intermediate vector.
//
// Against the two passes it saves a launch and the intermediate's write and
// read, and reads the vector once per down hop instead of once per panel: the
// better form while an XCD's L2 and the last-level cache serve those reads.
#include "cols.hpp"

namespace edl {

// Sum of part[0 .. n) in every thread, in block order per thread slice and a
// fixed tree (as k_lz_beta's); nw waves of a one-dimensional block.
static __device__ double cols_sum(const double* __restrict__ part, int n, double* sh, int nw) {
  const int per = (n + (int)blockDim.x - 1) / (int)blockDim.x;
  const int a = (int)threadIdx.x * per, e = min(a + per, n);
  double x = 0.0;
  for (int k = a; k < e; ++k) x += part[k];
  return block_sum_all(x, sh, nw);
}

// States of LzScalars::pad between the launches of a step: 0 no phase B
// pending (the chain's first step), 1 pending with alpha_k known, 3 pending
// with alpha_k still in the column launch's partials.
template <typename T>
__global__ __launch_bounds__(256) void k_chain_b(TwoPassView V, T* qa, T* qb, LzChain L) {
  __shared__ double sh[16];
  __shared__ double sh2[16];
  LzScalars s = *L.sc;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (s.stopped || !s.pad) {
    if (lead) *L.sc2 = s;
    return;
  }
  if (s.pad == 3) {
    s.alpha_k = cols_sum(L.part_dw, L.ndw, sh2, blockDim.x >> 6);
    s.nsteps = s.k + 1;
    s.pad = 1;
    if (lead) L.alpha[s.k] = s.alpha_k;
  }
  const bool last = s.k + 1 >= L.nmax;
  if (last) s.stopped = 1;
  if (lead) *L.sc2 = s;
  if (last && !L.x) return;
  typedef typename Row16<T>::type VT;
  constexpr int VW = 16 / (int)sizeof(T);
  T* __restrict__ qn = ((s.k + 1) & 1) ? qb : qa;
  const T* __restrict__ qk = (s.k & 1) ? qb : qa;
  const int dimup = V.dimup;
  if (L.x) {
    const double cx = L.ccoef[s.k] / s.s_cur;
    for (int col = blockIdx.x; col < V.dimdw; col += gridDim.x)
      for (int row = threadIdx.x; row < dimup; row += blockDim.x)
        L.x[(size_t)col * dimup + row] += cx * (double)qk[(size_t)col * V.ld + row];
    if (last) return;
  }
  // the padded columns as one run of 16-byte pieces (the padding rows are zero
  // in both vectors and stay so)
  const T am = (T)(s.alpha_k / s.s_cur);
  T* bst = L.basis ? static_cast<T*>(L.basis) + (size_t)s.k * V.ld * V.dimdw : nullptr;
  if (bst && lead) L.bscale[s.k] = s.s_cur;
  const size_t n = (size_t)V.ld * V.dimdw / VW, step = (size_t)gridDim.x * blockDim.x;
  double nrm = 0.0;
  constexpr int U = 2;
  for (size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += U * step) {
    VT a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * step;
      a[u] = i < n ? reinterpret_cast<const VT*>(qn)[i] : (VT)0;
      b[u] = i < n ? reinterpret_cast<const VT*>(qk)[i] : (VT)0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * step;
      if (i >= n) break;
      const VT r = a[u] - am * b[u];
      reinterpret_cast<VT*>(qn)[i] = r;
      if (bst) reinterpret_cast<VT*>(bst)[i] = b[u];
#pragma unroll
      for (int e = 0; e < VW; ++e) nrm += (double)r[e] * (double)r[e];
    }
  }
  const double v = block_sum_all(nrm, sh, blockDim.x >> 6);
  if (threadIdx.x == 0) L.part_up[blockIdx.x] = v;
}

// C columns a block, a row a thread at a time.  H16: the up spin's hops two to
// a word in table order (SpinTable::pk16), +-h from a register, a missing
// second hop reading a zero row after the last string.
template <typename T, int C, int MODE, bool H16>
__global__ __launch_bounds__(1024) void k_cols(TwoPassView V, InterParams I, const T* __restrict__ lut_up,
                                               const T* __restrict__ lut_dw, T* qa, T* qb, T* outp, LzChain L) {
  typedef typename Vec<T, C>::type VT;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double sh[16];
  __shared__ double sh2[16];
  __shared__ T lut[H16 ? 1 : 256];
  VT* P = reinterpret_cast<VT*>(smem);
  const T* __restrict__ q = qa;
  T* __restrict__ out = outp;
  LzScalars s{};
  if (MODE == 1) {
    s = *L.sc2;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (s.stopped) {
      if (lead) *L.sc = s;
      return;
    }
    if (s.pad) {
      const double b = sqrt(cols_sum(L.part_up, L.nup, sh2, blockDim.x >> 6));
      if (lead) L.beta[s.k + 1] = b;
      s.pad = 0;
      if (!(b > L.brk_tol * (fabs(s.alpha_k) + s.beta_k))) {
        s.stopped = 1;
        if (lead) *L.sc = s;
        return;
      }
      s.s_old = s.s_cur;
      s.s_cur = b;
      s.beta_k = b;
      s.k += 1;
    }
    if (lead) {
      LzScalars n = s;
      n.pad = 3;
      *L.sc = n;
    }
    q = (s.k & 1) ? qb : qa;
    out = (s.k & 1) ? qa : qb;
  }
  const int dimup = V.dimup, dimdw = V.dimdw;
  const size_t ld = (size_t)V.ld;
  const int npan = (dimdw + C - 1) / C;
  const int pan = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
  double part = 0.0;
  const double inv_s = MODE == 1 ? 1.0 / s.s_cur : 1.0;
  if (pan < npan) {
    const T ts = (T)inv_s;
    const T bo = MODE == 1 ? (T)(s.beta_k / s.s_old) : (T)0;
    const int c0 = pan * C;
    for (int r = threadIdx.x; r < dimup; r += blockDim.x) {
      VT x;
#pragma unroll
      for (int j = 0; j < C; ++j) Vec<T, C>::set(x, j, c0 + j < dimdw ? q[(size_t)(c0 + j) * ld + r] : (T)0);
      P[r] = x;
    }
    if (H16) {
      if (threadIdx.x == 0) {
        VT z;
#pragma unroll
        for (int j = 0; j < C; ++j) Vec<T, C>::set(z, j, (T)0);
        P[dimup] = z;
      }
    } else {
      for (int k = threadIdx.x; k < 256; k += blockDim.x) lut[k] = lut_up[k];
    }
    uint32_t sd[C];
    double dgd[C];
    int off[C], nd[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int c = c0 + j < dimdw ? c0 + j : c0;
      sd[j] = (uint32_t)V.map_dw[c];
      dgd[j] = V.dg_dw[c];
      off[j] = V.off_dw[c];
      nd[j] = c0 + j < dimdw ? V.off_dw[c + 1] - off[j] : 0;
    }
    const bool one_orb = I.norb == 1 && I.npairs == 0;
    const double u0 = I.U[0];
    const T l0 = lut_up[0];
    __syncthreads();
    for (int r0 = 0; r0 < dimup; r0 += blockDim.x) {
      const int row = r0 + (int)threadIdx.x;
      if (row >= dimup) continue;
      T acc[C], dw[C], o0[C];
#pragma unroll
      for (int j = 0; j < C; ++j) {
        o0[j] = (MODE == 1 && c0 + j < dimdw) ? out[(size_t)(c0 + j) * ld + row] : (T)0;
        dw[j] = (T)0;
        // down hops: eight neighbour columns in flight
        for (int k0 = 0; k0 < nd[j]; k0 += 8) {
          uint32_t w[8];
          T x[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) w[k] = V.csr_dw[off[j] + min(k0 + k, nd[j] - 1)];
#pragma unroll
          for (int k = 0; k < 8; ++k) x[k] = k0 + k < nd[j] ? q[(size_t)(w[k] & 0xFFFFFFu) * ld + row] : (T)0;
#pragma unroll
          for (int k = 0; k < 8; ++k) dw[j] += lut_dw[w[k] >> 24] * x[k];
        }
      }
      const uint32_t su = (uint32_t)V.map_up[row];
      const double dgu = V.dg_up[row];
      const VT self = P[row];
#pragma unroll
      for (int j = 0; j < C; ++j) {
        const double u = one_orb ? u0 * (double)__popc(su & sd[j] & I.orb_mask[0]) : inter2(I, su, sd[j]);
        acc[j] = (T)(dgu + dgd[j] + u) * Vec<T, C>::get(self, j);
      }
      if (H16) {
        const int nw = (V.cnt_up[row] + 1) >> 1;
        const uint32_t zpad = (uint32_t)dimup | ((uint32_t)dimup << 16);
        for (int k0 = 0; k0 < nw; k0 += 4) {
          uint32_t w[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) w[k] = k0 + k < nw ? V.pk16_up[(size_t)(k0 + k) * dimup + row] : zpad;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const T cl = flip_sign(l0, (w[k] << 16) & 0x80000000u), ch = flip_sign(l0, w[k] & 0x80000000u);
            const VT xl = P[w[k] & 0x7FFFu], xh = P[(w[k] >> 16) & 0x7FFFu];
#pragma unroll
            for (int j = 0; j < C; ++j) acc[j] += cl * Vec<T, C>::get(xl, j);
#pragma unroll
            for (int j = 0; j < C; ++j) acc[j] += ch * Vec<T, C>::get(xh, j);
          }
        }
      } else {
        const int nu = V.cnt_up[row];
        for (int k0 = 0; k0 < nu; k0 += 8) {
          uint32_t w[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) w[k] = k0 + k < nu ? V.pk_up[(size_t)(k0 + k) * dimup + row] : 255u << 24;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const T cf = lut[w[k] >> 24];
            const VT x = P[w[k] & 0xFFFFFFu];
#pragma unroll
            for (int j = 0; j < C; ++j) acc[j] += cf * Vec<T, C>::get(x, j);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < C; ++j) {
        if (c0 + j >= dimdw) continue;
        T t = acc[j] + dw[j];
        if (MODE == 1) {
          t = t * ts - bo * o0[j];
          part += (double)t * (double)Vec<T, C>::get(self, j);
        }
        out[(size_t)(c0 + j) * ld + row] = t;
      }
    }
  }
  if (MODE == 1) {
    const double v = block_sum_all(part * inv_s, sh, blockDim.x >> 6);
    if (threadIdx.x == 0) L.part_dw[blockIdx.x] = v;
  }
}

// ---------------------------------------------------------------- host side
static size_t cols_lds(const TwoPassView& V, int C, size_t elem) { return (size_t)(V.dimup + 1) * C * elem; }
constexpr size_t kColsLds = 150 * 1024;

bool cols_ok(const TwoPassView& V, int C, size_t elem) {
  return (C == 1 || C == 2 || C == 4) && V.pk_up && V.csr_dw && cols_lds(V, C, elem) <= kColsLds;
}

int cols_grid(const TwoPassView& V, const TwoPassCfg& cfg) {
  const int npan = (V.dimdw + cfg.one_C - 1) / cfg.one_C;
  return (npan + 7) / 8 * 8;
}

template <typename T, int C, int MODE>
static void launch_cols_c(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, T* qa, T* qb,
                          T* out, const LzChain& L, const TwoPassCfg& cfg, hipStream_t st) {
  const size_t lds = cols_lds(V, C, sizeof(T));
  EDL_CHECK(cols_ok(V, C, sizeof(T)) && cfg.one_threads >= 64 && cfg.one_threads <= 1024 && cfg.one_threads % 64 == 0,
            "launch_cols: panel exceeds LDS or bad block size");
  const dim3 g(cols_grid(V, cfg)), b(cfg.one_threads);
  if (V.pk16_up && V.nv_up == 1) {
    set_lds_limit((const void*)k_cols<T, C, MODE, true>, (int)kColsLds);
    hipLaunchKernelGGL((k_cols<T, C, MODE, true>), g, b, lds, st, V, I, lut_up, lut_dw, qa, qb, out, L);
  } else {
    set_lds_limit((const void*)k_cols<T, C, MODE, false>, (int)kColsLds);
    hipLaunchKernelGGL((k_cols<T, C, MODE, false>), g, b, lds, st, V, I, lut_up, lut_dw, qa, qb, out, L);
  }
  EDL_HIP(hipGetLastError());
}

template <typename T>
void launch_cols(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, T* qa, T* qb, T* out,
                 const LzChain* L, const TwoPassCfg& cfg, hipStream_t st) {
  const LzChain A = L ? *L : LzChain{};
  switch (cfg.one_C) {
    case 1:
      return L ? launch_cols_c<T, 1, 1>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st)
               : launch_cols_c<T, 1, 0>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st);
    case 2:
      return L ? launch_cols_c<T, 2, 1>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st)
               : launch_cols_c<T, 2, 0>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st);
    case 4:
      return L ? launch_cols_c<T, 4, 1>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st)
               : launch_cols_c<T, 4, 0>(V, I, lut_up, lut_dw, qa, qb, out, A, cfg, st);
    default: throw Error("launch_cols: unsupported panel width");
  }
}
template void launch_cols<double>(const TwoPassView&, const InterParams&, const double*, const double*, double*,
                                  double*, double*, const LzChain*, const TwoPassCfg&, hipStream_t);
template void launch_cols<float>(const TwoPassView&, const InterParams&, const float*, const float*, float*, float*,
                                 float*, const LzChain*, const TwoPassCfg&, hipStream_t);

// Four pieces of 16 bytes a thread at least, at most four blocks a CU.
int chain_b_grid(const TwoPassView& V) {
  const size_t pieces = (size_t)V.ld * V.dimdw / 4;
  return (int)std::max<size_t>(1, std::min<size_t>(1024, pieces / (256 * 4)));
}
template <typename T>
void launch_chain_b(const TwoPassView& V, T* qa, T* qb, const LzChain& L, hipStream_t st) {
  EDL_CHECK(V.ld % 32 == 0 && L.sc2 && L.nup == chain_b_grid(V), "launch_chain_b: padded layout and its own partials");
  hipLaunchKernelGGL(k_chain_b<T>, dim3(chain_b_grid(V)), dim3(256), 0, st, V, qa, qb, L);
  EDL_HIP(hipGetLastError());
}
template void launch_chain_b<double>(const TwoPassView&, double*, double*, const LzChain&, hipStream_t);
template void launch_chain_b<float>(const TwoPassView&, float*, float*, const LzChain&, hipStream_t);
void launch_chain_alpha(const LzChain& L, hipStream_t st) {
  hipLaunchKernelGGL(k_lz_alpha, dim3(1), dim3(256), 0, st, L, L.ndw);
  EDL_HIP(hipGetLastError());
}

}  // namespace edl
