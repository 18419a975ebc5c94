// One-launch H x v: a block stages C whole columns in LDS, gathers their up
// hops there and their down hops from the neighbour columns in global memory
// (consecutive rows: whole cache lines, the hop list uniform over a wave and
// held in scalar registers).  No intermediate vector.
//
// Against the two passes it saves a launch and the intermediate's round trip,
// and reads the vector from L2 once per down hop: the better form where launches
// are the cost (ring8, 4 900 states fp64: 8.2 us against 17.9 for the two; 3x4,
// 853 776 states: 18.3 against 18.9; 3x5 (7,4), 8.8e6 states fp32: 112 against 85).
#include "cols.hpp"

namespace edl {

// C columns a block, a row a thread at a time.  H16: the up spin's hops two to
// a word in table order (SpinTable::pk16), +-h from a register, a missing
// second hop reading a zero row after the last string.
template <typename T, int C, bool H16>
__global__ __launch_bounds__(1024) void k_cols(TwoPassView V, InterParams I, const T* __restrict__ lut_up,
                                               const T* __restrict__ lut_dw, const T* __restrict__ q,
                                               T* __restrict__ out) {
  typedef typename Vec<T, C>::type VT;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ T lut[H16 ? 1 : 256];
  VT* P = reinterpret_cast<VT*>(smem);
  const int dimup = V.dimup, dimdw = V.dimdw;
  const size_t ld = (size_t)V.ld;
  const int npan = (dimdw + C - 1) / C;
  const int pan = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
  if (pan < npan) {
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
      T acc[C], dw[C];
#pragma unroll
      for (int j = 0; j < C; ++j) {
        dw[j] = (T)0;
        // down hops: eight neighbour columns in flight
        for (int k0 = 0; k0 < nd[j]; k0 += 8) {
          T x[8], cf[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const uint32_t w = V.csr_dw[off[j] + min(k0 + k, nd[j] - 1)];
            x[k] = k0 + k < nd[j] ? q[(size_t)(w & 0xFFFFFFu) * ld + row] : (T)0;
            cf[k] = lut_dw[w >> 24];
          }
#pragma unroll
          for (int k = 0; k < 8; ++k) dw[j] += cf[k] * x[k];
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
        if (c0 + j < dimdw) out[(size_t)(c0 + j) * ld + row] = acc[j] + dw[j];
      }
    }
  }
}

// ---------------------------------------------------------------- host side
static size_t cols_lds(const TwoPassView& V, int C, size_t elem) { return (size_t)(V.dimup + 1) * C * elem; }
constexpr size_t kColsLds = 150 * 1024;

bool cols_ok(const TwoPassView& V, int C, size_t elem) {
  return (C == 1 || C == 2 || C == 4) && V.pk_up && V.csr_dw && cols_lds(V, C, elem) <= kColsLds;
}

template <typename T, int C>
static void launch_cols_c(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, const T* q,
                          T* out, const TwoPassCfg& cfg, hipStream_t st) {
  const size_t lds = cols_lds(V, C, sizeof(T));
  EDL_CHECK(cols_ok(V, C, sizeof(T)) && cfg.one_threads >= 64 && cfg.one_threads <= 1024 && cfg.one_threads % 64 == 0,
            "launch_cols: panel exceeds LDS or bad block size");
  const dim3 g(((V.dimdw + C - 1) / C + 7) / 8 * 8), b(cfg.one_threads);
  if (V.pk16_up && V.nv_up == 1) {
    set_lds_limit((const void*)k_cols<T, C, true>, (int)kColsLds);
    hipLaunchKernelGGL((k_cols<T, C, true>), g, b, lds, st, V, I, lut_up, lut_dw, q, out);
  } else {
    set_lds_limit((const void*)k_cols<T, C, false>, (int)kColsLds);
    hipLaunchKernelGGL((k_cols<T, C, false>), g, b, lds, st, V, I, lut_up, lut_dw, q, out);
  }
  EDL_HIP(hipGetLastError());
}

template <typename T>
void launch_cols(const TwoPassView& V, const InterParams& I, const T* lut_up, const T* lut_dw, const T* q, T* out,
                 const TwoPassCfg& cfg, hipStream_t st) {
  switch (cfg.one_C) {
    case 1: return launch_cols_c<T, 1>(V, I, lut_up, lut_dw, q, out, cfg, st);
    case 2: return launch_cols_c<T, 2>(V, I, lut_up, lut_dw, q, out, cfg, st);
    case 4: return launch_cols_c<T, 4>(V, I, lut_up, lut_dw, q, out, cfg, st);
    default: throw Error("launch_cols: unsupported panel width");
  }
}
template void launch_cols<double>(const TwoPassView&, const InterParams&, const double*, const double*, const double*,
                                  double*, const TwoPassCfg&, hipStream_t);
template void launch_cols<float>(const TwoPassView&, const InterParams&, const float*, const float*, const float*,
                                 float*, const TwoPassCfg&, hipStream_t);

}  // namespace edl
