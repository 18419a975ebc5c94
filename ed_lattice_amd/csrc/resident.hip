// Lanczos chains of small sectors, each run whole by one block: the vector
// q_k in LDS, q_{k-1} and t = H q_k - ... in registers, the hop tables in LDS,
// every reduction inside the block.  A step is two barriers and no launch.
//
// The launches of a step (up, beta, down, alpha; two passes over global
// memory) cost such a sector their latency: 35 us a step on the 8-ring at
// half filling (4 900 states), 51 us for 16 chains of its N+-1 sectors.
//
// What bounds it: one CU's LDS (a hop is a 4-byte table word and an element)
// and VALU; the chip is filled only by as many chains as CUs.  Position, diagonal
// and second vector of an element stay in registers: with 8 elements a thread and
// more in fp64, 12 in fp32, some of them spill (6.1 us a step at 4 900 states, 32
// at 15 876), and the callers take the form up to a timed number of states.
#include <algorithm>

#include "resident.hpp"

namespace edl {

constexpr int kResMaxRows = 16;  // elements per thread at 1024 threads

// Sum over a row of 16 lanes, in every lane of the row (DPP moves, a fixed tree).
template <int CTRL>
static __device__ __forceinline__ double dpp_add(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const int l2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xF, 0xF, true);
  const int h2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xF, 0xF, true);
  return v + __hiloint2double(h2, l2);
}
static __device__ __forceinline__ double row_sum(double v) {
  v = dpp_add<0xB1>(v);   // quad_perm 1,0,3,2
  v = dpp_add<0x4E>(v);   // quad_perm 2,3,0,1
  v = dpp_add<0x141>(v);  // row_half_mirror
  return dpp_add<0x140>(v);  // row_mirror
}
static __device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the block in every thread; one barrier.  `sh` has 16 slots of a
// buffer that alternates between calls, so that a wave may write the next
// call's slots while others still read this one's.
static __device__ __forceinline__ double block_sum_all(double v, double* sh, int nw) {
  v = row_sum(v);
  v = (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
  const int lane = threadIdx.x & 63;
  if (lane == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const int r = lane & 15;
  return row_sum(r < nw ? sh[r] : 0.0);
}

// The coefficient of a one-magnitude hop word: bits 30 and 31 are the top bits
// of +-2.0 (0 for a padding word), in fp32 and, as the high word, in fp64.
static __device__ __forceinline__ float word_coef(uint32_t w, float) { return __uint_as_float(w & 0xC0000000u); }
static __device__ __forceinline__ double word_coef(uint32_t w, double) { return __hiloint2double((int)(w & 0xC0000000u), 0); }

// One element of a seed (SeedSpec) at target (jup, jdw).
static __device__ __forceinline__ double res_seed(const ResChain& C, uint32_t tu, uint32_t td, int jup, int jdw) {
  const SeedTerm a{C.seed.op, C.seed.ispin, C.seed.io - 1};
  double v = seed_term(a, C.gs, C.gs_dimup, tu, td, jup, jdw);
  if (C.seed.jo > 0) {
    const SeedTerm b{C.seed.op, C.seed.ispin, C.seed.jo - 1};
    v += seed_term(b, C.gs, C.gs_dimup, tu, td, jup, jdw);
  }
  return v;
}

// EPT elements a thread (e = thread + i * threads, natural order).  ONE: both
// spins have one hopping magnitude (cids 0 and 1), the coefficient is +-h from
// a register; otherwise it is read from the tables in LDS.
template <typename T, int EPT, bool ONE>
__global__ __launch_bounds__(1024) void k_lz_resident(const ResChain* __restrict__ chains, InterParams I, int steps) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double sh[2][16];
  __shared__ T lut[ONE ? 1 : 512];
  const ResChain& C = chains[blockIdx.x];
  const TwoPassView& V = C.V;
  const int dimup = V.dimup, dimdw = V.dimdw, D = dimup * dimdw;
  const int nthr = blockDim.x, nw = nthr >> 6, tid = threadIdx.x;
  const bool start = C.src || C.gs;
  LzScalars s{};
  if (!start) {
    s = *C.sc;
    if (s.stopped) return;
  }
  // LDS: vector, hop words of both spins in groups of four ([group][string],
  // 16 bytes each), group counts.  A word is the neighbour's offset in dwords
  // from the column's (up) or the row's (down) first element and the
  // coefficient: with ONE the top two bits of +-2.0 (word_coef; 0 pads), else
  // the cid in bits 16 .. 23 (255 pads).
  T* q = reinterpret_cast<T*>(smem);
  const int gu = (V.kup + 3) >> 2, gd = (V.kdw + 3) >> 2;
  uint4* wu = reinterpret_cast<uint4*>(smem + ((size_t)D * sizeof(T) + 15) / 16 * 16);
  uint4* wd = wu + gu * dimup;
  uint8_t* cu = reinterpret_cast<uint8_t*>(wd + gd * dimdw);
  uint8_t* cd = cu + dimup;
  constexpr uint32_t W = sizeof(T) / 4;
  auto stage = [&](const uint32_t* __restrict__ pk, const int32_t* __restrict__ cnt, int dim, int ng, uint32_t step,
                   uint4* w, uint8_t* c) {
    for (int i = tid; i < ng * dim; i += nthr) {
      const int g = i / dim, a = i - g * dim, n = cnt[a];
      uint32_t x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 4 * g + j;
        x[j] = ONE ? 0u : 255u << 16;
        if (k < n) {
          const uint32_t v = pk[(size_t)k * dim + a];
          const uint32_t at = (v & 0xFFFFFFu) * step;
          x[j] = ONE ? at | 0x40000000u | ((v >> 24) & 1u) << 31 : at | (v >> 24) << 16;
        }
      }
      w[i] = uint4{x[0], x[1], x[2], x[3]};
    }
    for (int i = tid; i < dim; i += nthr) c[i] = (uint8_t)((cnt[i] + 3) >> 2);
  };
  stage(V.pk_up, V.cnt_up, dimup, gu, W, wu, cu);
  stage(V.pk_dw, V.cnt_dw, dimdw, gd, W * (uint32_t)dimup, wd, cd);
  const T* lu = reinterpret_cast<const T*>(C.lut_up);
  const T* ld = reinterpret_cast<const T*>(C.lut_dw);
  if (!ONE)
    for (int i = tid; i < 256; i += nthr) {
      lut[i] = i < 255 ? lu[i] : (T)0;
      lut[256 + i] = i < 255 ? ld[i] : (T)0;
    }
  const T hu = lu[0] * (T)0.5, hd = ld[0] * (T)0.5;  // (word_coef gives +-2)
  // the thread's elements: position, diagonal, q_{k-1} or t
  uint32_t pos[EPT];
  T dg[EPT], o[EPT];
  const bool one_orb = I.norb == 1 && I.npairs == 0;
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int e = tid + i * nthr;
    const int idw = e < D ? e / dimup : 0, iup = e < D ? e - idw * dimup : 0;
    pos[i] = (uint32_t)iup | ((uint32_t)idw << 16);
    const uint32_t su = (uint32_t)V.map_up[iup], sd = (uint32_t)V.map_dw[idw];
    const double u = one_orb ? I.U[0] * (double)__popc(su & sd & I.orb_mask[0]) : inter2(I, su, sd);
    dg[i] = (T)(V.dg_up[iup] + V.dg_dw[idw] + u);
    o[i] = (T)0;
  }
  int buf = 0;
  auto total = [&](double v) -> double {
    const double r = block_sum_all(v, sh[buf], nw);
    buf ^= 1;
    return r;
  };
  if (start) {
    // q_0, <seed|seed> in fp64 and the stored vector's norm
    double n2 = 0.0, ss = 0.0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = tid + i * nthr;
      if (e >= D) continue;
      const int iup = (int)(pos[i] & 0xFFFFu), idw = (int)(pos[i] >> 16);
      const double v = C.gs ? res_seed(C, (uint32_t)V.map_up[iup], (uint32_t)V.map_dw[idw], iup, idw) : C.src[e];
      const T qv = (T)v;
      q[e] = qv;
      n2 += v * v;
      ss += (double)qv * (double)qv;
    }
    for (int k = tid; k < C.nmax; k += nthr) C.alpha[k] = C.beta[k] = 0.0;
    n2 = total(n2);
    ss = total(ss);
    s.stopped = (n2 == 0.0 || ss == 0.0) ? 1 : 0;
    s.s_cur = ss > 0.0 ? sqrt(ss) : 1.0;
    s.s_old = 1.0;
    s.norm2 = n2;
    __syncthreads();  // alpha, beta zeroed before thread 0 writes them
  } else {
    const T* qk = reinterpret_cast<const T*>((s.k & 1) ? C.q1 : C.q0);
    const T* qo = reinterpret_cast<const T*>((s.k & 1) ? C.q0 : C.q1);
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = tid + i * nthr;
      if (e < D) {
        q[e] = qk[e];
        o[i] = qo[e];
      }
    }
    __syncthreads();
  }
  bool broke = false;  // breakdown: q holds r, o holds q_k
  for (int n = 0; n < steps && !s.stopped; ++n) {
    if (s.pad) {
      // phase B of step k (o = t): r = t - alpha_k q_k / s_k becomes q_{k+1}
      if (s.k + 1 >= C.nmax) {
        s.stopped = 1;
        break;
      }
      const T am = (T)(s.alpha_k / s.s_cur);
      double nrm = 0.0;
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int e = tid + i * nthr;
        if (e >= D) continue;
        const T qv = q[e];
        const T r = o[i] - am * qv;
        q[e] = r;  // (every gather of q_k was before the sum that gave alpha_k)
        o[i] = qv;
        nrm += (double)r * (double)r;
      }
      const double b = sqrt(total(nrm));
      if (tid == 0) C.beta[s.k + 1] = b;
      s.pad = 0;
      if (!(b > C.brk_tol * (fabs(s.alpha_k) + s.beta_k))) {
        s.stopped = 1;
        broke = true;
        break;
      }
      s.s_old = s.s_cur;
      s.s_cur = b;
      s.beta_k = b;
      s.k += 1;
    }
    // t = H q_k / s_k - beta_k q_{k-1} / s_{k-1}, alpha_k
    const double inv_s = 1.0 / s.s_cur;
    const T ts = (T)inv_s, bo = (T)(s.beta_k / s.s_old);
    T* bst = C.basis ? reinterpret_cast<T*>(C.basis) + (size_t)s.k * D : nullptr;
    const double cx = C.x ? C.ccoef[s.k] * inv_s : 0.0;
    if (bst && tid == 0) C.bscale[s.k] = s.s_cur;
    double part = 0.0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = tid + i * nthr;
      if (e >= D) continue;
      const int iup = (int)(pos[i] & 0xFFFFu), idw = (int)(pos[i] >> 16);
      const unsigned char* qc = reinterpret_cast<const unsigned char*>(q + (e - iup));  // its column
      const unsigned char* qr = reinterpret_cast<const unsigned char*>(q + iup);        // its row
      const T qv = q[e];
      T au = (T)0, ad = (T)0;
      auto gather = [&](const uint4& w, const unsigned char* base, const T* l, T& acc) {
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
        T x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[j] = *reinterpret_cast<const T*>(base + (ONE ? ww[j] << 2 : (ww[j] & 0xFFFFu) << 2));
#pragma unroll
        for (int j = 0; j < 4; ++j) acc += (ONE ? word_coef(ww[j], (T)0) : l[ww[j] >> 16]) * x[j];
      };
      const int nu = cu[iup], nd = cd[idw];
      for (int g = 0; g < nu; ++g) gather(wu[g * dimup + iup], qc, lut, au);
      for (int g = 0; g < nd; ++g) gather(wd[g * dimdw + idw], qr, lut + (ONE ? 0 : 256), ad);
      if (ONE) {
        au *= hu;
        ad *= hd;
      }
      au += dg[i] * qv;
      const T t = (au + ad) * ts - bo * o[i];
      o[i] = t;
      part += (double)t * (double)qv;
      if (bst) bst[e] = qv;
      if (C.x) C.x[e] += cx * (double)qv;
    }
    const double a = total(part * inv_s);
    if (tid == 0) C.alpha[s.k] = a;
    s.alpha_k = a;
    s.nsteps = s.k + 1;
    s.pad = 1;
  }
  if (C.q0) {
    T* ql = reinterpret_cast<T*>(((broke ? s.k + 1 : s.k) & 1) ? C.q1 : C.q0);
    T* qo = reinterpret_cast<T*>(((broke ? s.k + 1 : s.k) & 1) ? C.q0 : C.q1);
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = tid + i * nthr;
      if (e < D) {
        ql[e] = q[e];
        qo[e] = o[i];
      }
    }
  }
  if (tid == 0) *C.sc = s;
}

// ---------------------------------------------------------------- host side
size_t res_lds_bytes(const Sector& s, size_t elem) {
  const SpinTable &u = s.sp[0], &d = s.sp[1];
  return (elem * (size_t)s.dim + 15) / 16 * 16 + 16 * ((size_t)((u.kmax + 3) / 4) * u.dim + (size_t)((d.kmax + 3) / 4) * d.dim) +
         (size_t)u.dim + (size_t)d.dim;
}

bool res_ok(const Sector& s, size_t elem) {
  const SpinTable &u = s.sp[0], &d = s.sp[1];
  if (!u.packed_ok || !d.packed_ok || s.nonlocal) return false;
  if (s.dim < 1 || s.dim > (int64_t)kResMaxRows * 1024 || u.dim > 65535 || d.dim > 65535) return false;
  if (u.kmax > 255 || d.kmax > 255) return false;
  // 160 KB less the static arrays
  return res_lds_bytes(s, elem) <= (size_t)(160 * 1024) - 4096 - 512 * elem;
}

template <typename T, int EPT>
static void launch_res_e(const ResChain* d, int n, int threads, size_t lds, bool one, const InterParams& I, int steps,
                         hipStream_t st) {
  const int lim = 160 * 1024 - 4096 - 512 * (int)sizeof(T);
  if (one) {
    set_lds_limit((const void*)k_lz_resident<T, EPT, true>, lim);
    hipLaunchKernelGGL((k_lz_resident<T, EPT, true>), dim3(n), dim3(threads), lds, st, d, I, steps);
  } else {
    set_lds_limit((const void*)k_lz_resident<T, EPT, false>, lim);
    hipLaunchKernelGGL((k_lz_resident<T, EPT, false>), dim3(n), dim3(threads), lds, st, d, I, steps);
  }
  EDL_HIP(hipGetLastError());
}

template <typename T>
void launch_resident(const ResChain* d, int n, int64_t max_dim, size_t lds, bool one, const InterParams& I, int steps,
                     hipStream_t st) {
  EDL_CHECK(n >= 1 && max_dim >= 1 && max_dim <= (int64_t)kResMaxRows * 1024, "launch_resident: bad chain set");
  // one element a thread up to 1024, then 1024 threads: where an element's
  // terms are added depends on its own chain's size alone, so a chain gives the
  // same bits in any group
  const int th = (int)std::min<int64_t>((max_dim + 63) / 64 * 64, 1024);
  const int rows = (int)((max_dim + th - 1) / th);
  for (int ept : {1, 2, 3, 4, 5, 8, 12, 16}) {
    if (rows > ept) continue;
    switch (ept) {
      case 1: return launch_res_e<T, 1>(d, n, th, lds, one, I, steps, st);
      case 2: return launch_res_e<T, 2>(d, n, th, lds, one, I, steps, st);
      case 3: return launch_res_e<T, 3>(d, n, th, lds, one, I, steps, st);
      case 4: return launch_res_e<T, 4>(d, n, th, lds, one, I, steps, st);
      case 5: return launch_res_e<T, 5>(d, n, th, lds, one, I, steps, st);
      case 8: return launch_res_e<T, 8>(d, n, th, lds, one, I, steps, st);
      case 12: return launch_res_e<T, 12>(d, n, th, lds, one, I, steps, st);
      default: return launch_res_e<T, 16>(d, n, th, lds, one, I, steps, st);
    }
  }
  throw Error("launch_resident: sector too large");
}
template void launch_resident<double>(const ResChain*, int, int64_t, size_t, bool, const InterParams&, int,
                                      hipStream_t);
template void launch_resident<float>(const ResChain*, int, int64_t, size_t, bool, const InterParams&, int,
                                     hipStream_t);

}  // namespace edl
