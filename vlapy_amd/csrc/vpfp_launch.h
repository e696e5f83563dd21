// Internal declarations shared by the translation units of libvpfp.so: the
// error state, the hardware block context the kernel bodies run on, launch
// helpers, and the row and drift dispatchers.  Each dispatcher is compiled in
// a source file of its own per storage type (vpfp_row.hip, vpfp_drift.hip),
// so that the template instantiations build in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "vpfp.h"
#include "vpfp_kernels.h"

namespace vpfp_impl {

// last error message of this thread (vpfp_last_error)
int fail(int code, const std::string& msg);

// VPFP_EHIP with the launch error, if the last launch failed
int launched();

struct GpuCtx {
  int tid, nthr, bid, nblk, bidy;
  __device__ __forceinline__ void sync() { __syncthreads(); }
  __device__ __forceinline__ void fence() { __threadfence(); }
  __device__ __forceinline__ unsigned arrive(unsigned* c) { return atomicAdd(c, 1u); }
  __device__ __forceinline__ void reset(unsigned* c) { __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ __forceinline__ bool any(bool p) { return __any(p); }
  // v of the lane opposite in bit MASK: a DPP move for MASK < 16 (row_mirror
  // and row_half_mirror pair lane l with 15 - l and 7 - l, which also differ
  // in the lower bits: callers only need equal higher bits)
  template <int MASK>
  __device__ __forceinline__ static unsigned dpp(unsigned v) {
    constexpr int ctrl = MASK == 1 ? 0xB1 : MASK == 2 ? 0x4E : MASK == 4 ? 0x141 : 0x140;
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xf, 0xf, true);
  }
  // (x, y) with the lanes of x whose bit MASK is set and the lanes of y whose
  // bit is clear exchanged (MASK 16 or 32)
  template <int MASK>
  __device__ __forceinline__ static void lane_swap(unsigned& x, unsigned& y) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    u2 r;
    if constexpr (MASK == 16)
      r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    else
      r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
  }
  // v plus the opposite lane's v
  template <int MASK>
  __device__ __forceinline__ double add_lane(double v) {
    return fold_lane<MASK>(v, v);
  }
  // lanes with bit MASK clear: lo of both lanes, else hi of both
  template <int MASK>
  __device__ __forceinline__ double fold_lane(double lo, double hi) {
    const unsigned long long l = __double_as_longlong(lo), h = __double_as_longlong(hi);
    if constexpr (MASK >= 16) {
      unsigned x0 = (unsigned)l, x1 = (unsigned)(l >> 32), y0 = (unsigned)h, y1 = (unsigned)(h >> 32);
      lane_swap<MASK>(x0, y0);
      lane_swap<MASK>(x1, y1);
      return __longlong_as_double(((unsigned long long)x1 << 32) | x0) +
             __longlong_as_double(((unsigned long long)y1 << 32) | y0);
    } else {
      const bool up = (tid & MASK) != 0;
      const unsigned long long s = up ? l : h;
      const unsigned r0 = dpp<MASK>((unsigned)s), r1 = dpp<MASK>((unsigned)(s >> 32));
      return (up ? hi : lo) + __longlong_as_double(((unsigned long long)r1 << 32) | r0);
    }
  }
  // v_mfma_f32_16x16x4_f32: D = A B + C (layout at vp::drift_dft_body)
  __device__ __forceinline__ vp::f4 mfma_16x16x4(float a, float b, vp::f4 acc) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    f4v cv = {acc.v[0], acc.v[1], acc.v[2], acc.v[3]};
    cv = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, cv, 0, 0, 0);
    return vp::f4{{cv[0], cv[1], cv[2], cv[3]}};
  }
};

#define VPFP_CTX \
  vpfp_impl::GpuCtx c{(int)threadIdx.x, (int)blockDim.x, (int)blockIdx.x, (int)gridDim.x, (int)blockIdx.y}

// LDS per workgroup on gfx950
constexpr int kMaxLds = 160 * 1024;

// dynamic LDS above 64 KiB must be enabled per kernel
template <class K>
int set_lds(K kern, int bytes) {
  if (bytes > 65536) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(VPFP_EHIP, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  }
  return VPFP_OK;
}

constexpr int qfor(int M) { return M < 8 ? M : 8; }

#define VPFP_SWITCH_M(M, CALL, MAXM)                 \
  switch (M) {                                       \
    case 2: return CALL(2);                          \
    case 4: return CALL(4);                          \
    case 8: return CALL(8);                          \
    case 16: return CALL(16);                        \
    case 32: return CALL(32);                        \
    case 64: return CALL(64);                        \
    case 128: return CALL(128);                      \
    case 256: return CALL(256);                      \
    case 512: return CALL(512);                      \
    case 1024: if (MAXM >= 1024) return CALL(1024);  \
      break;                                         \
    case 2048: if (MAXM >= 2048) return CALL(2048);  \
      break;                                         \
    case 4096: if (MAXM >= 4096) return CALL(4096);  \
      break;                                         \
  }

// Row kernels (vpfp_row.hip): q = values per thread (0: row-count rule).
// The plain kernels take f itself, the _bg kernels delta-f storage
// (a.bg and a.bg_hat set).
int row_dispatch_plain(const vp::RowArgs<double>& a, hipStream_t s, int q);
int row_dispatch_plain(const vp::RowArgs<float>& a, hipStream_t s, int q);
int row_dispatch_bg(const vp::RowArgs<double>& a, hipStream_t s, int q);
int row_dispatch_bg(const vp::RowArgs<float>& a, hipStream_t s, int q);

// The same over the segments of several batches of one nv (vpfp_group_*);
// the dispatch fills in the segments' first workgroups
int row_multi_dispatch_plain(const vp::RowMulti<double>& m, hipStream_t s, int q);
int row_multi_dispatch_plain(const vp::RowMulti<float>& m, hipStream_t s, int q);
int row_multi_dispatch_bg(const vp::RowMulti<double>& m, hipStream_t s, int q);
int row_multi_dispatch_bg(const vp::RowMulti<float>& m, hipStream_t s, int q);

// Drift kernels (vpfp_drift.hip): C columns per tile, gx workgroups striding
// over the column tiles; gy > 0: a batch of gy instances (grid y = instance)
int drift_dispatch(const vp::DriftArgs<double>& a, int C, int gx, hipStream_t s, int gy);
int drift_dispatch(const vp::DriftArgs<float>& a, int C, int gx, hipStream_t s, int gy);
// several batches of one nx (vpfp_group_*): segment s has n_inst * gx workgroups
int drift_multi_dispatch(const vp::DriftMulti<double>& m, int C, hipStream_t s);
int drift_multi_dispatch(const vp::DriftMulti<float>& m, int C, hipStream_t s);

}  // namespace vpfp_impl
