// Internal launcher declarations shared by the kernel translation units and
// the C ABI layer (abi.hip). Launchers assume validated arguments.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/ringmaster_amd.h"
#include "rmx_common.h"
#include "rmx_wgmap.h"

namespace rmx {

hipError_t launch_attn_fwd(const rmx_attn_layout& L, const rmx_fwd_problem* probs, int n,
                           hipStream_t stream);
hipError_t launch_attn_bwd_delta(const rmx_attn_layout& L, const void* out, int out_f32,
                                 const uint16_t* dout, float* delta, const float* lse, float* nlse,
                                 int sq, hipStream_t stream);
// A split dK/dV launch's workspace: `base` holds n splits x (dV, dK) of `grad` elements each, a
// gradient being rows [problem][batch, kv head][key] of head_dim; `empty` one word per key block
// ([problem][batch, kv head][block], RMX_MASK_DOC only): 1 where no query attends it.
struct SplitParts {
  float* base;
  int32_t* empty;
  int64_t grad;
};
__host__ __device__ constexpr int split_key_blocks(int sk) { return (sk + 127) / 128; }
// How a launch's key blocks are split over workgroups (n = 1: not at all), the elements of its
// dK (or dV) and its key blocks.
struct DkdvSplit {
  int n;
  int64_t grad, blocks;
  size_t bytes() const { return n > 1 ? (size_t)n * 2 * (size_t)grad * 4 + (size_t)blocks * 4 : 0; }
  SplitParts at(void* ws) const {
    float* const base = static_cast<float*>(ws);
    return {base, reinterpret_cast<int32_t*>(base + n * 2 * grad), grad};
  }
};
DkdvSplit dkdv_split(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n);
hipError_t launch_dkdv_fold(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n,
                            const DkdvSplit& split, void* ws, hipStream_t stream);
// ws: split.bytes() of workspace
hipError_t launch_attn_bwd(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n,
                           const DkdvSplit& split, void* ws, hipStream_t stream);
hipError_t launch_lse_merge(float* out, float* lse, const void* blk_out, int blk_type,
                            const float* blk_lse, int batch, int seq, int heads, int head_dim,
                            const int64_t* os, const int64_t* ls, const int64_t* bos,
                            const int64_t* bls, int init, hipStream_t stream);
hipError_t launch_cast_half(const float* const* src, uint16_t* const* dst, const int64_t* n,
                            int count, int f16, hipStream_t stream);
hipError_t launch_zigzag(const void* src, void* dst, int batch, int seq, int world, int rank,
                         int64_t row_bytes, int64_t bstride, const void* pad_row, int scatter,
                         hipStream_t stream);
hipError_t launch_linear_scan_fwd(const float* a, const float* b, const float* hin, float* h,
                                  float* chunk_state, int batch, int L, int d, int groups,
                                  int world, hipStream_t stream);
hipError_t launch_linear_scan_bwd(const float* a, const float* h, const float* hin,
                                  const float* dh, float* da, float* db, float* dhin, int batch,
                                  int L, int d, int groups, int world, hipStream_t stream);
// L-parallel (chained) scan: channel tiling, chunk length and workspace layout of one shape
struct ScanChunkPlan {
  int V, amode, cw_log2, lg_log2, CT, TC, ntiles, nchunks;
  bool two_pass;  // reduce-then-rescan instead of the single pass with look-back
  size_t words_off, bytes;
};
ScanChunkPlan scan_chunk_plan(int batch, int L, int d, int groups);
hipError_t launch_linear_scan_fwd_chunked(const ScanChunkPlan& p, const float* a, const float* b,
                                          const float* hin, float* h, float* cs, void* ws,
                                          int batch, int L, int d, int groups, int world,
                                          hipStream_t stream);
// the failure word of an L-parallel scan's workspace (after a stream synchronize)
int read_linear_scan_failure(const void* ws, hipStream_t stream, hipError_t* err);
hipError_t launch_linear_scan_bwd_chunked(const ScanChunkPlan& p, const float* a, const float* h,
                                          const float* hin, const float* dh, float* da, float* db,
                                          float* dhin, void* ws, int batch, int L, int d,
                                          int groups, hipStream_t stream);

hipError_t launch_mamba2_correction(const uint16_t* out, uint16_t* y, const float* h_final,
                                    float* h_final_out, const uint16_t* C, const float* cum_A,
                                    const float* h_prev, const int32_t* seq_idx, int batch, int T,
                                    int nheads, int head_dim, int ngroups, int d_state,
                                    hipStream_t stream);
size_t mamba2_bwd_workspace(int batch, int T, int nheads, int head_dim, int ngroups,
                            int d_state);
hipError_t mamba2_bwd_scratch(void** out);
hipError_t launch_mamba2_correction_bwd(const uint16_t* gy, const float* ghf, const uint16_t* C,
                                        const float* cum_A, const float* h_prev,
                                        const int32_t* seq_idx, uint16_t* gC, float* g_cumA,
                                        float* g_hprev, void* workspace, int batch, int T,
                                        int nheads, int head_dim, int ngroups, int d_state,
                                        hipStream_t stream);
hipError_t launch_mamba2_dt_cumsum(const void* dt, int dt_f32, const float* bias, const float* A,
                                   int softplus, float* cum_A, float* e, float* decay, int rows,
                                   int T, int H, hipStream_t stream);
hipError_t launch_mamba2_dt_cumsum_bwd(const void* dt, int dt_f32, const float* bias,
                                       const float* A, int softplus, const float* g_cum,
                                       const float* g_e, const float* g_decay, const float* decay,
                                       float* g_dt, float* g_A, float* g_bias, int rows, int T,
                                       int H, int closed, void* ws, hipStream_t stream);
size_t mamba2_dt_bwd_workspace(int rows, int T, int H);
hipError_t launch_mamba2_chunk_state(const uint16_t* x, const uint16_t* B, const float* e,
                                     const float* cum_A, const int32_t* t0, float* state,
                                     int rows, int T, int H, int D, int G, int N,
                                     hipStream_t stream);
size_t mamba2_chunk_state_bwd_workspace(int rows, int H, int D, int N);
hipError_t launch_mamba2_chunk_state_bwd(const uint16_t* x, const uint16_t* B, const float* e,
                                         const float* cum_A, const int32_t* t0,
                                         const float* g_state, uint16_t* g_x, uint16_t* g_B,
                                         float* g_e, float* g_cum, int rows, int T, int H, int D,
                                         int G, int N, void* workspace, hipStream_t stream);
hipError_t launch_causal_conv1d_cp(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                   const int32_t* doc, uint16_t* y, int world, int batch, int C,
                                   int L, int W, int act, hipStream_t stream);
hipError_t launch_causal_conv1d_cp_bwd(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                       const int32_t* doc, const uint16_t* dy, uint16_t* dx,
                                       float* dw, float* db, int world, int batch, int C, int L,
                                       int W, int act, hipStream_t stream);

}  // namespace rmx

namespace rmx {

// ---------------------------------------------------------------------------
// 16-bit element types of the attention kernels (RMX_DTYPE_BF16, RMX_DTYPE_F16).
// Operands travel as bf16x8 bit patterns in both cases (loads, LDS tiles, transposed
// reads and the sign flip of V are bit operations on 16-bit lanes); only the MFMA and
// the fp32 <-> 16-bit conversions (round to nearest even) depend on the type.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int DT>
__device__ __forceinline__ f32x16 mfma32t(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  if constexpr (DT == RMX_DTYPE_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// Two floats -> two packed 16-bit elements (lo in bits 0..15).
template <int DT>
__device__ __forceinline__ uint32_t cvt_pk(float lo, float hi) {
  if constexpr (DT == RMX_DTYPE_F16) {
    const f32x2 f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
  } else {
    return cvt_pk_bf16(lo, hi);
  }
}
template <int DT>
__device__ __forceinline__ uint16_t f2e(float f) {
  if constexpr (DT == RMX_DTYPE_F16)
    return __builtin_bit_cast(uint16_t, (_Float16)f);
  else
    return f2bf(f);
}
template <int DT>
__device__ __forceinline__ float e2f(uint32_t bits16) {
  if constexpr (DT == RMX_DTYPE_F16)
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
  else
    return bf2f((uint16_t)bits16);
}
template <int DT>
__device__ __forceinline__ bf16x8 pack8t(const float* v) {
  u32x4 u;
  u[0] = cvt_pk<DT>(v[0], v[1]);
  u[1] = cvt_pk<DT>(v[2], v[3]);
  u[2] = cvt_pk<DT>(v[4], v[5]);
  u[3] = cvt_pk<DT>(v[6], v[7]);
  return __builtin_bit_cast(bf16x8, u);
}

// ---------------------------------------------------------------------------
// Attention dropout. Element (batch b, q head h, query q, key k) of a call with
// dropout is kept when
//   fmix32(bhmix ^ (q + q0) * kDropQ ^ (k + k0) * kDropK) >= threshold,
//   bhmix = fmix32(seed_lo ^ fmix32(seed_hi ^ (b * hq + h) * kDropBH)),
// with fmix32 the MurmurHash3 finalizer, threshold = floor(p 2^32) and (q0, k0) the
// problem's coordinate offsets (a ring block's place in the gathered sequence).
// Kept probabilities are scaled by 1 / (1 - p); lse is that of the undropped scores.
// Every element is its own counter, so each kernel evaluates the mask in whatever
// lane layout it holds the scores in, and the forward and both backward kernels
// agree on it bit for bit.
constexpr uint32_t kDropQ = 0x85ebca77u, kDropK = 0xc2b2ae3du, kDropBH = 0x9e3779b9u;
__device__ __forceinline__ uint32_t fmix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x85ebca6bu;
  x ^= x >> 13;
  x *= 0xc2b2ae35u;
  x ^= x >> 16;
  return x;
}
__device__ __forceinline__ uint32_t drop_bhmix(const rmx_attn_layout& L, int bb, int head) {
  return fmix32(L.drop_seed_lo ^ fmix32(L.drop_seed_hi ^ (uint32_t)(bb * L.hq + head) * kDropBH));
}
// qterm = bhmix ^ (q + q0) * kDropQ, kterm = (k + k0) * kDropK
__device__ __forceinline__ bool drop_keep(uint32_t qterm, uint32_t kterm, uint32_t thr) {
  return fmix32(qterm ^ kterm) >= thr;
}

// Host side: whether a forward or dQ launch (head dims up to 128) runs workgroups of 4 waves
// (128 queries) instead of 8 (256): while they are at most one per CU. A 4-wave workgroup has
// one wave per SIMD and takes about 0.75 of an 8-wave one's time for the same keys, so twice the
// workgroups win as long as they run at once: forward / dQ, us, 8 -> 4 waves: 2048^2 causal, 8
// heads of 128 (64 workgroups of 8) 63 -> 49 / 69 -> 55, 16 heads (128) 66 -> 53 / 73 -> 58; past
// that, 4096^2 unmasked of 16 heads (256) 146 -> 194 / 181 -> 188.
template <class Prob>
inline bool half_workgroups(const rmx_attn_layout& L, const Prob* probs, int n) {
  int64_t wgs = 0;
  for (int i = 0; i < n; ++i) wgs += (int64_t)L.batch * L.hq * ((probs[i].sq + 127) / 128);
  return wgs <= 256;
}

// Host side: the keep threshold floor(p 2^32) and the scale 1 / (1 - p) of dropout p.
inline void drop_params(float p, uint32_t* thr, float* scale) {
  if (!(p > 0.f)) {
    *thr = 0u;
    *scale = 1.f;
    return;
  }
  const double t = (double)p * 4294967296.0;
  *thr = t >= 4294967295.0 ? 4294967295u : (uint32_t)t;
  *scale = (float)(1.0 / (1.0 - (double)p));
}

// Host side: order[] = problem indices sorted by cost[] descending (stable).
inline void order_by_cost(int n, const long long* cost, int* order) {
  for (int i = 0; i < n; ++i) order[i] = i;
  for (int i = 1; i < n; ++i) {
    const int o = order[i];
    int j = i - 1;
    while (j >= 0 && cost[order[j]] < cost[o]) {
      order[j + 1] = order[j];
      --j;
    }
    order[j + 1] = o;
  }
}

}  // namespace rmx
