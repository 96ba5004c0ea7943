// Block-attention backward for gfx950 using the GLOBAL (ring-merged) out/lse.
//
// Reference semantics: the explicit global-lse backward of
// ring/p2p_attn.py:243-281 and ring/varlen_blocks.py:176-200:
//   P  = exp(scale*Q K^T + mask - lse)     (lse = global, natural log)
//   dV = P^T dO;  dP = dO V^T;  delta = rowsum(dO * O_global)
//   dS = P * (dP - delta);  dQ = scale dS K;  dK = scale dS^T Q
// with the GQA fold of dK/dV over the q-head group (:193-197).
//
// Two kernels, no atomics:
//   * attn_bwd_dq   (Q-major, lane = query): S^T, dP^T, dQ^T = K^T dS^T; the
//     fp32 dq rows are owned by one workgroup.
//   * attn_bwd_dkdv (KV-major, lane = key): S, dP, dV += P^T dO,
//     dK += dS^T Q; the workgroup owns its keys and loops over every q-head
//     of the GQA group, so the fold needs no cross-workgroup reduction.
//
// This unit holds the delta kernel, the dispatch over head dims and the head-dim-256
// instantiations; the head-dim-64 and -128 ones are in attn_bwd_vf.hip, built with
// VGPR-form MFMAs (the kernels themselves: attn_bwd_kernels.h).
#include "attn_bwd_kernels.h"

namespace rmx {

// ---------------------------------------------------------------- delta
// delta = rowsum(dout * out). `out` is the bf16 output (o_* strides) or, when
// OUT_F32, the fp32 merged output (a_* strides): the fp32 form keeps the bf16
// rounding of out (up to |dout|*|out|*2^-9 per element) out of dS = P (dP - delta).
// With nlse, the same pass writes nlse = -lse log2(e) (the per-query exponent
// offset of the dK/dV kernel) at the same [b, h, s] position. Rows run query-fastest
// (row = (b, h, q)), so the 4-byte delta, lse and nlse words of neighbouring rows share
// cache lines; head-fastest rows put each word on its own line (8x the written bytes).
template <int HD, bool OUT_F32, int DT>
__global__ __launch_bounds__(256) void attn_bwd_delta_kernel(const rmx_attn_layout L,
                                                             const void* __restrict__ out,
                                                             const uint16_t* __restrict__ dout,
                                                             float* __restrict__ delta,
                                                             const float* __restrict__ lse,
                                                             float* __restrict__ nlse, int sq) {
  constexpr int TPR = HD / 8;  // threads per row
  const int rows = L.batch * sq * L.hq;
  const int row = blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  const int part = threadIdx.x % TPR;
  float acc = 0.f;
  int bb = 0, q = 0, h = 0;
  if (row < rows && 8 * part >= L.head_dim) {  // columns past the head dim: nothing to add
    q = row % sq;
    h = (row / sq) % L.hq;
    bb = row / (L.hq * sq);
  } else if (row < rows) {
    q = row % sq;
    h = (row / sq) % L.hq;
    bb = row / (L.hq * sq);
    const int64_t off = bb * L.o_sb + (int64_t)q * L.o_ss + h * L.o_sh + 8 * part;
    const u32x4 b = ld16(dout + off);
    float o[8];
    if (OUT_F32) {
      const float* op = reinterpret_cast<const float*>(out) + bb * L.a_sb + (int64_t)q * L.a_ss +
                        h * L.a_sh + 8 * part;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(op);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(op + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o[i] = x0[i];
        o[4 + i] = x1[i];
      }
    } else {
      const u32x4 a = ld16(reinterpret_cast<const uint16_t*>(out) + off);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o[2 * i] = e2f<DT>(a[i] & 0xffffu);
        o[2 * i + 1] = e2f<DT>(a[i] >> 16);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc += o[2 * i] * e2f<DT>(b[i] & 0xffffu);
      acc += o[2 * i + 1] * e2f<DT>(b[i] >> 16);
    }
  }
#pragma unroll
  for (int m = TPR / 2; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 64);
  if (row < rows && part == 0) {
    const int64_t lo = bb * L.l_sb + h * L.l_sh + q;
    delta[lo] = acc;
    if (nlse) nlse[lo] = lse[lo] * -kLog2e;
  }
}

template <int HD, int DT>
static void launch_delta_t(const rmx_attn_layout& L, const void* out, int out_f32,
                           const uint16_t* dout, float* delta, const float* lse, float* nlse,
                           int sq, int64_t rows, hipStream_t stream) {
  constexpr int RPB = 256 / (HD / 8);  // rows per block
  const int grid = (int)((rows + RPB - 1) / RPB);
  if (out_f32)
    hipLaunchKernelGGL((attn_bwd_delta_kernel<HD, true, DT>), dim3(grid), dim3(256), 0, stream, L,
                       out, dout, delta, lse, nlse, sq);
  else
    hipLaunchKernelGGL((attn_bwd_delta_kernel<HD, false, DT>), dim3(grid), dim3(256), 0, stream,
                       L, out, dout, delta, lse, nlse, sq);
}

hipError_t launch_attn_bwd_delta(const rmx_attn_layout& L, const void* out, int out_f32,
                                 const uint16_t* dout, float* delta, const float* lse, float* nlse,
                                 int sq, hipStream_t stream) {
  const int64_t rows = (int64_t)L.batch * sq * L.hq;
  if (rows == 0) return hipSuccess;
  const bool f16 = L.dtype == RMX_DTYPE_F16;
  if (L.head_dim > 128 && f16)
    launch_delta_t<256, RMX_DTYPE_F16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  else if (L.head_dim > 128)
    launch_delta_t<256, RMX_DTYPE_BF16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  else if (L.head_dim > 64 && f16)
    launch_delta_t<128, RMX_DTYPE_F16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  else if (L.head_dim > 64)
    launch_delta_t<128, RMX_DTYPE_BF16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  else if (f16)
    launch_delta_t<64, RMX_DTYPE_F16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  else
    launch_delta_t<64, RMX_DTYPE_BF16>(L, out, out_f32, dout, delta, lse, nlse, sq, rows, stream);
  return hipGetLastError();
}

// ---------------------------------------------------------------- dK/dV splits
// Workgroups per key block of a dK/dV launch. The launch's time is estimated for every
// number of splits from the tile counts of its key blocks (the masks' own ranges; documents,
// whose ranges only the device knows, count as causal: the longest they can be): a tile and a
// workgroup cost what the kernels measure on a lone CU,
// workgroups run in rounds over the CUs, and a split launch adds the fold kernel and the
// partial gradients' traffic. Launches of many rounds stay whole. Whole -> split, us a launch:
// 4096^2 causal 32/8 heads of 128 365 -> 266 (2), 2048^2 182 -> 91 (3), 512^2 56 -> 33 (4);
// 4096^2 causal 16/4 heads of 256 803 -> 296 (4), of 64 236 -> 92 (4); the same 4096^2 with
// 32 KV heads of 128 fills the chip and stays whole (267; an earlier build 321, in two 419).
// A packed ring's backward (every kernel of it), whole -> split: 4 ranks x 1024 tokens, 8/2 heads of
// 128, documents of 64 tokens 269 -> 214, of 2048 504 -> 321; 8 x 766, 4/2 heads of 64, of 364 217 -> 209;
// over 22 rings of the range at most 1.02 of the whole one's time.
DkdvSplit dkdv_split(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n) {
  constexpr int kCu = 256, kBkv = 128, kMaxSplit = 16;
  DkdvSplit out{1, 0, 0};
  const int hd = L.head_dim > 128 ? 256 : L.head_dim > 64 ? 128 : 64;
  const int bq = hd == 256 ? 32 : 64, G = L.hq / L.hkv;
  // us: per tile, per workgroup, of the fold launch
  const double tile = hd == 256 ? 1.6 : hd == 128 ? 1.4 : 1.1, wg = hd == 256 ? 12. : hd == 128 ? 6. : 4.,
               fold = 5.;
  const int64_t per = (int64_t)L.batch * L.hkv;
  int64_t blocks = 0, keys = 0;
  for (int i = 0; i < n; ++i) {
    const rmx_bwd_problem& p = probs[i];
    if (p.sq == 0 || p.sk == 0 || p.dkv_mode == RMX_GRAD_NONE) continue;
    blocks += per * split_key_blocks(p.sk);
    keys += per * p.sk;
  }
  if (blocks == 0 || blocks >= 4 * kCu) return out;
  int64_t tiles = 0;  // of all blocks
  int longest = 0;
  for (int i = 0; i < n; ++i) {
    const rmx_bwd_problem& p = probs[i];
    if (p.sq == 0 || p.sk == 0 || p.dkv_mode == RMX_GRAD_NONE) continue;
    const int64_t nqt = (p.sq + bq - 1) / bq, off = (int64_t)p.sk - p.sq + p.window_right;
    for (int64_t k0 = 0; k0 < p.sk; k0 += kBkv) {
      int64_t lo = 0, hi = nqt;
      if (L.mask != RMX_MASK_FULL) {
        lo = k0 - off <= 0 ? 0 : (k0 - off) / bq;
        if (lo > nqt) lo = nqt;
      }
      if (p.has_window) {
        const int64_t qmax = k0 + kBkv - 1 + (int64_t)p.window_left - ((int64_t)p.sk - p.sq);
        hi = qmax < 0 ? 0 : (qmax / bq + 1 < nqt ? qmax / bq + 1 : nqt);
      }
      const int t = hi > lo ? (int)(hi - lo) * G : 0;
      tiles += per * t;
      longest = t > longest ? t : longest;
    }
  }
  double best = 0;
  for (int s = 1; s <= kMaxSplit && (s == 1 || s <= longest); ++s) {
    const double one = wg + tile * ((longest + s - 1) / s);
    const double share = (wg * blocks * s + tile * tiles) / kCu;  // an even share of the work
    // even blocks run in whole rounds; uneven ones fill the CUs behind the longest
    const bool even = tiles == blocks * (int64_t)longest;
    double t = even ? one * ((blocks * s + kCu - 1) / kCu) : (share > one ? share : one) + 0.5 * tile;
    if (s > 1) t += fold + 1e6 * (double)s * keys * L.head_dim * 8 * 2 / 4e12;
    if (s == 1 || t < best) {
      best = t;
      out.n = s;
    }
  }
  out.grad = keys * L.head_dim;
  out.blocks = blocks;
  return out;
}

struct FoldParams {
  rmx_attn_layout L;
  rmx_bwd_problem P[RMX_MAX_BATCHED];
  SplitParts parts;
  int nsplit;
};

// Sum of the splits' partial dV (blockIdx.y 0) and dK (1) rows, stored in their problem's mode.
// Bound by its traffic (nsplit fp32 reads per element); a thread owns 4 columns of a row, HD / 4
// threads a row, the splits' loads four at a time in flight.
template <int HD, int DT>
__global__ __launch_bounds__(256) void dkdv_fold_kernel(const FoldParams prm) {
  constexpr int CPR = HD / 4, RPB = 256 / CPR;
  const rmx_attn_layout& L = prm.L;
  const int g = blockIdx.y, D = L.head_dim, per = L.batch * L.hkv;
  const int col = 4 * (threadIdx.x % CPR);
  // problem p of this workgroup, its first row and key block (a split launch has under 1024 key
  // blocks: rows fit 32 bits); one problem per workgroup keeps p and its fields in scalars
  int p = 0, wg = blockIdx.x, row0 = 0, block = 0;
  for (int n; wg >= (n = (per * prm.P[p].sk + RPB - 1) / RPB); ++p) {
    wg -= n;
    row0 += per * prm.P[p].sk;
    block += per * split_key_blocks(prm.P[p].sk);
  }
  const rmx_bwd_problem& P = prm.P[p];
  const int local = wg * RPB + threadIdx.x / CPR;  // (batch, kv head, key)
  if (col >= D || local >= per * P.sk) return;
  const int bh = local / P.sk, key = local - bh * P.sk;
  const int bb = bh / L.hkv, h = bh % L.hkv;
  // (an empty block is its first workgroup's, which has stored it if the mode writes)
  if (L.mask == RMX_MASK_DOC && prm.parts.empty[block + bh * split_key_blocks(P.sk) + key / 128]) return;
  const float* src = prm.parts.base + g * prm.parts.grad + (int64_t)(row0 + local) * D + col;
  f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 4
  for (int s = 1; s < prm.nsplit; ++s)
    v += *reinterpret_cast<const f32x4*>(src + s * 2 * prm.parts.grad);
  const int mode = P.dkv_mode;
  const bool rd = mode == RMX_GRAD_ACC_F32 || mode == RMX_GRAD_ACC_FINAL;
  const bool w32 = mode == RMX_GRAD_WRITE_F32 || mode == RMX_GRAD_ACC_F32;
  float* const acc = (g ? P.dk_acc : P.dv_acc) + bb * L.ka_sb + (int64_t)key * L.ka_ss + h * L.ka_sh + col;
  uint16_t* const bf = (g ? P.dk : P.dv) + bb * L.dk_sb + (int64_t)key * L.dk_ss + h * L.dk_sh + col;
  const bool vec = (!(rd || w32) || ((uintptr_t)acc & 15) == 0) && (w32 || ((uintptr_t)bf & 7) == 0);
  if (vec) {
    if (rd) v += *reinterpret_cast<const f32x4*>(acc);
    if (w32) {
      *reinterpret_cast<f32x4*>(acc) = v;
    } else {
      u32x2 w;
      w[0] = cvt_pk<DT>(v[0], v[1]);
      w[1] = cvt_pk<DT>(v[2], v[3]);
      *reinterpret_cast<u32x2*>(bf) = w;
    }
    return;
  }
  for (int e = 0; e < 4; ++e) {  // a caller pointer below vector alignment
    const float x = rd ? acc[e] + v[e] : v[e];
    if (w32)
      acc[e] = x;
    else
      bf[e] = f2e<DT>(x);
  }
}

template <int HD>
static void launch_fold_t(const FoldParams& prm, int n, bool f16, hipStream_t stream) {
  constexpr int RPB = 256 / (HD / 4);
  int wgs = 0;
  for (int i = 0; i < n; ++i)
    wgs += (prm.L.batch * prm.L.hkv * prm.P[i].sk + RPB - 1) / RPB;
  const dim3 grid(wgs, 2);
  if (f16)
    hipLaunchKernelGGL((dkdv_fold_kernel<HD, RMX_DTYPE_F16>), grid, dim3(256), 0, stream, prm);
  else
    hipLaunchKernelGGL((dkdv_fold_kernel<HD, RMX_DTYPE_BF16>), grid, dim3(256), 0, stream, prm);
}

hipError_t launch_dkdv_fold(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n,
                            const DkdvSplit& split, void* ws, hipStream_t stream) {
  FoldParams prm;
  prm.L = L;
  for (int i = 0; i < n; ++i) prm.P[i] = probs[i];
  prm.parts = split.at(ws);
  prm.nsplit = split.n;
  const bool f16 = L.dtype == RMX_DTYPE_F16;
  if (L.head_dim > 128)
    launch_fold_t<256>(prm, n, f16, stream);
  else if (L.head_dim > 64)
    launch_fold_t<128>(prm, n, f16, stream);
  else
    launch_fold_t<64>(prm, n, f16, stream);
  return hipGetLastError();
}

// the head-dim-64 and -128 launches are instantiated in attn_bwd_vf.hip
extern template hipError_t launch_bwd_t<64, RMX_DTYPE_BF16, false>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<64, RMX_DTYPE_BF16, true>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<64, RMX_DTYPE_F16, false>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<64, RMX_DTYPE_F16, true>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<128, RMX_DTYPE_BF16, false>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<128, RMX_DTYPE_BF16, true>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<128, RMX_DTYPE_F16, false>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);
extern template hipError_t launch_bwd_t<128, RMX_DTYPE_F16, true>(const rmx_attn_layout&,
    const rmx_bwd_problem*, int, const DkdvSplit&, void*, hipStream_t);

template <int DT, bool DROP>
static hipError_t launch_bwd_hd(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n,
                                const DkdvSplit& split, void* ws, hipStream_t stream) {
  if (L.head_dim > 128) return launch_bwd_t<256, DT, DROP>(L, probs, n, split, ws, stream);
  if (L.head_dim > 64) return launch_bwd_t<128, DT, DROP>(L, probs, n, split, ws, stream);
  return launch_bwd_t<64, DT, DROP>(L, probs, n, split, ws, stream);
}

hipError_t launch_attn_bwd(const rmx_attn_layout& L, const rmx_bwd_problem* probs, int n,
                           const DkdvSplit& split, void* ws, hipStream_t stream) {
  const bool f16 = L.dtype == RMX_DTYPE_F16, drop = L.dropout_p > 0.f;
  if (drop)
    return f16 ? launch_bwd_hd<RMX_DTYPE_F16, true>(L, probs, n, split, ws, stream)
               : launch_bwd_hd<RMX_DTYPE_BF16, true>(L, probs, n, split, ws, stream);
  return f16 ? launch_bwd_hd<RMX_DTYPE_F16, false>(L, probs, n, split, ws, stream)
             : launch_bwd_hd<RMX_DTYPE_BF16, false>(L, probs, n, split, ws, stream);
}

}  // namespace rmx
