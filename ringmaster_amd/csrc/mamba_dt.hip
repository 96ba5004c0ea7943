// Mamba2 CP chunk decay from dt (strategies/mamba.py:276-283): per row (rank
// shard x batch) and head,
//   e_t = softplus(dt_t + dt_bias) when dt_softplus, else dt_t
//   cum_A_t = sum_{s<=t} A e_s,   decay = exp(cum_A_{T-1})
// and the gradient of that map. softplus follows torch (beta 1, threshold 20:
// x > 20 -> x).
//
// Both directions are a prefix (suffix) sum along T. The rows of a call are few (8 for 8
// ranks), so a workgroup per row leaves the chip idle: walking T = 8192 tokens of 64 heads
// that way took 1958 us forward and 1806 us backward, the softplus on 8 of 256 CUs. The
// tokens are cut into chunks, one workgroup each: 512 threads, HT = 8..64 heads (the least
// that covers H) by 512 / HT runs of 16 tokens, a thread holding its run in registers (16
// loads in flight, softplus computed once). The chunks meet through the output itself, so no
// workspace is needed and no workgroup waits for another:
//   forward: chunk scans (each from zero) / the scan of the chunks' last tokens, in place /
//     every other token plus the last token of the chunk before;
//   backward: chunk sums of g_cum into g_dt at each chunk's first token / those turned into
//     what enters each chunk / the chunks, each reading its own first token before the
//     barrier that precedes its stores; with a workspace they leave their parts of dA and
//     d(bias) there and a fourth launch adds those in order (see mamba2_dt_fold_kernel).
// A sequence of one chunk is one launch. At 8 rows x 8192 x 64 the three launches take 19 + 5 + 9
// us forward and the four 4 + 5 + 24 + 4 us backward, 25 MB and 42 MB moved by the first and the
// third of these;
// cum_A's rms error falls from 1e-6 to 6e-8 (shorter chains of sums).
#include "rmx_kernels.h"

namespace rmx {

struct DtArgs {
  const void* dt;        // [rows, T, H] bf16 or fp32
  int dt_f32;
  const float* bias;     // [H] or null
  const float* A;        // [H]
  int softplus;
  float* cum_A;          // fwd out [rows, T, H]
  float* e_out;          // fwd out [rows, T, H] (effective dt) or null
  const float* g_e;      // bwd in [rows, T, H] (direct gradient of e) or null
  float* decay;          // fwd out / bwd in [rows, H]
  const float* g_cum;    // bwd in [rows, T, H] or null
  const float* g_decay;  // bwd in [rows, H] or null
  float* g_dt;           // bwd out [rows, T, H] (fp32)
  float* g_A;            // bwd += [H]
  float* g_bias;         // bwd += [H] (softplus only) or null
  float* part;           // bwd workspace or null: dA and d(bias) parts [2][rows * nchunk][H]
  int rows, T, H;
  int nchunk;
};

__device__ __forceinline__ float dt_at(const DtArgs& a, int64_t i) {
  return a.dt_f32 ? reinterpret_cast<const float*>(a.dt)[i]
                  : bf2f(reinterpret_cast<const uint16_t*>(a.dt)[i]);
}
// softplus(x) = max(x, 0) + log1p(z) and its derivative, with z = exp(-|x|). log1p(z) =
// 2 atanh(s) with s = z / (2 + z) <= 1/3, and 2 s = z - s z: z - s (z - R), R = a s^2 the atanh
// series past its first term (cut at 2e-9 of the whole). The roundings of s (ds), of z - s z and of the
// sum are carried along, so that one is left: e's rms error is 3.40e-8 on a layer's steps
// against 3.44e-8 with the library's log1pf(expf(x)) (3.52e-8 without the corrections, which cost
// 2 us). The first forward kernel takes 17-19 us instead of 28. (A shorter
// exp too, the hardware's exp2 with a first-order correction: 1 us less, but an rms error of
// 4.4e-8.)
__device__ __forceinline__ float add_log1p(float x, float z) {  // x + log1p(z), 0 <= z <= 1
#pragma clang fp contract(off)  // ds is the residual of the rounded s
  const float r = __builtin_amdgcn_rcpf(2.f + z), s = z * r, q = s * s;
  const float ds = fmaf(-s, z, fmaf(-2.f, s, z)) * r;  // (z - 2 s is exact)
  float a = 2.f / 15.f;
  a = fmaf(a, q, 2.f / 13.f);
  a = fmaf(a, q, 2.f / 11.f);
  a = fmaf(a, q, 2.f / 9.f);
  a = fmaf(a, q, 2.f / 7.f);
  a = fmaf(a, q, 2.f / 5.f);
  a = fmaf(a, q, 2.f / 3.f);
  const float h = fmaf(-s, z, z);  // z - s z, its rounding error next
  const float low = fmaf(-fmaf(-a * q, r, ds), z, fmaf(-s, z, z - h));
  const float t = x + h, b = t - x;  // and that of x + h (Knuth's two-sum)
  return t + (low + ((x - (t - b)) + (h - b)));
}
// d softplus / dx = 1 / (1 + z) for x >= 0, z / (1 + z) below: the quotient by the reciprocal and one
// residual step against the unrounded 1 + z. Its rms error for x in [-4, -2), [0.5, 1) and [2, 4) is
// 3.50, 2.69 and 1.83e-8; of expf(x) / (expf(x) + 1) 4.78, 3.27 and 2.18e-8; of z times a refined
// reciprocal of the rounded 1 + z 5.13, 3.76 and 3.74e-8, 0.4 us sooner.
__device__ __forceinline__ float softplus_grad(float x, float z) {
#pragma clang fp contract(off)
  const float d = 1.f + z, dl = z - (d - 1.f), r = __builtin_amdgcn_rcpf(d);
  const float m = x >= 0.f ? 1.f : z, q = m * r;
  return fmaf(fmaf(-dl, q, fmaf(-d, q, m)), r, q);
}
__device__ __forceinline__ float softplus_t(float x) {
  return x > 20.f ? x : add_log1p(fmaxf(x, 0.f), expf(-fabsf(x)));
}

constexpr int kDtThreads = 512;
constexpr int kDtRun = 16;  // tokens per thread
template <int HT>
struct DtCfg {
  static constexpr int NS = kDtThreads / HT;     // runs per workgroup
  static constexpr int CT = NS * kDtRun;         // tokens per chunk
};

// A workgroup's chunk and a thread's run: [t0, t0 + n) of head h, run s of the chunk.
template <int HT>
struct DtPos {
  int row, h, s, c, n;
  bool hv;
  int64_t t0, base;  // element of (row, t0, h)
  // of workgroup rb (row, head block) and chunk ci
  __device__ __forceinline__ DtPos(const DtArgs& a, int rb, int ci) {
    const int hb = (a.H + HT - 1) / HT;
    c = ci;
    row = rb / hb;
    h = (rb % hb) * HT + (int)(threadIdx.x % HT);
    s = threadIdx.x / HT;
    hv = h < a.H;
    t0 = (int64_t)c * DtCfg<HT>::CT + s * kDtRun;
    n = !hv || t0 >= a.T ? 0 : (a.T - t0 < kDtRun ? (int)(a.T - t0) : kDtRun);
    base = ((int64_t)row * a.T + t0) * a.H + h;
  }
  __device__ __forceinline__ explicit DtPos(const DtArgs& a)
      : DtPos(a, blockIdx.x / a.nchunk, blockIdx.x % a.nchunk) {}
};

// sum of the values of the runs before s (or after s) at this thread's head
template <int HT, bool AFTER>
__device__ __forceinline__ float dt_other_runs(const float (*part)[HT], int s) {
  float v = 0.f;
  const int col = threadIdx.x % HT;
  if (AFTER) {
    for (int r = DtCfg<HT>::NS - 1; r > s; --r) v += part[r][col];
  } else {
    for (int r = 0; r < s; ++r) v += part[r][col];
  }
  return v;
}

// ---------------------------------------------------------------- forward
// cum_A within the chunk (from zero), e; with one chunk also the decay
template <int HT>
__global__ __launch_bounds__(kDtThreads) void mamba2_dt_scan_kernel(const DtArgs a) {
  __shared__ float part[DtCfg<HT>::NS][HT];
  const DtPos<HT> p(a);
  const float Ah = p.hv ? a.A[p.h] : 0.f;
  const float bh = (p.hv && a.bias) ? a.bias[p.h] : 0.f;
  float c[kDtRun];
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) c[i] = i < p.n ? dt_at(a, p.base + (int64_t)i * a.H) : 0.f;
  float run = 0.f;
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) {
    const float e = a.softplus ? softplus_t(c[i] + bh) : c[i];
    if (a.e_out && i < p.n) a.e_out[p.base + (int64_t)i * a.H] = e;
    run += i < p.n ? Ah * e : 0.f;
    c[i] = run;
  }
  part[p.s][threadIdx.x % HT] = run;
  __syncthreads();
  const float before = dt_other_runs<HT, false>(part, p.s);
#pragma unroll
  for (int i = 0; i < kDtRun; ++i)
    if (i < p.n) a.cum_A[p.base + (int64_t)i * a.H] = before + c[i];
  if (a.nchunk == 1 && p.n > 0 && p.t0 + p.n == a.T)
    a.decay[(int64_t)p.row * a.H + p.h] = expf(before + run);
}

// What the chunks hand on, in place, one value per chunk and head: INCL: x[c] := sum_{c'<=c}
// x[c'] (and the decay of the whole row); else x[c] := first + sum_{c'>c} x[c'] (SUFFIX), or
// -sum_{c'<c} x[c']. 16 waves x 64 heads; wave w folds a sixteenth of the chunks.
enum { kDtInclusive, kDtSuffix, kDtNegPrefix };
template <int KIND>
__global__ __launch_bounds__(1024) void mamba2_dt_chunks_kernel(const DtArgs a, float* x, int CT,
                                                                int at_end) {
  __shared__ float part[16][64];
  const int hb = (a.H + 63) / 64;
  const int row = blockIdx.x / hb, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int h = (blockIdx.x % hb) * 64 + lane;
  const bool hv = h < a.H;
  const int n = a.nchunk;
  const int lo = (int)((int64_t)n * w / 16), hi = (int)((int64_t)n * (w + 1) / 16);
  auto at = [&](int c) -> int64_t {  // the chunk's last (at_end) or first token
    const int64_t first = (int64_t)c * CT, end = first + CT < a.T ? first + CT : a.T;
    return ((int64_t)row * a.T + (at_end ? end - 1 : first)) * a.H + h;
  };
  float s = 0.f;
  if (hv) {
#pragma unroll 8
    for (int c = lo; c < hi; ++c) s += x[at(c)];
  }
  part[w][lane] = s;
  __syncthreads();
  if (!hv) return;
  float run = 0.f;
  if (KIND == kDtSuffix) {
    if (a.g_decay) run = a.g_decay[(int64_t)row * a.H + h] * a.decay[(int64_t)row * a.H + h];
    for (int v = 15; v > w; --v) run += part[v][lane];
#pragma unroll 8
    for (int c = hi - 1; c >= lo; --c) {
      const float v = x[at(c)];
      x[at(c)] = run;
      run += v;
    }
  } else {
    for (int v = 0; v < w; ++v) run += part[v][lane];
#pragma unroll 8
    for (int c = lo; c < hi; ++c) {
      const float v = x[at(c)];
      if (KIND == kDtNegPrefix) x[at(c)] = -run;
      run += v;
      if (KIND == kDtInclusive) x[at(c)] = run;
    }
    if (KIND == kDtInclusive && w == 15) a.decay[(int64_t)row * a.H + h] = expf(run);
  }
}

// chunk c > 0: every token but the last (already final) plus the last token of chunk c - 1
template <int HT>
__global__ __launch_bounds__(kDtThreads) void mamba2_dt_carry_kernel(const DtArgs a) {
  const DtPos<HT> p(a);
  if (p.c == 0 || p.n <= 0) return;
  const int64_t first = (int64_t)p.c * DtCfg<HT>::CT;
  const int64_t end = first + DtCfg<HT>::CT < a.T ? first + DtCfg<HT>::CT : a.T;
  const float in = a.cum_A[((int64_t)p.row * a.T + first - 1) * a.H + p.h];
  const int n = p.t0 + p.n == end ? p.n - 1 : p.n;
  float c[kDtRun];
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) c[i] = i < n ? a.cum_A[p.base + (int64_t)i * a.H] : 0.f;
#pragma unroll
  for (int i = 0; i < kDtRun; ++i)
    if (i < n) a.cum_A[p.base + (int64_t)i * a.H] = in + c[i];
}

// ---------------------------------------------------------------- backward
// g_dt at the chunk's first token := sum of the chunk's g_cum
template <int HT>
__global__ __launch_bounds__(kDtThreads) void mamba2_dt_sums_kernel(const DtArgs a) {
  __shared__ float part[DtCfg<HT>::NS][HT];
  const DtPos<HT> p(a);
  float g[kDtRun];
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) g[i] = i < p.n ? a.g_cum[p.base + (int64_t)i * a.H] : 0.f;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) s += g[i];
  part[p.s][threadIdx.x % HT] = s;
  __syncthreads();
  if (p.s == 0 && p.hv) a.g_dt[p.base] = s + dt_other_runs<HT, true>(part, 0);
}

// G_t = g_cum_t (+ g_decay decay at t = T-1);  R_s = sum_{t>=s} G_t, or (CLOSED: g_cum_{T-1}
// stands for minus the sum of the others) R_s = -sum_{t<s} G_t, summed from the front so that
// the small R of early tokens keep their precision;
// g_e_s = A R_s (+ the direct g_e_s);  g_A += sum_s R_s e_s;  g_dt_s = g_e_s softplus'(dt_s + bias)
// (or g_e_s);  g_bias += sum_s g_dt_s (softplus only).
// One chunk, `in` entering it: g_dt of the thread's run and its parts of g_A and g_bias, added to
// pa and pb.
template <int HT, bool CLOSED>
__device__ __forceinline__ void dt_bwd_chunk(const DtArgs& a, const DtPos<HT>& p, float Ah, float bh,
                                             float in, float (*part)[HT], float& pa, float& pb) {
  float g[kDtRun], x[kDtRun], d[kDtRun];
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) {
    const int64_t at = p.base + (int64_t)i * a.H;
    g[i] = i < p.n && a.g_cum ? a.g_cum[at] : 0.f;
    x[i] = i < p.n ? dt_at(a, at) : 0.f;
    d[i] = i < p.n && a.g_e ? a.g_e[at] : 0.f;
  }
  float run = 0.f;
  if (CLOSED) {
#pragma unroll
    for (int i = 0; i < kDtRun; ++i) {
      const float v = g[i];
      g[i] = run;
      run -= v;
    }
  } else {
#pragma unroll
    for (int i = kDtRun - 1; i >= 0; --i) {
      run += g[i];
      g[i] = run;
    }
  }
  part[p.s][threadIdx.x % HT] = run;
  __syncthreads();  // (also: every thread has read the chunk's first g_dt)
  in += dt_other_runs<HT, !CLOSED>(part, p.s);
#pragma unroll
  for (int i = 0; i < kDtRun; ++i) {
    const float R = in + g[i], y = x[i] + bh;
    const float ge = Ah * R + d[i];
    float e = x[i], gdt = ge;
    if (a.softplus) {
      const float z = expf(-fabsf(y));
      e = y > 20.f ? y : add_log1p(fmaxf(y, 0.f), z);
      gdt = y > 20.f ? ge : ge * softplus_grad(y, z);
    }
    if (i < p.n) {
      pa += R * e;
      pb += gdt;
      a.g_dt[p.base + (int64_t)i * a.H] = gdt;
    }
  }
}

// The runs' sums of g_A and g_bias at this thread's head, valid in run 0.
template <int HT>
__device__ __forceinline__ void dt_runs_total(float (*red)[DtCfg<HT>::NS][HT], int s, float& pa,
                                              float& pb) {
  const int col = threadIdx.x % HT;
  red[0][s][col] = pa;
  red[1][s][col] = pb;
  __syncthreads();
  if (s == 0) {
    pa += dt_other_runs<HT, true>(red[0], 0);
    pb += dt_other_runs<HT, true>(red[1], 0);
  }
}

template <int HT, bool CLOSED>
__global__ __launch_bounds__(kDtThreads) void mamba2_dt_bwd_kernel(const DtArgs a) {
  __shared__ float part[DtCfg<HT>::NS][HT];
  __shared__ float red[2][DtCfg<HT>::NS][HT];
  const DtPos<HT> p(a);
  const float Ah = p.hv ? a.A[p.h] : 0.f;
  const float bh = (p.hv && a.bias) ? a.bias[p.h] : 0.f;
  float in = 0.f;  // what enters the chunk
  if (p.hv) {
    if (a.nchunk > 1 && a.g_cum)
      in = a.g_dt[((int64_t)p.row * a.T + (int64_t)p.c * DtCfg<HT>::CT) * a.H + p.h];
    else if (!CLOSED && a.g_decay)
      in = a.g_decay[(int64_t)p.row * a.H + p.h] * a.decay[(int64_t)p.row * a.H + p.h];
  }
  float pa = 0.f, pb = 0.f;
  dt_bwd_chunk<HT, CLOSED>(a, p, Ah, bh, in, part, pa, pb);
  dt_runs_total<HT>(red, p.s, pa, pb);
  if (p.s != 0 || !p.hv) return;
  const bool gb = a.softplus && a.g_bias;
  if (a.part) {
    const int64_t n = (int64_t)a.rows * a.nchunk, at = ((int64_t)p.row * a.nchunk + p.c) * a.H + p.h;
    a.part[at] = pa;
    if (gb) a.part[n * a.H + at] = pb;
  } else {
    atomicAdd(a.g_A + p.h, pa);
    if (gb) atomicAdd(a.g_bias + p.h, pb);
  }
}

// One workgroup walks all chunks of a row, so that each head's dA and d(bias) are one sum.
template <int HT, bool CLOSED>
__global__ __launch_bounds__(kDtThreads) void mamba2_dt_bwd_serial_kernel(const DtArgs a) {
  __shared__ float part[DtCfg<HT>::NS][HT];
  __shared__ float red[2][DtCfg<HT>::NS][HT];
  const DtPos<HT> p0(a, blockIdx.x, 0);
  const float Ah = p0.hv ? a.A[p0.h] : 0.f;
  const float bh = (p0.hv && a.bias) ? a.bias[p0.h] : 0.f;
  float in = 0.f;
  if (!CLOSED && p0.hv && a.g_decay)
    in = a.g_decay[(int64_t)p0.row * a.H + p0.h] * a.decay[(int64_t)p0.row * a.H + p0.h];
  float pa = 0.f, pb = 0.f;
  for (int i = 0; i < a.nchunk; ++i) {
    const DtPos<HT> p(a, blockIdx.x, CLOSED ? i : a.nchunk - 1 - i);
    dt_bwd_chunk<HT, CLOSED>(a, p, Ah, bh, in, part, pa, pb);
    in += part[0][threadIdx.x % HT] + dt_other_runs<HT, true>(part, 0);
    __syncthreads();  // the next chunk writes part
  }
  dt_runs_total<HT>(red, p0.s, pa, pb);
  if (p0.s != 0 || !p0.hv) return;
  atomicAdd(a.g_A + p0.h, pa);
  if (a.softplus && a.g_bias) atomicAdd(a.g_bias + p0.h, pb);
}

// dA (blockIdx.y 0) and d(bias) (1) += the chunks' parts, in a fixed order, so that a call
// repeats bit for bit: added by atomics, chunks arrive in any order. 16 heads by 64 shares of the
// parts per workgroup. 512 parts of 64 heads: 4 us, and the chunk kernel, without the atomics
// of 512 workgroups on 128 words, 24 us instead of 29.
__global__ __launch_bounds__(1024) void mamba2_dt_fold_kernel(const DtArgs a) {
  __shared__ float sum[64][16];
  const int col = threadIdx.x % 16, share = threadIdx.x / 16;
  const int h = blockIdx.x * 16 + col;
  const int64_t n = (int64_t)a.rows * a.nchunk;
  const float* x = a.part + blockIdx.y * n * a.H + h;
  float v = 0.f;
  if (h < a.H) {
    const int64_t hi = n * (share + 1) / 64;
#pragma unroll 8
    for (int64_t i = n * share / 64; i < hi; ++i) v += x[i * a.H];
  }
  sum[share][col] = v;
  __syncthreads();
  if (share < 8) {
    v = 0.f;
    for (int i = 0; i < 8; ++i) v += sum[8 * share + i][col];
  }
  __syncthreads();
  if (share < 8) sum[share][col] = v;
  __syncthreads();
  if (share || h >= a.H) return;
  for (int i = 1; i < 8; ++i) v += sum[i][col];
  atomicAdd((blockIdx.y ? a.g_bias : a.g_A) + h, v);
}

// ---------------------------------------------------------------- launchers
template <int HT>
static int dt_grid(DtArgs& a) {
  a.nchunk = (int)(((int64_t)a.T + DtCfg<HT>::CT - 1) / DtCfg<HT>::CT);
  return (int)((int64_t)a.rows * ((a.H + HT - 1) / HT) * a.nchunk);
}

template <int HT>
static void launch_dt_fwd(DtArgs a, hipStream_t stream) {
  const unsigned grid = (unsigned)dt_grid<HT>(a), rows = (unsigned)(a.rows * ((a.H + 63) / 64));
  hipLaunchKernelGGL((mamba2_dt_scan_kernel<HT>), dim3(grid), dim3(kDtThreads), 0, stream, a);
  if (a.nchunk == 1) return;
  hipLaunchKernelGGL((mamba2_dt_chunks_kernel<kDtInclusive>), dim3(rows), dim3(1024), 0, stream, a,
                     a.cum_A, DtCfg<HT>::CT, 1);
  hipLaunchKernelGGL((mamba2_dt_carry_kernel<HT>), dim3(grid), dim3(kDtThreads), 0, stream, a);
}

// Heads per workgroup: the least that covers H.
static int dt_heads(int H) { return H <= 8 ? 8 : H <= 16 ? 16 : H <= 32 ? 32 : 64; }

size_t mamba2_dt_bwd_workspace(int rows, int T, int H) {
  const int64_t CT = kDtThreads / dt_heads(H) * kDtRun, nchunk = ((int64_t)T + CT - 1) / CT;
  return nchunk > 1 ? (size_t)rows * nchunk * H * 8 : 0;
}

template <int HT, bool CLOSED>
static void launch_dt_bwd(DtArgs a, hipStream_t stream) {
  const unsigned grid = (unsigned)dt_grid<HT>(a), rows = (unsigned)(a.rows * ((a.H + 63) / 64));
  // Without a workspace the chunks' parts are added by atomics. One or two rows go chunk by
  // chunk instead: with one sum per row and head they repeat bit for bit (two sums added to zero
  // commute). 1 x 8192 x 64: 608 us (one workgroup),
  // with the workspace 18.
  if (a.nchunk > 1 && !a.part && a.rows <= 2) {
    hipLaunchKernelGGL((mamba2_dt_bwd_serial_kernel<HT, CLOSED>), dim3(grid / a.nchunk),
                       dim3(kDtThreads), 0, stream, a);
    return;
  }
  if (a.nchunk > 1 && a.g_cum) {
    hipLaunchKernelGGL((mamba2_dt_sums_kernel<HT>), dim3(grid), dim3(kDtThreads), 0, stream, a);
    hipLaunchKernelGGL((mamba2_dt_chunks_kernel<CLOSED ? kDtNegPrefix : kDtSuffix>), dim3(rows),
                       dim3(1024), 0, stream, a, a.g_dt, DtCfg<HT>::CT, 0);
  }
  hipLaunchKernelGGL((mamba2_dt_bwd_kernel<HT, CLOSED>), dim3(grid), dim3(kDtThreads), 0, stream, a);
  if (a.part)
    hipLaunchKernelGGL(mamba2_dt_fold_kernel, dim3((a.H + 15) / 16, a.softplus && a.g_bias ? 2 : 1),
                       dim3(1024), 0, stream, a);
}

template <class F>
static void by_heads(int H, F f) {
  switch (dt_heads(H)) {
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    case 32: f(std::integral_constant<int, 32>{}); break;
    default: f(std::integral_constant<int, 64>{});
  }
}

hipError_t launch_mamba2_dt_cumsum(const void* dt, int dt_f32, const float* bias, const float* A,
                                   int softplus, float* cum_A, float* e, float* decay, int rows,
                                   int T, int H, hipStream_t stream) {
  const DtArgs a{dt, dt_f32, bias, A, softplus, cum_A, e, nullptr, decay, nullptr, nullptr, nullptr,
                 nullptr, nullptr, nullptr, rows, T, H, 0};
  if ((int64_t)rows * T * H == 0) return hipSuccess;
  by_heads(H, [&](auto ht) { launch_dt_fwd<ht.value>(a, stream); });
  return hipGetLastError();
}

hipError_t launch_mamba2_dt_cumsum_bwd(const void* dt, int dt_f32, const float* bias,
                                       const float* A, int softplus, const float* g_cum,
                                       const float* g_e, const float* g_decay, const float* decay,
                                       float* g_dt, float* g_A, float* g_bias, int rows, int T,
                                       int H, int closed, void* ws, hipStream_t stream) {
  const DtArgs a{dt, dt_f32, bias, A, softplus, nullptr, nullptr, g_e, const_cast<float*>(decay),
                 g_cum, g_decay, g_dt, g_A, g_bias, static_cast<float*>(ws), rows, T, H, 0};
  if ((int64_t)rows * T * H == 0) return hipSuccess;
  by_heads(H, [&](auto ht) {
    if (closed)
      launch_dt_bwd<ht.value, true>(a, stream);
    else
      launch_dt_bwd<ht.value, false>(a, stream);
  });
  return hipGetLastError();
}

}  // namespace rmx
