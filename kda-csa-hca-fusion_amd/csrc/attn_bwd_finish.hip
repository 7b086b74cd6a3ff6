// The last stage of the attention and indexer backwards for gfx950: the sums
// of the key passes' partials, the L2-norm backwards of the compressed and the
// window rows, and the backward of the softmax-gated compression
// (ops_csa.py:198-305, ops_hca.py:132-141), reading the compression's inputs
// and writing their gradients in their own storage type and row stride.
//
// Per block: dk = sum of the chunks' partials; dr = (dk - y (y.dk)) / |raw|
// (y the normalised row); with w = softmax over the block's tokens (per
// channel) of Z + B: dC_j = w_j dr, dZ_j = w_j (C_j - r) dr, dB_j += dZ_j.
// Per token with a window: dx = (dk - y (y.dk)) / |x|, added to dC or written
// to dlocal.
//
// bwd_block_kernel  a group of HD / 8 lanes per block (8 channels a lane) walks
//   the block's tokens, both branches of the overlapped form included: short
//   blocks (CSA, the indexer's keys).
// bwd_rows_kernel   one workgroup per block and token range: the lane groups
//   take tokens (and chunks) in turn, the block's maximum, sum and dk meet in
//   LDS: long blocks (HCA).
// sum_rows_kernel   column sums of the per-block dB terms (and of the sink's).
//
// Bound: HBM (each input read once or from L2, each gradient written once).
// The rows of a block were taken by one workgroup with a thread per channel
// and a serial loop over 128 tokens: 152 us at B2 T8192, m' = 128, c = 128
// (128 workgroups), with about 20 small kernels around it (fp32 copies of the
// inputs, zero fills, adds and conversions of the outputs, library sums); now
// 23 us and three launches of sum_rows_kernel (5 us each).

#include "attn_common.h"
#include "kch_csa.h"
#include "kch_kernels.h"

namespace kch {

namespace {

constexpr float kEps = 1e-12f;

template <typename O>
__device__ __forceinline__ void store8(O* p, const float (&v)[8]) {
  if constexpr (sizeof(O) == 4) {
    reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
  } else {
    typedef O o8 __attribute__((ext_vector_type(8)));
    o8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (O)v[i];
    *reinterpret_cast<o8*>(p) = r;
  }
}

// sum over the aligned group of LPR lanes (8 or 16); every lane gets it
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int m = LPR / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

__device__ __forceinline__ void add8(const float* p, float (&v)[8]) {
  float x[8];
  Load8<float>::run(p, x);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] += x[i];
}

// dr (8 channels) of a compressed row from dk, its normalised and raw rows
template <int LPR>
__device__ __forceinline__ void row_norm_bwd(const float* y, const float* raw, int normalize, const float (&dk)[8],
                                             float (&r)[8], float (&dr)[8]) {
  float yv[8];
  Load8<float>::run(y, yv);
  Load8<float>::run(raw, r);
  float yd = 0.f, rr = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    yd += yv[i] * dk[i];
    rr += r[i] * r[i];
  }
  yd = group_sum<LPR>(yd);
  const float nrm = sqrtf(group_sum<LPR>(rr));
#pragma unroll
  for (int i = 0; i < 8; ++i)
    dr[i] = !normalize ? dk[i] : (nrm > kEps ? (dk[i] - yv[i] * yd) / nrm : dk[i] / kEps);
}

// The window row's gradient of token ti (all lanes of its group), 8 channels.
template <int HD, typename T>
__device__ __forceinline__ void window_bwd(const BwdFinish& p, size_t ti, int lc, float (&dx)[8]) {
  float x[8], dk[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) dk[i] = 0.f;
  for (int ci = 0; ci < p.win_nc; ++ci) add8(p.part_w + ((size_t)ci * p.B * p.T + ti) * HD + 8 * lc, dk);
  Load8<T>::run(static_cast<const T*>(p.lsrc) + ti * p.ldl + 8 * lc, x);
  const float rl = p.rl[ti];
  float yd = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] *= rl;
    yd += x[i] * dk[i];
  }
  yd = group_sum<HD / 8>(yd);
  const bool big = rl < 1e12f;  // rl = 1 / max(|x|, eps): for |x| <= eps the norm is the constant eps
#pragma unroll
  for (int i = 0; i < 8; ++i) dx[i] = (big ? dk[i] - x[i] * yd : dk[i]) * rl;
}

// token (b, j)'s dC, dZ and dB terms of one branch; dx added to dC when given
template <int HD, typename T, typename O>
__device__ __forceinline__ void token_bwd(const T* C, const float (&lg)[8], const float (&mx)[8],
                                          const float (&den)[8], const float (&r)[8], const float (&dr)[8],
                                          const float* dx, O* dC, O* dZ, float* dB) {
  float c[8], oc[8], oz[8];
  Load8<T>::run(C, c);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float w = expf(lg[i] - mx[i]) / den[i];
    oz[i] = w * (c[i] - r[i]) * dr[i];
    oc[i] = w * dr[i] + (dx ? dx[i] : 0.f);
  }
  store8<O>(dC, oc);
  store8<O>(dZ, oz);
  if (dB) store8<float>(dB, oz);
}

template <int HD, typename T>
__device__ __forceinline__ void logits8(const T* z, const float* bp, float (&lg)[8]) {
  float b[8];
  Load8<T>::run(z, lg);
  Load8<float>::run(bp, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) lg[i] += b[i];
}

template <int HD, typename T, typename O, bool OVL>
__global__ __launch_bounds__(128) void bwd_block_kernel(BwdFinish p) {
  constexpr int LPR = HD / 8, RG = 128 / LPR;
  const int lc = threadIdx.x % LPR;
  const long long g = (long long)blockIdx.x * RG + threadIdx.x / LPR, ng = (long long)p.B * p.nb;
  const bool live = g < ng;  // (no early return: the group sums shuffle)
  const int b = live ? (int)(g / p.nb) : 0, n = live ? (int)(g - (long long)b * p.nb) : 0;
  const int m = p.m;
  float dk[8], r[8], dr[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) dk[i] = 0.f;
  // the chunks from the first one that holds a query seeing block n
  const float* part = p.part_b + ((size_t)b * p.nchunk * p.nb + n) * HD + 8 * lc;
#pragma unroll 8
  for (int ci = ((n + 1) * m - 1) / p.part_qc; ci < p.nchunk; ++ci) add8(part + (size_t)ci * p.nb * HD, dk);
  const size_t ri = ((size_t)b * p.nb + n) * HD + 8 * lc;
  row_norm_bwd<LPR>(p.kc + ri, p.raw + ri, p.normalize, dk, r, dr);

  const T* C = static_cast<const T*>(p.C);
  const T* Z = static_cast<const T*>(p.Z);
  const T* Cb = static_cast<const T*>(p.Cb);
  const T* Zb = static_cast<const T*>(p.Zb);
  const size_t t0 = (size_t)b * p.T + (size_t)n * m;  // the block's first token; the second branch: t0 - m
  const bool two = OVL && n > 0;
  float mx[8], den[8], lg[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    mx[i] = -INFINITY;
    den[i] = 0.f;
  }
#pragma unroll 4
  for (int j = 0; j < m; ++j) {
    logits8<HD, T>(Z + (t0 + j) * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
#pragma unroll
    for (int i = 0; i < 8; ++i) mx[i] = fmaxf(mx[i], lg[i]);
  }
  if (two) {
#pragma unroll 4
    for (int j = 0; j < m; ++j) {
      logits8<HD, T>(Zb + (t0 - m + j) * p.ldZb + 8 * lc, p.Bb + j * HD + 8 * lc, lg);
#pragma unroll
      for (int i = 0; i < 8; ++i) mx[i] = fmaxf(mx[i], lg[i]);
    }
  }
#pragma unroll 4
  for (int j = 0; j < m; ++j) {
    logits8<HD, T>(Z + (t0 + j) * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
#pragma unroll
    for (int i = 0; i < 8; ++i) den[i] += expf(lg[i] - mx[i]);
  }
  if (two) {
#pragma unroll 4
    for (int j = 0; j < m; ++j) {
      logits8<HD, T>(Zb + (t0 - m + j) * p.ldZb + 8 * lc, p.Bb + j * HD + 8 * lc, lg);
#pragma unroll
      for (int i = 0; i < 8; ++i) den[i] += expf(lg[i] - mx[i]);
    }
  }
#pragma unroll 2
  for (int j = 0; j < m; ++j) {
    const size_t ti = t0 + j, o = ti * HD + 8 * lc;
    float dx[8];
    if (p.win > 0) window_bwd<HD, T>(p, ti, lc, dx);
    if (live) {
      logits8<HD, T>(Z + ti * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
      token_bwd<HD, T, O>(C + ti * p.ldC + 8 * lc, lg, mx, den, r, dr, p.win > 0 && !p.dlocal ? dx : nullptr,
                          static_cast<O*>(p.dC) + o, static_cast<O*>(p.dZ) + o, p.dBp + ((size_t)g * m + j) * HD + 8 * lc);
      if (p.dlocal && p.win > 0) store8<O>(static_cast<O*>(p.dlocal) + o, dx);
    }
  }
  if constexpr (OVL) {
    if (!live) return;
    for (int j = 0; j < m; ++j) {
      float* db = p.dBbp + ((size_t)g * m + j) * HD + 8 * lc;
      const float zero[8] = {};
      if (two) {
        const size_t ti = t0 - m + j, o = ti * HD + 8 * lc;
        logits8<HD, T>(Zb + ti * p.ldZb + 8 * lc, p.Bb + j * HD + 8 * lc, lg);
        token_bwd<HD, T, O>(Cb + ti * p.ldCb + 8 * lc, lg, mx, den, r, dr, nullptr, static_cast<O*>(p.dCb) + o,
                            static_cast<O*>(p.dZb) + o, db);
      } else {
        store8<float>(db, zero);
      }
      if (n == p.nb - 1) {  // the last block's second branch feeds no block
        const size_t o = (t0 + j) * HD + 8 * lc;
        store8<O>(static_cast<O*>(p.dCb) + o, zero);
        store8<O>(static_cast<O*>(p.dZb) + o, zero);
      }
    }
  }
}

template <int HD, typename T, typename O>
__global__ __launch_bounds__(256) void bwd_rows_kernel(BwdFinish p, int split) {
  constexpr int LPR = HD / 8, RG = 256 / LPR;
  __shared__ __attribute__((aligned(16))) float red[RG][HD], tot[HD];
  const int tid = threadIdx.x, lc = tid % LPR, rg = tid / LPR;
  const int part_of = blockIdx.x % split, n = (blockIdx.x / split) % p.nb, b = blockIdx.x / split / p.nb;
  const int m = p.m;
  // v of every lane group combined over the groups, back to the 8 channels of each lane
  auto combine = [&](float (&v)[8], bool is_max) {
    store8<float>(&red[rg][8 * lc], v);
    __syncthreads();
    if (tid < HD) {
      float s = red[0][tid];
#pragma unroll
      for (int i = 1; i < RG; ++i) s = is_max ? fmaxf(s, red[i][tid]) : s + red[i][tid];
      tot[tid] = s;
    }
    __syncthreads();
    Load8<float>::run(&tot[8 * lc], v);
  };
  float dk[8], r[8], dr[8], mx[8], den[8], lg[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    dk[i] = den[i] = 0.f;
    mx[i] = -INFINITY;
  }
  const float* part = p.part_b + ((size_t)b * p.nchunk * p.nb + n) * HD + 8 * lc;
#pragma unroll 4
  for (int ci = ((n + 1) * m - 1) / p.part_qc + rg; ci < p.nchunk; ci += RG) add8(part + (size_t)ci * p.nb * HD, dk);
  combine(dk, false);
  const size_t ri = ((size_t)b * p.nb + n) * HD + 8 * lc;
  row_norm_bwd<LPR>(p.kc + ri, p.raw + ri, p.normalize, dk, r, dr);
  const T* C = static_cast<const T*>(p.C);
  const T* Z = static_cast<const T*>(p.Z);
  const size_t t0 = (size_t)b * p.T + (size_t)n * m;
#pragma unroll 4
  for (int j = rg; j < m; j += RG) {
    logits8<HD, T>(Z + (t0 + j) * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
#pragma unroll
    for (int i = 0; i < 8; ++i) mx[i] = fmaxf(mx[i], lg[i]);
  }
  combine(mx, true);
#pragma unroll 4
  for (int j = rg; j < m; j += RG) {
    logits8<HD, T>(Z + (t0 + j) * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
#pragma unroll
    for (int i = 0; i < 8; ++i) den[i] += expf(lg[i] - mx[i]);
  }
  combine(den, false);
  // this workgroup's tokens (whole lane groups, so that the group sums see all their lanes)
  const int per = (m + split - 1) / split, lo = part_of * per, hi = min(m, lo + per);
  for (int j = lo + rg; j < hi; j += RG) {
    const size_t ti = t0 + j, o = ti * HD + 8 * lc;
    float dx[8];
    if (p.win > 0) window_bwd<HD, T>(p, ti, lc, dx);
    logits8<HD, T>(Z + ti * p.ldZ + 8 * lc, p.Bpos + j * HD + 8 * lc, lg);
    token_bwd<HD, T, O>(C + ti * p.ldC + 8 * lc, lg, mx, den, r, dr, p.win > 0 && !p.dlocal ? dx : nullptr,
                        static_cast<O*>(p.dC) + o, static_cast<O*>(p.dZ) + o,
                        p.dBp + (((size_t)b * p.nb + n) * m + j) * HD + 8 * lc);
    if (p.dlocal && p.win > 0) store8<O>(static_cast<O*>(p.dlocal) + o, dx);
  }
}

// out[s, c] = sign * sum of x[r, c] over the rows r of slice s (blockIdx.y of
// gridDim.y), 16 columns a workgroup, 64 rows at a time
__global__ __launch_bounds__(256) void sum_rows_kernel(const float* x, float* out, long long rows, int cols,
                                                       float sign) {
  __shared__ float red[64][17];
  const int c = threadIdx.x % 4, rl = threadIdx.x / 4;
  const int c0 = blockIdx.x * 16 + 4 * c;
  const long long per = (rows + gridDim.y - 1) / gridDim.y, r0 = per * blockIdx.y;
  const long long r1 = min(rows, r0 + per);
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if ((cols & 3) == 0 && c0 < cols) {
#pragma unroll 4
    for (long long r = r0 + rl; r < r1; r += 64) {
      const float4 v = *reinterpret_cast<const float4*>(x + r * cols + c0);
      s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
    }
  } else {
    for (long long r = r0 + rl; r < r1; r += 64)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c0 + e < cols) s[e] += x[r * cols + c0 + e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[rl][4 * c + e] = s[e];
  __syncthreads();
  if (threadIdx.x < 16 && blockIdx.x * 16 + threadIdx.x < cols) {
    float t = 0.f;
#pragma unroll 8
    for (int i = 0; i < 64; ++i) t += red[i][threadIdx.x];
    out[(size_t)blockIdx.y * cols + blockIdx.x * 16 + threadIdx.x] = sign * t;
  }
}

// row slices of the column sums: enough workgroups to fill the chip, at least 128 rows each
int sum_slices(long long rows, int cols) {
  const long long wg = (cols + 15) / 16;
  long long s = (512 + wg - 1) / wg;
  if (s > rows / 128) s = rows / 128;
  return s < 1 ? 1 : (int)s;
}

template <int HD, typename T, typename O>
void launch_finish(const BwdFinish& p, hipStream_t s) {
  constexpr int RG = 128 / (HD / 8);
  const long long ng = (long long)p.B * p.nb;
  if (!p.Cb && p.m >= 32) {
    // long blocks: up to four workgroups a block while the grid is small
    int split = 1;
    while (split < 4 && ng * split < 512) split *= 2;
    hipLaunchKernelGGL((bwd_rows_kernel<HD, T, O>), dim3((unsigned)(ng * split)), dim3(256), 0, s, p, split);
    return;
  }
  const dim3 g((unsigned)((ng + RG - 1) / RG));
  if (p.Cb)
    hipLaunchKernelGGL((bwd_block_kernel<HD, T, O, true>), g, dim3(128), 0, s, p);
  else
    hipLaunchKernelGGL((bwd_block_kernel<HD, T, O, false>), g, dim3(128), 0, s, p);
}

template <int HD>
hipError_t finish_types(const BwdFinish& p, hipStream_t s) {
  if (p.odt != DT_F32 && p.odt != p.cdt) return hipErrorInvalidValue;
  if (p.cdt == DT_F32)
    launch_finish<HD, float, float>(p, s);
  else if (p.cdt == DT_BF16)
    p.odt == DT_BF16 ? launch_finish<HD, bf16_t, bf16_t>(p, s) : launch_finish<HD, bf16_t, float>(p, s);
  else
    p.odt == DT_F16 ? launch_finish<HD, _Float16, _Float16>(p, s) : launch_finish<HD, _Float16, float>(p, s);
  return hipGetLastError();
}

size_t al256f(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

hipError_t bwd_finish_launch(const BwdFinish& p, int HD, hipStream_t s) {
  if ((long long)p.B * p.nb == 0) return hipSuccess;
  return HD == 64 ? finish_types<64>(p, s) : finish_types<128>(p, s);
}

size_t sum_rows_ws_bytes(long long rows, int cols) {
  const int s = sum_slices(rows, cols);
  return s > 1 ? al256f((size_t)s * cols * 4) : 0;
}

hipError_t sum_rows_launch(const float* x, float* out, long long rows, int cols, float sign, void* ws, hipStream_t s) {
  const int sl = sum_slices(rows, cols);
  const dim3 g((cols + 15) / 16, sl);
  hipLaunchKernelGGL(sum_rows_kernel, g, dim3(256), 0, s, x, sl > 1 ? static_cast<float*>(ws) : out, rows, cols,
                     sl > 1 ? 1.f : sign);
  if (sl > 1)
    hipLaunchKernelGGL(sum_rows_kernel, dim3((cols + 15) / 16, 1), dim3(256), 0, s, static_cast<const float*>(ws), out,
                       (long long)sl, cols, sign);
  return hipGetLastError();
}

}  // namespace kch
