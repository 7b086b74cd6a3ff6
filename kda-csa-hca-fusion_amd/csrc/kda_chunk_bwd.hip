// KDA chunked backward for gfx950: the gradients of naive_chunk_kda
// (/root/reference/ops_kda.py:340-536, which the reference differentiates with
// autograd; its tests pin them to the recurrent ones, run_correctness.py:
// 1032-1092) in the chunk form, for bf16 / fp16 / fp32 inputs, K and V in
// {64, 128}, chunks of 64 tokens. Arithmetic is fp32; every matrix product
// is an MFMA product of two-part bf16 splits (x = hi + lo; hi*hi + hi*lo +
// lo*hi, about 2^-16 relative per product).
//
// Per chunk (q^ = scale q, G = in-chunk cumsum of the clamped gate, natural
// log units, G_l = G at the chunk's last token):
//   M[i][j]   = beta_i sum_ch k_i k_j e^(G_i - G_j)     (j < i)
//   Aqk[i][j] = sum_ch q^_i k_j e^(G_i - G_j)           (j <= i)
//   X = (I + M)^-1,   Bk = beta k e^G,   Bv = beta v
//   W = X Bk,   U = X Bv,   Qg = q^ e^G,   Kd = k e^(G_l - G),   el = e^(G_l)
//   v_n = U - W S_n;   o = Qg S_n + Aqk v_n;   S_n+1 = el S_n + Kd^T v_n
// with the exponents of M and Aqk clamped at 50 (ops_kda.py:414,516).
// Backward, dS' = dL/dS_n+1:
//   dv_n = Aqk^T dO + Kd dS'          dS_n = Qg^T dO + el dS' - W^T dv_n
//   dBv  = X^T dv_n                   (dU = dv_n)
//   dBk  = -dBv S_n^T                 (= X^T dW with dW = -dv_n S_n^T)
//   dM   = -dBv v_n^T, strictly lower (= -X^T dX X^T: dX = dv_n v_n^T (I + M)^T
//                                      because (I + M) v_n = Bv - Bk S_n)
//   dAqk = dO v_n^T (j <= i),  dQg = dO S_n^T,  dKd = v_n dS'^T,
//   del  = rowsum(S_n * dS')
// then the elementwise chains back to q, k, v, g and beta; dg is the in-chunk
// suffix sum of dG plus the gradient of G_l.
//
// Kernels (one launch each):
//   cb_prep_kernel  per (b, hv, chunk): M, Aqk, X, W, U, Qg, Kd, el -> workspace
//   cb_fwd_kernel   per (b, hv, slice of V), chunks in order: S_n, v_n
//   cb_bwd_kernel   per (b, hv, slice of V), chunks in reverse: dS', dv_n, dS_0
//   cb_grad_kernel  per (b, hv, chunk): dq, dk, dv, dg, dbeta (or per-value-head
//                   partials that kda_bwd_reduce_launch sums when HV > H)
// Every operand that passes from one kernel to the next is split once, where
// it is made, and lies in the workspace in the order the matrix instruction
// reads it (Rec): a consumer's fragment is two 16-byte loads a lane, whole
// 1 KB tiles, with no conversion, transpose or LDS staging. The states S_n and
// dS' alone stay fp32, in the same order (del multiplies them; a wave of
// cb_grad_kernel splits each once, for its products). Between the two products
// of a state kernel's chunk the state and v_n (dv_n) pass through LDS as split
// planes; the transposed fragments that cb_grad_kernel reads are taken from the
// planes by transposing reads, those of the states from a transpose in LDS.
// The decay-weighted products (M, Aqk and their gradients) factor as
// e^(G_i - G_a) e^(G_a - G_j) around token a = 31 and run on MFMA when every
// gate of the chunk (channel tile) is <= 0 and every |G - G_a| <= 60 nats:
// the factors then stay in fp32 range with normal low parts, and no exponent
// reaches the clamp. Otherwise they are formed exactly, one exponential per
// (i, j, channel), with the clamp and its zero gradient.

#include <atomic>
#include <type_traits>

#include "kch_device.h"
#include "kch_kernels.h"

namespace kch {

namespace {

constexpr int C = 64;
constexpr int kAnc = 31;
constexpr float kLn2Inv = 1.4426950408889634f;
constexpr float kCap = 50.f;
constexpr float kAncRange = 60.f;

__device__ __forceinline__ float ex(float x) { return __builtin_amdgcn_exp2f(x * kLn2Inv); }

struct Sp {
  bf16x8 hi, lo;
};

__device__ __forceinline__ Sp sp8(const float* f) {
  Sp s;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bf16_t h = (bf16_t)f[i];
    s.hi[i] = h;
    s.lo[i] = (bf16_t)(f[i] - (float)h);
  }
  return s;
}

__device__ __forceinline__ f32x4 mm3(const Sp& a, const Sp& b, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, acc, 0, 0, 0);
}

// Buffer addressing: a scalar base, one 32-bit byte offset per lane and a
// constant, so no 64-bit address lives in vector registers; an offset at or
// past `bytes` reads zero and stores nothing, which is how rows past the end
// of a sequence drop out.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(unsigned)bytes, 0x00020000);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// N consecutive values of InT as dwords
template <typename InT, int N>
__device__ __forceinline__ auto buf_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  if constexpr (N * sizeof(InT) == 32) {
    const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, 0);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  } else if constexpr (N * sizeof(InT) == 16) {
    const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return a;
  } else {
    static_assert(N * sizeof(InT) == 8, "dwords");
    const u32x2 a = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    return a;
  }
}

// a b with b of NP exact parts (1: b.lo is zero)
template <int NP>
__device__ __forceinline__ f32x4 mmp(const Sp& a, const Sp& b, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, acc, 0, 0, 0);
  if constexpr (NP == 2) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, acc, 0, 0, 0);
}

// parts of an input value: bf16 is one part exactly
template <typename T> constexpr int kParts = std::is_same<T, bf16_t>::value ? 1 : 2;

struct Sp4 {
  bf16x4 hi, lo;
};

__device__ __forceinline__ Sp4 sp4(f32x4 f) {
  Sp4 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bf16_t h = (bf16_t)f[i];
    s.hi[i] = h;
    s.lo[i] = (bf16_t)(f[i] - (float)h);
  }
  return s;
}

// Fragment tiles: a matrix of R rows and D contraction columns as tiles of
// 16 x 32, tile (r / 16) * (D / 32) + d / 32; in a tile lane r % 16 + 16 (d %
// 32 / 8) holds columns d .. d + 7 of its row, the high parts of all lanes
// before the low parts (1024 bf16 a tile).
constexpr int kTile = 1024;

__device__ __forceinline__ Sp ft_load(const bf16_t* m, int tile) {
  const bf16_t* p = m + (size_t)tile * kTile + 8 * (threadIdx.x & 63);
  return {*reinterpret_cast<const bf16x8*>(p), *reinterpret_cast<const bf16x8*>(p + 512)};
}

__device__ __forceinline__ Sp ft_load(__amdgpu_buffer_rsrc_t m, int off, int tile) {
  const int v = 16 * (threadIdx.x & 63), so = 2 * (off + tile * kTile);
  return {__builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(m, v, so, 0)),
          __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(m, v + 1024, so, 0))};
}

__device__ __forceinline__ void ft_store(bf16_t* m, int tile, int lane, const Sp& s) {
  bf16_t* p = m + (size_t)tile * kTile + 8 * lane;
  *reinterpret_cast<bf16x8*>(p) = s.hi;
  *reinterpret_cast<bf16x8*>(p + 512) = s.lo;
}

// The same tiles in fp32 (as many bytes): columns d .. d + 3 of all lanes before
// d + 4 .. d + 7.
struct F8 {
  f32x4 a, b;
};

__device__ __forceinline__ F8 ft_load_f32(__amdgpu_buffer_rsrc_t m, int off, int tile) {
  const int v = 16 * (threadIdx.x & 63), so = 2 * (off + tile * kTile);
  return {__builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(m, v, so, 0)),
          __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(m, v + 1024, so, 0))};
}

__device__ __forceinline__ void ft_store_f32(bf16_t* m, int tile, int lane, f32x4 a, f32x4 b) {
  float* p = reinterpret_cast<float*>(m + (size_t)tile * kTile) + 4 * lane;
  *reinterpret_cast<f32x4*>(p) = a;
  *reinterpret_cast<f32x4*>(p + 256) = b;
}

// Accumulator rows 16 tc + 4 kq + e, column r16 into a matrix whose rows are
// the accumulator's columns (row tile tr) and whose contraction columns (nk
// tiles of 32) are the accumulator's rows.
__device__ __forceinline__ void ft_store_acc(bf16_t* m, int tr, int nk, int tc, const Sp4& s) {
  const int l = threadIdx.x & 63, r16 = l & 15, kq = l >> 4;
  bf16_t* p = m + (size_t)(tr * nk + (tc >> 1)) * kTile + 8 * (r16 + 16 * (2 * (tc & 1) + (kq >> 1))) +
              4 * (kq & 1);
  *reinterpret_cast<bf16x4*>(p) = s.hi;
  *reinterpret_cast<bf16x4*>(p + 512) = s.lo;
}

// 4 rows (this lane: r0 .. r0 + 3, r0 by lane / 16) of column col0 + lane % 16
// of an LDS plane of row stride ld
__device__ __forceinline__ bf16x4 tr4(const bf16_t* plane, int ld, int r0, int col0) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  const int n = threadIdx.x & 15;
  return __builtin_bit_cast(
      bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(
                  plane + (r0 + (n >> 2)) * ld + col0 + 4 * (n & 3))));
}

__device__ __forceinline__ bf16x8 cat4(bf16x4 a, bf16x4 b) {
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// rows r0 + 8 kq .. + 7 of column col0 + lane % 16
__device__ __forceinline__ bf16x8 tr8(const bf16_t* plane, int ld, int r0, int col0) {
  const int r = r0 + 8 * ((threadIdx.x & 63) >> 4);
  return cat4(tr4(plane, ld, r, col0), tr4(plane, ld, r + 4, col0));
}

__device__ __forceinline__ Sp plane8(const bf16_t* hi, const bf16_t* lo, int off) {
  return {*reinterpret_cast<const bf16x8*>(hi + off), *reinterpret_cast<const bf16x8*>(lo + off)};
}

// the wave's index, known to be uniform
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// 8 consecutive fp32 values (16-byte aligned)
__device__ __forceinline__ void ld8c(const float* p, float* f) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
  f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

// 8 fp32 values ld apart
__device__ __forceinline__ void ld8s(const float* p, int ld, float* f) {
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = p[i * ld];
}

// 8 consecutive input values (16-byte aligned), as fp32
template <typename T>
__device__ __forceinline__ void ld8g(const T* p, float* f) {
  if constexpr (sizeof(T) == 4) {
    ld8c(reinterpret_cast<const float*>(p), f);
  } else {
    const uint4 r = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 x = Pair<T>::cvt(w[i]);
      f[2 * i] = x.x;
      f[2 * i + 1] = x.y;
    }
  }
}

__device__ __forceinline__ void zero8(float* f) {
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = 0.f;
}

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// sum over the 16 lanes of a DPP row (every lane receives it)
__device__ __forceinline__ float row16_sum(float v) {
  v += dppf<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dppf<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dppf<0x141>(v);  // row_half_mirror
  v += dppf<0x140>(v);  // row_mirror
  return v;
}

// sum over the four lanes of a quad
__device__ __forceinline__ float quad_sum(float v) {
  v += dppf<0xB1>(v);
  return v + dppf<0x4E>(v);
}

// Workspace record of one (b, hv, chunk), offsets in bf16 elements: fragment
// tiles (rows x contraction), U as accumulator tiles (16 tokens x 16 columns, a
// float4 of 4 tokens a lane) and el as floats. cb_fwd_kernel is the only reader
// of the first three, so cb_bwd_kernel puts dS' over W1 and KD2 (2 K V <= 4 C K)
// and dv_n over U.
template <int K, int V>
struct Rec {
  static constexpr int W1 = 0;                 // W        C x K
  static constexpr int KD2 = 2 * C * K;        // Kd^T     K x C
  static constexpr int U = 4 * C * K;          // U        fp32
  static constexpr int KD1 = U + 2 * C * V;    // Kd       C x K
  static constexpr int QG2 = KD1 + 2 * C * K;  // Qg^T     K x C
  static constexpr int W2 = QG2 + 2 * C * K;   // -W^T     K x C
  static constexpr int AQ = W2 + 2 * C * K;    // Aqk^T    C x C
  static constexpr int XT = AQ + 2 * C * C;    // X^T      C x C
  static constexpr int EL = XT + 2 * C * C;    // el       fp32 [K]
  static constexpr int FL = EL + 2 * K;        // per 64 channels: decay products factored (int)
  static constexpr int RS = FL + 128;
  static constexpr int DSN = 0;                // dL/dS after the chunk, K x V, fp32
  static constexpr int DVN = U;                // dL/dv_n transposed, V x C
  static_assert(V <= 2 * C && RS % 128 == 0, "record layout");
};

struct CbWs {
  bf16_t* rec;  // [B*HV*NT][RS]
  bf16_t* sn;   // [B*HV*NT] state at the start of each chunk, fp32 tiles K x V
  bf16_t* vn;   // [B*HV*NT] v_n, tiles C x V
  float* part;  // [B,T,HV,3K+1] per-value-head partials (HV > H), else null
  int nt;
};

constexpr int NTH = 512;  // threads of the per-chunk kernels: 8 waves, two per SIMD

// sum over the eight lanes of a half DPP row
__device__ __forceinline__ float oct_sum(float v) {
  v = quad_sum(v);
  return v + dppf<0x141>(v);  // row_half_mirror
}

// In-place inclusive prefix sums down the C = 64 rows of columns [0, NCOL) of
// an LDS matrix with row stride ld (Rev: suffix sums, from the last row up),
// plus init[column] when init is given, by all NTH threads: column
// tid % NCOL, a segment of C / (NTH / NCOL) rows each; the segment totals
// meet in tot [NTH]. Ends with a barrier.
template <int NCOL, bool Rev>
__device__ __forceinline__ void col_scan(float* m, int ld, float* tot, const float* init) {
  constexpr int NSEG = NTH / NCOL, SL = C / NSEG;
  const int col = threadIdx.x % NCOL, seg = threadIdx.x / NCOL;
  const int r0 = Rev ? (NSEG - 1 - seg) * SL : seg * SL;
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < SL; ++r) {
    const int row = Rev ? r0 + SL - 1 - r : r0 + r;
    s += m[row * ld + col];
    m[row * ld + col] = s;
  }
  tot[seg * NCOL + col] = s;
  __syncthreads();
  float off = init ? init[col] : 0.f;
  for (int q = 0; q < seg; ++q) off += tot[q * NCOL + col];
#pragma unroll
  for (int r = 0; r < SL; ++r) m[(r0 + r) * ld + col] += off;
  __syncthreads();
}

// ---------------------------------------------------------------------------
// cb_prep_kernel: one workgroup (8 waves) per (b, hv, chunk), two per CU (16-bit
// inputs). Bound by HBM writes (K = V = 128: 224 KB a chunk; W and Kd in both
// orders, which the two state kernels need) and by the chain of phases between
// barriers, which the second workgroup fills: k is held as stored, q and v are
// read where they are used (L2), X takes M's place as split planes, 72 KB of
// LDS in all. 4096 chunks: 329 us (467 with fp32 copies of k, q, v and X, 138 KB
// and one workgroup a CU; 420 before the second orders were written).
// ---------------------------------------------------------------------------
template <int K, int V, typename InT>
__global__ __launch_bounds__(NTH, sizeof(InT) == 4 ? 2 : 4) void cb_prep_kernel(KdaBwdParams p, CbWs w) {
  using R = Rec<K, V>;
  constexpr unsigned SZ = sizeof(InT);
  constexpr int LK = K + 4, LC = C + 4, LX = C + 8, LI = K + 16 / (int)SZ;
  __shared__ __attribute__((aligned(16))) InT sk[C * LI];
  __shared__ __attribute__((aligned(16))) float sG[C * LK], stot[NTH], sb[C];
  // M (fp32), then the split planes of X
  __shared__ __attribute__((aligned(16))) bf16_t sX[2][C * LX];
  __shared__ int sflag[K / 64];
  float* const sM = reinterpret_cast<float*>(sX);
  static_assert(C * LC * 4 <= 4 * C * LX, "M fits where X goes");

  const int tid = threadIdx.x, l = tid & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
  const int nt = w.nt;
  const int n = blockIdx.x % nt, bh = blockIdx.x / nt;
  const int hv = bh % p.HV, b = bh / p.HV, h = hv / (p.HV / p.H);
  const int T = p.T, t0 = n * C;
  const float scale = (float)p.scale;
  const bool clampg = p.g_clamp_min > -INFINITY;
  const float gmin = (float)p.g_clamp_min;
  bf16_t* rec = w.rec + (size_t)blockIdx.x * R::RS;
  // the chunk's rows of an input, zero past the sequence's end
  const int last = min(T - 1 - t0, C - 1);
  auto rows = [&](const void* x, int heads, int head, int D) {
    return buf(static_cast<const char*>(x) + (((size_t)b * T + t0) * heads + head) * D * SZ,
               (size_t)(last + 1) * heads * D * SZ);
  };
  const __amdgpu_buffer_rsrc_t qb = rows(p.q, p.H, h, K), kb = rows(p.k, p.H, h, K),
                               gb = rows(p.g, p.HV, hv, K), vb = rows(p.v, p.HV, hv, V);
  const unsigned rq = p.H * K * SZ, rg = p.HV * K * SZ, rv = p.HV * V * SZ;
  typedef InT in8 __attribute__((ext_vector_type(8)));
  auto cvt8 = [](auto raw, float* f) {
    const in8 t = __builtin_bit_cast(in8, raw);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = to_f32((InT)t[i]);
  };
  // 8 tokens of one channel, rows r0 .. r0 + 7 of row stride ld
  auto col8 = [&](__amdgpu_buffer_rsrc_t r, unsigned ld, int r0, int ch, float* f) {
    const unsigned o = r0 * ld + ch * SZ;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (SZ == 4)
        f[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, o + i * ld, 0, 0));
      else
        f[i] = to_f32(__builtin_bit_cast(InT, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, o + i * ld, 0, 0)));
    }
  };

  if (tid < K / 64) sflag[tid] = 1;
  __syncthreads();
  for (int it = tid; it < C * (K / 8); it += NTH) {
    const int c = it / (K / 8), c8 = (it % (K / 8)) * 8;
    const auto kr = buf_load<InT, 8>(kb, c * rq + c8 * SZ);
    float fg[8];
    cvt8(buf_load<InT, 8>(gb, c * rg + c8 * SZ), fg);
    *reinterpret_cast<in8*>(&sk[c * LI + c8]) = __builtin_bit_cast(in8, kr);
    bool pos = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float gc = clampg ? fmaxf(fg[i], gmin) : fg[i];
      pos |= gc > 0.f;
      sG[c * LK + c8 + i] = gc;
    }
    if (pos) sflag[c8 / 64] = 0;
  }
  if (tid < C) {
    const int t = t0 + tid;
    sb[tid] = t < T ? to_f32(static_cast<const InT*>(p.beta)[(size_t)(b * T + t) * p.HV + hv]) : 0.f;
  }
  __syncthreads();
  col_scan<K, false>(sG, LK, stot, nullptr);
  if (tid < K) {
    const float ga = sG[kAnc * LK + tid];
    if (sG[tid] - ga > kAncRange || ga - sG[(C - 1) * LK + tid] > kAncRange) sflag[tid / 64] = 0;
  }
  __syncthreads();
  bool anchored = true;
#pragma unroll
  for (int i = 0; i < K / 64; ++i) anchored &= sflag[i] != 0;
  if (tid < K / 64) reinterpret_cast<int*>(rec + R::FL)[tid] = sflag[tid];

  // M and Aqk: wave wv owns column tile wv & 3 (j) of row tiles rt0, rt0 + 1 (i)
  {
    const int rt0 = 2 * (wv >> 2), jc = 16 * (wv & 3) + r16;
    f32x4 am[2], aa[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) am[u] = aa[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (anchored) {
      decltype(buf_load<InT, 8>(qb, 0)) qc[2], qn[2];
      auto qload = [&](int ks, auto& o) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          o[u] = buf_load<InT, 8>(qb, (16 * (rt0 + u) + r16) * rq + (ks + 8 * kq) * SZ);
      };
      qload(0, qc);
#pragma unroll 1
      for (int ks = 0; ks < K; ks += 32) {
        const int ch = ks + 8 * kq;
        if (ks + 32 < K) qload(ks + 32, qn);
        float fb[8], gj[8], ga[8];
        ld8g(&sk[jc * LI + ch], fb);
        ld8c(&sG[jc * LK + ch], gj);
        ld8c(&sG[kAnc * LK + ch], ga);
#pragma unroll
        for (int i = 0; i < 8; ++i) fb[i] *= ex(ga[i] - gj[i]);
        const Sp bs = sp8(fb);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int i0 = 16 * (rt0 + u) + r16;
          float fk[8], fq[8], gi[8];
          ld8g(&sk[i0 * LI + ch], fk);
          cvt8(qc[u], fq);
          ld8c(&sG[i0 * LK + ch], gi);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float P = ex(gi[i] - ga[i]);
            fk[i] *= P;
            fq[i] *= scale;
            fq[i] *= P;
          }
          am[u] = mm3(sp8(fk), bs, am[u]);
          aa[u] = mm3(sp8(fq), bs, aa[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) qc[u] = qn[u];
      }
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 16 * (rt0 + u) + 4 * kq + e;
          float m = 0.f, a = 0.f;
          if (jc <= i) {
#pragma unroll 1
            for (int c8 = 0; c8 < K; c8 += 8) {
              float fq[8];
              cvt8(buf_load<InT, 8>(qb, i * rq + c8 * SZ), fq);
#pragma unroll
              for (int z = 0; z < 8; ++z) {
                const int ch = c8 + z;
                const float x =
                    ex(fminf(sG[i * LK + ch] - sG[jc * LK + ch], kCap)) * to_f32(sk[jc * LI + ch]);
                m += to_f32(sk[i * LI + ch]) * x;
                a += scale * fq[z] * x;
              }
            }
          }
          am[u][e] = m;
          aa[u][e] = a;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x4 a;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * (rt0 + u) + 4 * kq + e;
        sM[i * LC + jc] = jc < i ? sb[i] * am[u][e] : 0.f;
        a[e] = jc <= i ? aa[u][e] : 0.f;
      }
      ft_store_acc(rec + R::AQ, wv & 3, 2, rt0 + u, sp4(a));
    }
  }
  // Qg^T and Kd^T (8 tokens of a channel), Kd (8 channels of a token), el
#pragma unroll 1
  for (int it = tid; it < K * (C / 8); it += NTH) {
    const int ch = it % K, c8 = it / K;
    const float Gl = sG[(C - 1) * LK + ch];
    float fq[8], fk[8];
    col8(qb, rq, 8 * c8, ch, fq);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float G = sG[(8 * c8 + i) * LK + ch];
      fq[i] *= scale;
      fq[i] *= ex(G);
      fk[i] = to_f32(sk[(8 * c8 + i) * LI + ch]) * ex(Gl - G);
    }
    const int tile = (ch >> 4) * 2 + (c8 >> 2), lane = (ch & 15) + 16 * (c8 & 3);
    ft_store(rec + R::QG2, tile, lane, sp8(fq));
    ft_store(rec + R::KD2, tile, lane, sp8(fk));
  }
#pragma unroll 1
  for (int it = tid; it < C * (K / 8); it += NTH) {
    const int c = it % C, k8 = it / C;
    float fk[8], gc[8], gl[8];
    ld8g(&sk[c * LI + 8 * k8], fk);
    ld8c(&sG[c * LK + 8 * k8], gc);
    ld8c(&sG[(C - 1) * LK + 8 * k8], gl);
#pragma unroll
    for (int i = 0; i < 8; ++i) fk[i] *= ex(gl[i] - gc[i]);
    ft_store(rec + R::KD1, (c >> 4) * (K / 32) + (k8 >> 2), (c & 15) + 16 * (k8 & 3), sp8(fk));
  }
  if (tid < K) reinterpret_cast<float*>(rec + R::EL)[tid] = ex(sG[(C - 1) * LK + tid]);
  __syncthreads();

  // X = (I + M)^-1, column cc by the eight lanes of a half row
  {
    const int cc = tid >> 3, part = tid & 7;
    float xr[8];
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) xr[jj] = 0.f;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float s = 0.f;
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        if (8 * jj < i) {
          const int j = 8 * jj + part;
          if (j < i) s += sM[i * LC + j] * xr[jj];
        }
      }
      s = oct_sum(s);
      const float xi = (i == cc ? 1.f : 0.f) - s;
      if (part == (i & 7)) xr[i >> 3] = xi;
    }
    __syncthreads();  // every read of M done
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) {
      const int o = (8 * jj + part) * LX + cc;
      const bf16_t hi = (bf16_t)xr[jj];
      sX[0][o] = hi;
      sX[1][o] = (bf16_t)(xr[jj] - (float)hi);
    }
  }
  __syncthreads();

  ft_store(rec + R::XT, wv, l,
           Sp{tr8(sX[0], LX, 32 * (wv & 1), 16 * (wv >> 1)), tr8(sX[1], LX, 32 * (wv & 1), 16 * (wv >> 1))});
  // W = X Bk in both orientations (the same fragments with the operands
  // exchanged) and U = X Bv, one tile of K (then of V) at a time over the
  // chunk's four row tiles, X's upper triangle left out
#pragma unroll 1
  for (int rtg = wv; rtg < K / 16 + V / 16; rtg += NTH / 64) {
    const bool isw = rtg < K / 16;
    const int r = 16 * (isw ? rtg : rtg - K / 16) + r16;
    Sp as[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int j0 = 32 * ks + 8 * kq;
      float fa[8];
      if (isw) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          fa[i] = to_f32(sk[(j0 + i) * LI + r]) * (sb[j0 + i] * ex(sG[(j0 + i) * LK + r]));
      } else {
        col8(vb, rv, j0, r, fa);
#pragma unroll
        for (int i = 0; i < 8; ++i) fa[i] *= sb[j0 + i];
      }
      as[ks] = sp8(fa);
    }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        if (2 * ks > ct) continue;
        const Sp xs = plane8(sX[0], sX[1], (16 * ct + r16) * LX + 32 * ks + 8 * kq);
        x = mm3(xs, as[ks], x);
        if (isw) y = mm3(as[ks], xs, y);
      }
      if (isw) {
        ft_store_acc(rec + R::W1, ct, K / 32, rtg, sp4(y));
        ft_store_acc(rec + R::W2, rtg, 2, ct, sp4(-x));
      } else {
        reinterpret_cast<f32x4*>(rec + R::U)[(ct * (V / 16) + rtg - K / 16) * 64 + l] = x;
      }
    }
  }
}

// (slice of V, head) of a state-kernel workgroup. Workgroups are dealt to the
// 8 XCDs round-robin; the NVS slices of a head are blocks 8 apart, so they
// share an XCD and its L2 and the head's per-chunk operands are read from HBM
// once.
template <int NVS>
__device__ __forceinline__ void slice_of(int& vs, int& bh) {
  const int g = blockIdx.x;
  if (NVS > 1 && (gridDim.x % (8 * NVS)) == 0) {
    vs = (g >> 3) % NVS;
    bh = g / (8 * NVS) * 8 + (g & 7);
  } else {
    vs = g % NVS;
    bh = g / NVS;
  }
}

// State rows in accumulators: wave wv owns rows [K/4 wv, K/4 (wv+1)) (KT tiles),
// lane: rows 4 kq + e of a tile, column r16 of the slice's column tile vt. Its
// split planes in LDS are [v][k].
template <int K, int VS>
struct StateTile {
  static constexpr int KT = K / 64, VT = VS / 16, LK = K + 8;

  // from fp32 [K][V] (null: zero) at column v0
  static __device__ __forceinline__ void load(f32x4 (&S)[KT][VT], const float* src, int V, int v0) {
    const int l = threadIdx.x & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          S[kt][vt][e] =
              src ? src[(size_t)(16 * (wv * KT + kt) + 4 * kq + e) * V + v0 + 16 * vt + r16] : 0.f;
  }

  static __device__ __forceinline__ void to_planes(const f32x4 (&S)[KT][VT], bf16_t* hi, bf16_t* lo) {
    const int l = threadIdx.x & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const Sp4 x = sp4(S[kt][vt]);
        const int o = (16 * vt + r16) * LK + 16 * (wv * KT + kt) + 4 * kq;
        *reinterpret_cast<bf16x4*>(hi + o) = x.hi;
        *reinterpret_cast<bf16x4*>(lo + o) = x.lo;
      }
  }

  // the wave's rows as fp32 fragment tiles K x V of the slice, transposed through
  // its own 16 rows of LDS (row stride VS + 4: stores and loads free of conflicts)
  static constexpr int LF = VS + 4;
  static __device__ __forceinline__ void store_tiles(bf16_t* dst, const f32x4 (&S)[KT][VT], float* tile, int V,
                                                     int v0) {
    const int l = threadIdx.x & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      wave_lds_sync();  // the last reads are done
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[(4 * kq + e) * LF + 16 * vt + r16] = S[kt][vt][e];
      wave_lds_sync();
#pragma unroll
      for (int vk = 0; vk < VS / 32; ++vk) {
        const float* p = tile + r16 * LF + 32 * vk + 8 * kq;
        ft_store_f32(dst, (wv * KT + kt) * (V / 32) + v0 / 32 + vk, l, *reinterpret_cast<const f32x4*>(p),
                     *reinterpret_cast<const f32x4*>(p + 4));
      }
    }
  }
};

// ---------------------------------------------------------------------------
// cb_fwd_kernel: one workgroup per (b, hv, VS columns of V), chunks in order.
// Bound by HBM (at K = V = 128: 96 KB read and 96 KB written a chunk) and by
// the chain of a chunk: two products with an LDS pass of split planes and a
// barrier after each. A wave's share of W, Kd^T, U and el of chunk n + 1 is in
// flight, in registers, through the whole of chunk n. At 64 heads of
// 64 chunks 213 us (3.7 TB/s), where splitting fp32 operands in every consumer
// and staging Kd through LDS took 456.
// ---------------------------------------------------------------------------
template <int K, int V, int VS>
__global__ __launch_bounds__(256, 1) void cb_fwd_kernel(KdaBwdParams p, CbWs w) {
  using R = Rec<K, V>;
  using ST = StateTile<K, VS>;
  constexpr int KT = ST::KT, VT = ST::VT, LK = ST::LK, LC = C + 8, KS = K / 32;
  __shared__ __attribute__((aligned(16))) bf16_t sS[2][VS * LK], sV[2][VS * LC];
  __shared__ __attribute__((aligned(16))) float sT[4][16 * ST::LF];
  const int tid = threadIdx.x, l = tid & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
  int vs, bh;
  slice_of<V / VS>(vs, bh);
  const int v0 = vs * VS, nt = w.nt;

  f32x4 S[KT][VT];
  const float* s0 = static_cast<const float*>(p.s0);
  ST::load(S, s0 ? s0 + (size_t)bh * K * V : nullptr, V, v0);
  ST::to_planes(S, sS[0], sS[1]);

  struct Ops {
    Sp w[KS], kd[KT][2];
    f32x4 u[VT], el[KT];
  };
  auto fetch = [&](int n, Ops& o) {
    const bf16_t* rec = w.rec + ((size_t)bh * nt + n) * R::RS;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) o.w[ks] = ft_load(rec + R::W1, wv * KS + ks);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
      o.u[vt] = reinterpret_cast<const f32x4*>(rec + R::U)[(wv * (V / 16) + v0 / 16 + vt) * 64 + l];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) o.kd[kt][ks] = ft_load(rec + R::KD2, (wv * KT + kt) * 2 + ks);
      o.el[kt] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(rec + R::EL) +
                                                 16 * (wv * KT + kt) + 4 * kq);
    }
  };
  auto chunk = [&](int n, Ops& cur, Ops& nxt) {
    const size_t ci = (size_t)bh * nt + n;
    if (n + 1 < nt) fetch(n + 1, nxt);
    // v_n = U - W S: the wave's 16 tokens
    f32x4 vn[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) vn[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
        vn[vt] = mm3(cur.w[ks], plane8(sS[0], sS[1], (16 * vt + r16) * LK + 32 * ks + 8 * kq), vn[vt]);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const Sp4 x = sp4(cur.u[vt] - vn[vt]);
      const int o = (16 * vt + r16) * LC + 16 * wv + 4 * kq;
      *reinterpret_cast<bf16x4*>(&sV[0][o]) = x.hi;
      *reinterpret_cast<bf16x4*>(&sV[1][o]) = x.lo;
    }
    ST::store_tiles(w.sn + ci * 2 * K * V, S, sT[wv], V, v0);
    __syncthreads();
#pragma unroll
    for (int vk = 0; vk < VS / 32; ++vk) {
      const Sp x = {tr8(sV[0], LC, 32 * vk, 16 * wv), tr8(sV[1], LC, 32 * vk, 16 * wv)};
      ft_store(w.vn + ci * 2 * C * V, wv * (V / 32) + v0 / 32 + vk, l, x);
    }
    // S = el S + Kd^T v_n
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) S[kt][vt] *= cur.el[kt];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const Sp b = plane8(sV[0], sV[1], (16 * vt + r16) * LC + 32 * ks + 8 * kq);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) S[kt][vt] = mm3(cur.kd[kt][ks], b, S[kt][vt]);
      }
    ST::to_planes(S, sS[0], sS[1]);
    __syncthreads();
  };
  Ops oa, ob;
  fetch(0, oa);
  __syncthreads();
#pragma unroll 1
  for (int n = 0; n < nt; n += 2) {
    chunk(n, oa, ob);
    if (n + 1 < nt) chunk(n + 1, ob, oa);
  }
}

// ---------------------------------------------------------------------------
// cb_bwd_kernel: one workgroup per (b, hv, VS columns of V), chunks in
// reverse; the shape of cb_fwd_kernel with dS' as the state, the operands of
// chunk n - 1 (and its dO rows, for the other of two LDS buffers) in flight
// through chunk n. Bound by HBM (at K = V = 128, bf16: 128 KB read and 96 KB
// written a chunk). 64 heads of 64 chunks: 302 us (3.0 TB/s; 683 with fp32
// operands, split by each wave and transposed through LDS).
// ---------------------------------------------------------------------------
template <int K, int V, int VS, typename InT>
__global__ __launch_bounds__(256, 1) void cb_bwd_kernel(KdaBwdParams p, CbWs w) {
  using R = Rec<K, V>;
  using ST = StateTile<K, VS>;
  constexpr int KT = ST::KT, VT = ST::VT, LK = ST::LK, LC = C + 8, KS = K / 32, LV = VS + 8;
  constexpr int NP = kParts<InT>, NDO = C * VS / 8 / 256;
  __shared__ __attribute__((aligned(16))) bf16_t sD[2][VS * LK], sdV[2][VS * LC], sdO[2][NP][C * LV];
  __shared__ __attribute__((aligned(16))) float sT[4][16 * ST::LF];
  const int tid = threadIdx.x, l = tid & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
  int vs, bh;
  slice_of<V / VS>(vs, bh);
  const int v0 = vs * VS, nt = w.nt, T = p.T;
  const int hv = bh % p.HV, b = bh / p.HV;
  const InT* dO = static_cast<const InT*>(p.d_o) + ((size_t)b * T * p.HV + hv) * V + v0;
  const size_t ldo = (size_t)p.HV * V;

  f32x4 D[KT][VT];
  const float* dsf = static_cast<const float*>(p.ds_final);
  ST::load(D, dsf ? dsf + (size_t)bh * K * V : nullptr, V, v0);
  ST::to_planes(D, sD[0], sD[1]);

  struct Ops {
    Sp aq[2], kd[KS], qg[KT][2], wt[KT][2];
    f32x4 el[KT];
    float d_o[NDO][8];
  };
  auto fetch = [&](int n, Ops& o) {
    const bf16_t* rec = w.rec + ((size_t)bh * nt + n) * R::RS;
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int it = tid + 256 * i, c = it / (VS / 8), v8 = it % (VS / 8), t = n * C + c;
      if (t < T)
        ld8g(dO + t * ldo + 8 * v8, o.d_o[i]);
      else
        zero8(o.d_o[i]);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) o.aq[ks] = ft_load(rec + R::AQ, wv * 2 + ks);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) o.kd[ks] = ft_load(rec + R::KD1, wv * KS + ks);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        o.qg[kt][ks] = ft_load(rec + R::QG2, (wv * KT + kt) * 2 + ks);
        o.wt[kt][ks] = ft_load(rec + R::W2, (wv * KT + kt) * 2 + ks);
      }
      o.el[kt] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(rec + R::EL) +
                                                 16 * (wv * KT + kt) + 4 * kq);
    }
  };
  auto put_do = [&](int buf, const Ops& o) {
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int it = tid + 256 * i, c = it / (VS / 8), v8 = it % (VS / 8);
      const Sp x = sp8(o.d_o[i]);
      *reinterpret_cast<bf16x8*>(&sdO[buf][0][c * LV + 8 * v8]) = x.hi;
      if constexpr (NP == 2) *reinterpret_cast<bf16x8*>(&sdO[buf][1][c * LV + 8 * v8]) = x.lo;
    }
  };
  auto chunk = [&](int n, Ops& cur, Ops& nxt) {
    const size_t ci = (size_t)bh * nt + n;
    bf16_t* rec = w.rec + ci * R::RS;
    if (n > 0) fetch(n - 1, nxt);
    // dv_n = Aqk^T dO + Kd dS': the wave's 16 tokens
    Sp dof[2][VT];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        dof[ks][vt].hi = tr8(sdO[n & 1][0], LV, 32 * ks, 16 * vt);
        if constexpr (NP == 2) dof[ks][vt].lo = tr8(sdO[n & 1][NP - 1], LV, 32 * ks, 16 * vt);
      }
    f32x4 dv[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) dv[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) dv[vt] = mmp<NP>(cur.aq[ks], dof[ks][vt], dv[vt]);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
        dv[vt] = mm3(cur.kd[ks], plane8(sD[0], sD[1], (16 * vt + r16) * LK + 32 * ks + 8 * kq), dv[vt]);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const Sp4 x = sp4(dv[vt]);
      const int o = (16 * vt + r16) * LC + 16 * wv + 4 * kq;
      *reinterpret_cast<bf16x4*>(&sdV[0][o]) = x.hi;
      *reinterpret_cast<bf16x4*>(&sdV[1][o]) = x.lo;
      ft_store_acc(rec + R::DVN, v0 / 16 + vt, 2, wv, x);
    }
    ST::store_tiles(rec + R::DSN, D, sT[wv], V, v0);
    __syncthreads();
    // dS = el dS' + Qg^T dO - W^T dv_n
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) D[kt][vt] *= cur.el[kt];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const Sp x = plane8(sdV[0], sdV[1], (16 * vt + r16) * LC + 32 * ks + 8 * kq);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          D[kt][vt] = mmp<NP>(cur.qg[kt][ks], dof[ks][vt], D[kt][vt]);
          D[kt][vt] = mm3(cur.wt[kt][ks], x, D[kt][vt]);
        }
      }
    ST::to_planes(D, sD[0], sD[1]);
    if (n > 0) put_do((n - 1) & 1, nxt);
    __syncthreads();
  };
  Ops oa, ob;
  fetch(nt - 1, oa);
  put_do((nt - 1) & 1, oa);
  __syncthreads();
#pragma unroll 1
  for (int n = nt - 1; n >= 0; n -= 2) {
    chunk(n, oa, ob);
    if (n > 0) chunk(n - 1, ob, oa);
  }
  if (p.ds0) {
    float* ds0 = static_cast<float*>(p.ds0) + (size_t)bh * K * V;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          ds0[(size_t)(16 * (wv * KT + kt) + 4 * kq + e) * V + v0 + 16 * vt + r16] = D[kt][vt][e];
  }
}

// ---------------------------------------------------------------------------
// cb_grad_kernel: one workgroup (4 waves) per (b, hv, chunk), two per CU.
// Bound by HBM (at K = V = 128, bf16: 288 KB read and 64 KB written a chunk).
// A wave owns whole columns of the chunk (16-channel tiles, all 64 tokens), so
// the gate sums, their reversed sums and the sums over tokens stay in its
// registers (in-lane steps and two shuffles), the key and query factors of the
// decay products are made once, by the lanes that need them, and S and dS'
// fragments are read by one wave only. The decay products contract over the
// tokens in accumulator order (lane kq: tokens 16 rt + 4 kq + e), which makes
// those registers the operand as they stand. The row offsets
// go through buffer addressing: as 64-bit lane addresses they spilled (805 us).
// 4096 chunks: 500 us (2.9 TB/s), where fp32 operands split by every reader, two
// waves a SIMD of one workgroup and a load round trip per step took 1190.
// ---------------------------------------------------------------------------
template <int K, int V, typename InT>
__global__ __launch_bounds__(256, 2) void cb_grad_kernel(KdaBwdParams p, CbWs w) {
  using R = Rec<K, V>;
  constexpr int LV = V + 8, LC = C + 8, KT = K / 64, VT = V / 64, VS = V / 32, NP = kParts<InT>;
  __shared__ __attribute__((aligned(16))) bf16_t sdB[2][C * LV], sdA[2][C * LC], sdM[2][C * LC];
  __shared__ __attribute__((aligned(16))) float sb[C], sbeta[2][4][C];

  const int tid = threadIdx.x, l = tid & 63, wv = wave_id(), r16 = l & 15, kq = l >> 4;
  const int nt = w.nt;
  const int n = blockIdx.x % nt, bh = blockIdx.x / nt;
  const int hv = bh % p.HV, b = bh / p.HV, h = hv / (p.HV / p.H);
  const int T = p.T, t0 = n * C, HV = p.HV;
  const float scale = (float)p.scale;
  const bool clampg = p.g_clamp_min > -INFINITY;
  const float gmin = (float)p.g_clamp_min;
  const bool direct = w.part == nullptr;
  const size_t ci = blockIdx.x;
  const __amdgpu_buffer_rsrc_t rec = buf(w.rec + ci * R::RS, 2 * (size_t)R::RS);
  const __amdgpu_buffer_rsrc_t sn = buf(w.sn + ci * 2 * K * V, 4 * (size_t)K * V);
  const __amdgpu_buffer_rsrc_t vng = buf(w.vn + ci * 2 * C * V, 4 * (size_t)C * V);
  // the chunk's rows of an input or gradient (row stride ld elements, first
  // element base0), up to the sequence's end
  const int last = min(T - 1 - t0, C - 1);
  constexpr unsigned SZ = sizeof(InT);
  auto rows = [&](const void* x, int heads, int head, int D) {
    return buf(static_cast<const char*>(x) + (((size_t)b * T + t0) * heads + head) * D * SZ,
               (size_t)(last + 1) * heads * D * SZ);
  };
  const unsigned rs = HV * V * SZ, rq = p.H * K * SZ, rg = HV * K * SZ;  // row strides, bytes
  const __amdgpu_buffer_rsrc_t dO = rows(p.d_o, HV, hv, V), vin = rows(p.v, HV, hv, V),
                               dvout = rows(p.dv, HV, hv, V);

  // dO rows 16 rt + r16, columns 32 ks + 8 kq .. + 7
  auto do_load = [&](unsigned od, int rt, int ks) {
    return buf_load<InT, 8>(dO, od + 16 * rt * rs + 32 * ks * SZ);
  };
  const unsigned od0 = r16 * rs + 8 * kq * SZ;
  auto do_split = [](auto raw) {
    Sp x;
    if constexpr (NP == 1) {
      x.hi = __builtin_bit_cast(bf16x8, raw);
      x.lo = bf16x8{};
    } else {
      typedef InT in8 __attribute__((ext_vector_type(8)));
      const in8 t = __builtin_bit_cast(in8, raw);
      float f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = to_f32((InT)t[i]);
      x = sp8(f);
    }
    return x;
  };
  auto raw_f32 = [](uint32_t r) {
    if constexpr (SZ == 4)
      return __uint_as_float(r);
    else
      return to_f32(__builtin_bit_cast(InT, (uint16_t)r));
  };
  auto load1 = [](__amdgpu_buffer_rsrc_t r, unsigned off) -> uint32_t {
    if constexpr (SZ == 4)
      return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    else
      return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  };
  auto store1 = [](float x, __amdgpu_buffer_rsrc_t r, unsigned off) {
    const InT y = from_f32<InT>(x);
    if constexpr (SZ == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), r, off, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, y), r, off, 0, 0);
  };
  auto dB_frag = [&](int rt, int ks) {
    return plane8(sdB[0], sdB[1], (16 * rt + r16) * LV + 32 * ks + 8 * kq);
  };
  // dO as the left operand
  auto mma_do = [](const Sp& a, const Sp& x, f32x4 acc) {
    if constexpr (SZ == 4) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, x.lo, acc, 0, 0, 0);
    if constexpr (NP == 2) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, x.hi, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, x.lo, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, x.hi, acc, 0, 0, 0);
  };

  // fp32 gradients also take the product of the low parts (against float64 at
  // K = V = 128: dq and dk 6.9e-6 -> 6.3e-6 of their norm, dg 1.4e-5 -> 9.9e-6)
  auto mmg = [](const Sp& a, const Sp& x, f32x4 acc) {
    if constexpr (SZ == 4) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, x.lo, acc, 0, 0, 0);
    return mm3(a, x, acc);
  };
  if (tid < C) {
    const int t = t0 + tid;
    sb[tid] = t < T ? to_f32(static_cast<const InT*>(p.beta)[(size_t)(b * T + t) * HV + hv]) : 0.f;
  }
  __syncthreads();

  bool factored = true;  // every block of 64 channels
#pragma unroll
  for (int i = 0; i < K / 64; ++i)
    factored &= __builtin_amdgcn_raw_buffer_load_b32(rec, 0, 2 * R::FL + 4 * i, 0) != 0;

  // phase 1: dBv^T = dv_n^T X (rows of V, lanes tokens); dv = beta dBv;
  // dbeta += v . dBv
  {
    f32x4 acc[VT][4];
#pragma unroll
    for (int u = 0; u < VT; ++u)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) acc[u][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    Sp a[VT][2];
    typedef InT in4 __attribute__((ext_vector_type(4)));
    decltype(buf_load<InT, 4>(vin, 0)) vr[VT][4];
#pragma unroll
    for (int u = 0; u < VT; ++u) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) a[u][ks] = ft_load(rec, R::DVN, (wv * VT + u) * 2 + ks);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        vr[u][ct] = buf_load<InT, 4>(vin, (16 * ct + r16) * rs + (16 * (wv * VT + u) + 4 * kq) * SZ);
    }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        if (2 * ks + 1 < ct) continue;  // X^T is upper triangular
        const Sp x = ft_load(rec, R::XT, ct * 2 + ks);
#pragma unroll
        for (int u = 0; u < VT; ++u) acc[u][ct] = mmg(a[u][ks], x, acc[u][ct]);
      }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int c = 16 * ct + r16;
      const float bb = sb[c];
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < VT; ++u) {
        const int vv = 16 * (wv * VT + u) + 4 * kq;
        const f32x4 x = acc[u][ct];
        const Sp4 y = sp4(x);
        *reinterpret_cast<bf16x4*>(&sdB[0][c * LV + vv]) = y.hi;
        *reinterpret_cast<bf16x4*>(&sdB[1][c * LV + vv]) = y.lo;
        const in4 vin4 = __builtin_bit_cast(in4, vr[u][ct]);
        in4 dr;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s += to_f32((InT)vin4[e]) * x[e];
          dr[e] = from_f32<InT>(bb * x[e]);
        }
        const unsigned o = c * rs + vv * SZ;
        if constexpr (SZ == 4)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, dr), dvout, o, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, dr), dvout, o, 0, 0);
      }
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (kq == 0) sbeta[0][wv][c] = s;
    }
  }
  __syncthreads();

  // phase 2: dAqk = dO v_n^T (j <= i), dM = -dBv v_n^T (j < i), transposed: the
  // wave's rows are tokens j of its tile, lanes tokens i
  {
    f32x4 a1[4], a2[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) a1[rt] = a2[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < VS; ++ks) {
      const Sp a = ft_load(vng, 0, wv * VS + ks);
      decltype(do_load(0, 0, 0)) d[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) d[rt] = do_load(od0, rt, ks);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        a1[rt] = mmp<NP>(a, do_split(d[rt]), a1[rt]);
        a2[rt] = mmg(a, dB_frag(rt, ks), a2[rt]);
      }
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const int i = 16 * rt + r16, j = 16 * wv + 4 * kq;
      f32x4 x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = j + e <= i ? a1[rt][e] : 0.f;
        y[e] = j + e < i ? -a2[rt][e] : 0.f;
      }
      if (!factored) {
        // for the exact decay terms, in fp32 and both orders, over Aqk^T and X^T
        float* xa = reinterpret_cast<float*>(w.rec + ci * R::RS + R::AQ);
#pragma unroll 1
        for (int z = 0; z < 8; ++z) {
          const int jj = j + (z & 3);
          float val = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if ((z & 3) == e) val = z < 4 ? x[e] : y[e];
          if (jj <= i) xa[(z < 4 ? 0 : C * C) + jj * C + i] = xa[(z < 4 ? 0 : C * C) + i * C + jj] = val;
        }
      }
      const Sp4 xs = sp4(x), ys = sp4(y);
      *reinterpret_cast<bf16x4*>(&sdA[0][i * LC + j]) = xs.hi;
      *reinterpret_cast<bf16x4*>(&sdA[1][i * LC + j]) = xs.lo;
      *reinterpret_cast<bf16x4*>(&sdM[0][i * LC + j]) = ys.hi;
      *reinterpret_cast<bf16x4*>(&sdM[1][i * LC + j]) = ys.lo;
    }
  }
  __syncthreads();

  // phase 3: the wave's channel tiles; lane: channel ch, tokens 16 rt + 4 kq + e
  float dbeta[4][4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) dbeta[rt][e] = 0.f;
#pragma unroll 1
  for (int kt = 0; kt < KT; ++kt) {
    const int ctg = wv * KT + kt, ch = 16 * ctg + r16;
    // dQg = dO S^T, dBk = -dBv S^T, dKd = v_n dS'^T; del
    f32x4 x1[4], x2[4], x3[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) x1[rt] = x2[rt] = x3[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float del = 0.f;
    // the next step's state tiles (read here only) are in flight through each
    // step, the gates, keys and queries through the last
    const __amdgpu_buffer_rsrc_t qb = rows(p.q, p.H, h, K), kb = rows(p.k, p.H, h, K),
                                 gb = rows(p.g, HV, hv, K);
    unsigned oq = 4 * kq * rq + ch * SZ, og = 4 * kq * rg + ch * SZ;
    unsigned od = od0;
    // (opaque, or the loop keeps every row's offset in a register of its own)
    asm volatile("" : "+v"(oq), "+v"(og), "+v"(od));
    uint32_t xg[4][4], xq[4][4], xk[4][4];
    F8 s1 = ft_load_f32(sn, 0, ctg * VS), s3 = ft_load_f32(rec, R::DSN, ctg * VS);
#pragma unroll
    for (int ks = 0; ks < VS; ++ks) {
      decltype(do_load(0, 0, 0)) d[4];
      Sp v[4];
      F8 n1, n3;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        d[rt] = do_load(od, rt, ks);
        v[rt] = ft_load(vng, 0, rt * VS + ks);
      }
      if (ks + 1 < VS) {
        n1 = ft_load_f32(sn, 0, ctg * VS + ks + 1);
        n3 = ft_load_f32(rec, R::DSN, ctg * VS + ks + 1);
      } else {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            xg[rt][e] = load1(gb, og + (16 * rt + e) * rg);
            xq[rt][e] = load1(qb, oq + (16 * rt + e) * rq);
            xk[rt][e] = load1(kb, oq + (16 * rt + e) * rq);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      float f1[8], f3[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f1[i] = s1.a[i]; f1[4 + i] = s1.b[i];
        f3[i] = s3.a[i]; f3[4 + i] = s3.b[i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) del += f1[i] * f3[i];
      const Sp b1 = sp8(f1), b3 = sp8(f3);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        x1[rt] = mma_do(do_split(d[rt]), b1, x1[rt]);
        x2[rt] = mmg(dB_frag(rt, ks), b1, x2[rt]);
        x3[rt] = mmg(v[rt], b3, x3[rt]);
      }
      __builtin_amdgcn_sched_barrier(0);
      s1 = n1;
      s3 = n3;
    }
    del += __shfl_xor(del, 16);
    del += __shfl_xor(del, 32);

    float G[4][4], kk[4][4], qq[4][4];
    unsigned pass = 0;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float g = raw_f32(xg[rt][e]);
        if (!clampg || g >= gmin) pass |= 1u << (4 * rt + e);
        G[rt][e] = clampg ? fmaxf(g, gmin) : g;
        qq[rt][e] = scale * raw_f32(xq[rt][e]);
        kk[rt][e] = raw_f32(xk[rt][e]);
      }
    // prefix sums over the chunk's tokens: in runs of 8 (lanes kq, kq + 1), then
    // over the runs
    float run = 0.f;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const float half = ((G[rt][0] + G[rt][1]) + G[rt][2]) + G[rt][3];
      const float before = __shfl_xor(half, 16);
      if (kq & 1) G[rt][0] += before;
#pragma unroll
      for (int e = 1; e < 4; ++e) G[rt][e] += G[rt][e - 1];
      const float t0r = __shfl(G[rt][3], 16 + r16), t1r = __shfl(G[rt][3], 48 + r16);
      const float off = kq < 2 ? run : run + t0r;
#pragma unroll
      for (int e = 0; e < 4; ++e) G[rt][e] += off;
      run = (run + t0r) + t1r;
    }
    const float Ga = __shfl(G[1][3], 48 + r16), Gl = __shfl(G[3][3], 48 + r16);
    const bool anchored =
        factored || __builtin_amdgcn_raw_buffer_load_b32(rec, 0, 2 * R::FL + 4 * (ctg / 4), 0) != 0;

    float dq[4][4], dk[4][4], dg[4][4], ext = 0.f;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const float4 b4 = *reinterpret_cast<const float4*>(&sb[16 * rt + 4 * kq]);
      const float bb[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float eG = ex(G[rt][e]), ed = ex(Gl - G[rt][e]);
        const float y1 = eG * x1[rt][e], y2 = -eG * x2[rt][e], y3 = ed * x3[rt][e];
        dq[rt][e] = y1;
        dk[rt][e] = y3 + bb[e] * y2;
        dg[rt][e] = qq[rt][e] * y1 - kk[rt][e] * y3 + bb[e] * kk[rt][e] * y2;
        ext += kk[rt][e] * y3;
        dbeta[rt][e] += kk[rt][e] * y2;
      }
    }
    ext += __shfl_xor(ext, 16);
    ext += __shfl_xor(ext, 32);
    ext += ex(Gl) * del;

    if (anchored) {
      // R1' = dM KN, R2 = dAqk KN, then C = dM^T (beta KP) + dAqk^T QP with
      // KN = k e^(G_a - G), KP = k e^(G - G_a), QP = q^ e^(G - G_a); one after
      // the other, as all accumulators at once do not fit the registers
      {
        f32x4 r1[4], r2[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) r1[rt] = r2[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          float f[8];
#pragma unroll
          for (int i = 0; i < 8; ++i)
            f[i] = kk[2 * ks + (i >> 2)][i & 3] * ex(Ga - G[2 * ks + (i >> 2)][i & 3]);
          const Sp bN = sp8(f);
          // tokens j <= i: rows of dM and dAqk
          auto rows = [&](const bf16_t* hi, const bf16_t* lo, int rt) {
            const int o = (16 * rt + r16) * LC + 32 * ks + 4 * kq;
            return Sp{cat4(*reinterpret_cast<const bf16x4*>(hi + o),
                           *reinterpret_cast<const bf16x4*>(hi + o + 16)),
                      cat4(*reinterpret_cast<const bf16x4*>(lo + o),
                           *reinterpret_cast<const bf16x4*>(lo + o + 16))};
          };
#pragma unroll
          for (int rt = 2 * ks; rt < 4; ++rt) {
            r1[rt] = mmg(rows(sdM[0], sdM[1], rt), bN, r1[rt]);
            r2[rt] = mmg(rows(sdA[0], sdA[1], rt), bN, r2[rt]);
          }
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const f32x4 bb = *reinterpret_cast<const f32x4*>(&sb[16 * rt + 4 * kq]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float P = ex(G[rt][e] - Ga);
            const float y1 = kk[rt][e] * (P * r1[rt][e]), y2 = P * r2[rt][e];
            dk[rt][e] += bb[e] * (P * r1[rt][e]);
            dq[rt][e] += y2;
            dg[rt][e] += bb[e] * y1 + qq[rt][e] * y2;
            dbeta[rt][e] += y1;
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      f32x4 cc[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) cc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        float fP[8], fQ[8];
#pragma unroll
        for (int z = 0; z < 2; ++z) {
          const f32x4 bb = *reinterpret_cast<const f32x4*>(&sb[16 * (2 * ks + z) + 4 * kq]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float P = ex(G[2 * ks + z][e] - Ga);
            fP[4 * z + e] = bb[e] * kk[2 * ks + z][e] * P;
            fQ[4 * z + e] = qq[2 * ks + z][e] * P;
          }
        }
        const Sp bP = sp8(fP), bQ = sp8(fQ);
        // tokens i >= j: columns of dM and dAqk
        auto cols = [&](const bf16_t* hi, const bf16_t* lo, int rt) {
          const int r0 = 32 * ks + 4 * kq;
          return Sp{cat4(tr4(hi, LC, r0, 16 * rt), tr4(hi, LC, r0 + 16, 16 * rt)),
                    cat4(tr4(lo, LC, r0, 16 * rt), tr4(lo, LC, r0 + 16, 16 * rt))};
        };
#pragma unroll
        for (int rt = 0; rt < 2 * ks + 2; ++rt) {
          cc[rt] = mmg(cols(sdM[0], sdM[1], rt), bP, cc[rt]);
          cc[rt] = mmg(cols(sdA[0], sdA[1], rt), bQ, cc[rt]);
        }
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float yc = ex(Ga - G[rt][e]) * cc[rt][e];
          dk[rt][e] += yc;
          dg[rt][e] -= kk[rt][e] * yc;
        }
    } else {
      // The exact products, one exponential per token pair and channel, with the
      // clamp at 50 and its zero gradient in dG: over tokens j in turn, each lane
      // adds the pair's term to its 16 tokens i (j < i: row i of dM and dAqk, j >
      // i: column i). G, k, q^ of the tile pass through the chunk's record (its
      // Kd, Qg^T and W^T are not read any more); token j + 1's values are in
      // flight through token j's 16 terms. Exact throughout (gates past 60 nats),
      // 16 heads of 128, bf16, whole backward: B1 T2048 567 us, B4 T1024 988, with
      // the terms staged in LDS by one workgroup a CU 892 and 1124.
      auto at = [&](unsigned v, int off) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rec, v, off, 0));
      };
      auto at4 = [&](unsigned v, int off) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rec, v, off, 0));
      };
      auto put = [&](float x, unsigned v, int off) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rec, v, off, 0);
      };
      constexpr int oG = 2 * R::KD1, ok = oG + 4 * C * K, oq2 = ok + 4 * C * K;
      constexpr int oA = 2 * R::AQ, oM = oA + 4 * C * C;
      unsigned vo = 4 * ch, vd = 4 * (4 * kq * (C + 1)), vr = 16 * kq;
      asm volatile("" : "+v"(vo), "+v"(vd), "+v"(vr));
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned v = vo + 16 * kq * K;
          const int o = 4 * (16 * rt + e) * K;
          put(G[rt][e], v, oG + o);
          put(kk[rt][e], v, ok + o);
          put(qq[rt][e], v, oq2 + o);
          const float a = at(vd, oA + 4 * (16 * rt + e) * (C + 1));  // dAqk[i][i]
          dq[rt][e] += a * kk[rt][e];
          dk[rt][e] += a * qq[rt][e];
        }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      float nG = at(vo, oG), nk = at(vo, ok), nq = at(vo, oq2);
#pragma unroll 1
      for (int j = 0; j < C; ++j) {
        const float Gj = nG, kj = nk, qj = nq, bk = sb[j] * nk;
        int i0 = 4 * kq;
        asm volatile("" : "+v"(i0));  // (as above)
        const int jn = 4 * K * min(j + 1, C - 1);
        nG = at(vo, oG + jn);
        nk = at(vo, ok + jn);
        nq = at(vo, oq2 + jn);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const f32x4 A = at4(vr, oA + 4 * (j * C + 16 * rt)), M = at4(vr, oM + 4 * (j * C + 16 * rt));
          const f32x4 bb = *reinterpret_cast<const f32x4*>(&sb[16 * rt + i0]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 16 * rt + e + i0;
            const float d0 = G[rt][e] - Gj, d = j < i ? d0 : -d0;
            const float E = ex(fminf(d, kCap)), x = E * kj;
            const float m = j < i ? M[e] * x : 0.f, a = j < i ? A[e] * x : 0.f;
            const float c = j > i ? (M[e] * bk + A[e] * qj) * E : 0.f;
            const float km = kk[rt][e] * m;
            dk[rt][e] += bb[e] * m + c;
            dq[rt][e] += a;
            dbeta[rt][e] += km;
            const float t = bb[e] * km + qq[rt][e] * a - kk[rt][e] * c;
            dg[rt][e] += d > kCap ? 0.f : t;
          }
        }
      }
    }
    // suffix sums of dG over the chunk's tokens, plus the G_l gradient
    run = ext;
#pragma unroll
    for (int rt = 3; rt >= 0; --rt) {
      const float half = ((dg[rt][3] + dg[rt][2]) + dg[rt][1]) + dg[rt][0];
      const float after = __shfl_xor(half, 16);
      if (!(kq & 1)) dg[rt][3] += after;
#pragma unroll
      for (int e = 2; e >= 0; --e) dg[rt][e] += dg[rt][e + 1];
      const float t1r = __shfl(dg[rt][0], 32 + r16), t0r = __shfl(dg[rt][0], r16);
      const float off = kq >= 2 ? run : run + t1r;
#pragma unroll
      for (int e = 0; e < 4; ++e) dg[rt][e] += off;
      run = (run + t1r) + t0r;
    }
    if (direct) {
      const __amdgpu_buffer_rsrc_t dqb = rows(p.dq, p.H, h, K), dkb = rows(p.dk, p.H, h, K),
                                   dgb = rows(p.dg, HV, hv, K);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          store1(scale * dq[rt][e], dqb, oq + (16 * rt + e) * rq);
          store1(dk[rt][e], dkb, oq + (16 * rt + e) * rq);
          store1((pass >> (4 * rt + e)) & 1 ? dg[rt][e] : 0.f, dgb, og + (16 * rt + e) * rg);
        }
    } else {
      const unsigned ld = HV * (3 * K + 1) * 4;
      const __amdgpu_buffer_rsrc_t prb =
          buf(w.part + ((size_t)(b * T + t0) * HV + hv) * (3 * K + 1), (size_t)(last + 1) * ld);
      unsigned op = 4 * kq * ld + 4 * ch;
      asm volatile("" : "+v"(op));
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned o = op + (16 * rt + e) * ld;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dq[rt][e]), prb, o, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dk[rt][e]), prb, o + 4 * K, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dg[rt][e]), prb, o + 8 * K, 0, 0);
        }
    }
  }
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float s = row16_sum(dbeta[rt][e]);
      if (r16 == 0) sbeta[1][wv][16 * rt + 4 * kq + e] = s;
    }
  __syncthreads();
  if (tid < C && t0 + tid < T) {
    const int t = t0 + tid;
    float s = 0.f;
#pragma unroll
    for (int z = 0; z < 4; ++z) s += sbeta[0][z][tid] + sbeta[1][z][tid];
    if (direct)
      static_cast<InT*>(p.dbeta)[(size_t)(b * T + t) * HV + hv] = from_f32<InT>(s);
    else
      w.part[((size_t)(b * T + t) * HV + hv) * (3 * K + 1) + 3 * K] = s;
  }
}

size_t al256(size_t x) { return (x + 255) & ~size_t(255); }

int cu_count() {
  // multiprocessor count of each device, queried once
  static std::atomic<int> counts[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int c = counts[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) c = 256;
    counts[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

size_t rec_bytes(int K, int V) {
  return 2 * ((size_t)10 * C * K + 2 * C * V + 4 * C * C + 2 * K + 128);
}

// Slices of V per state workgroup: 32 columns when 64-column slices would
// leave half of the CUs without one (a workgroup's share of a chunk is then
// half as long; the rows of W, Kd and Qg that both halves read come from their
// XCD's L2). Forward and backward of
// 16 heads of 128 at T 2048: B 4 (128 workgroups of 64 columns) 966 us against
// 870 with 32, B 5 (160) 1113 against 1169; heads of 64 at B 8 (128) 831 against
// 777, B 12 (192) 1112 against 1129.
template <int K, int V, int VS, typename InT>
hipError_t state_launch(const KdaBwdParams& p, const CbWs& w, hipStream_t s) {
  const unsigned grid = (unsigned)((size_t)p.B * p.HV * (V / VS));
  hipLaunchKernelGGL((cb_fwd_kernel<K, V, VS>), dim3(grid), dim3(256), 0, s, p, w);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((cb_bwd_kernel<K, V, VS, InT>), dim3(grid), dim3(256), 0, s, p, w);
  return hipGetLastError();
}

template <int K, int V, typename InT>
hipError_t cb_launch(const KdaBwdParams& p, const CbWs& w, hipStream_t s) {
  constexpr int dt = sizeof(InT) == 4 ? DT_F32 : (std::is_same<InT, bf16_t>::value ? DT_BF16 : DT_F16);
  const unsigned chunks = (unsigned)((size_t)p.B * p.HV * w.nt);
  hipLaunchKernelGGL((cb_prep_kernel<K, V, InT>), dim3(chunks), dim3(NTH), 0, s, p, w);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (2LL * p.B * p.HV * (V / 64) <= cu_count())
    e = state_launch<K, V, 32, InT>(p, w, s);
  else
    e = state_launch<K, V, 64, InT>(p, w, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((cb_grad_kernel<K, V, InT>), dim3(chunks), dim3(256), 0, s, p, w);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (w.part) {
    KdaBwdParams q = p;
    q.part = w.part;
    return kda_bwd_reduce_launch(q, V, dt, s);
  }
  return hipSuccess;
}

template <typename InT>
hipError_t cb_by_shape(const KdaBwdParams& p, const CbWs& w, hipStream_t s) {
  if (p.K == 128 && p.V == 128) return cb_launch<128, 128, InT>(p, w, s);
  if (p.K == 128 && p.V == 64) return cb_launch<128, 64, InT>(p, w, s);
  if (p.K == 64 && p.V == 128) return cb_launch<64, 128, InT>(p, w, s);
  return cb_launch<64, 64, InT>(p, w, s);
}

}  // namespace

bool kda_chunk_bwd_supported(int K, int V, int dtype) {
  return dtype != DT_F64 && (K == 64 || K == 128) && (V == 64 || V == 128);
}

size_t kda_chunk_bwd_ws_bytes(int B, int T, int H, int HV, int K, int V) {
  const size_t nt = (size_t)(T + C - 1) / C;
  const size_t chunks = (size_t)B * HV * nt;
  size_t total = al256(chunks * rec_bytes(K, V));
  total += al256(chunks * K * V * 4);
  total += al256(chunks * C * V * 4);
  if (HV != H) total += al256((size_t)B * T * HV * (3 * K + 1) * 4);
  return total;
}

hipError_t kda_chunk_bwd_dispatch(KdaBwdParams p, int dtype, void* ws, hipStream_t stream) {
  const int nt = (p.T + C - 1) / C;
  const size_t chunks = (size_t)p.B * p.HV * nt;
  char* base = static_cast<char*>(ws);
  CbWs w;
  w.nt = nt;
  w.rec = reinterpret_cast<bf16_t*>(base);
  base += al256(chunks * rec_bytes(p.K, p.V));
  w.sn = reinterpret_cast<bf16_t*>(base);
  base += al256(chunks * p.K * p.V * 4);
  w.vn = reinterpret_cast<bf16_t*>(base);
  base += al256(chunks * C * p.V * 4);
  w.part = p.HV != p.H ? reinterpret_cast<float*>(base) : nullptr;
  if (dtype == DT_F32) return cb_by_shape<float>(p, w, stream);
  if (dtype == DT_BF16) return cb_by_shape<bf16_t>(p, w, stream);
  return cb_by_shape<_Float16>(p, w, stream);
}

}  // namespace kch
