// The STE surrogate's backward for the CSA indexer (ops_csa.py:1033-1099) for
// gfx950, in fp32; queries, head weights and their gradients in their own
// storage type.
//
// soft = softmax over the visible blocks n of the indexer logits
//   lg_n = sum_h w_h relu(a_hn),  a_hn = scale qn_h . k_n
// (ops_csa.py:503-572); the selected columns of soft receive dsel (the slot
// gradients, scattered densely: 0 off the selection). Backward:
//   D = sum_n soft_n dsel_n,  dl_n = soft_n (dsel_n - D),
//   dw_h = sum_n dl_n relu(a_hn),  dqn_h = sum_n dl_n w_h [a_hn > 0] scale k_n,
//   dk_n = sum_t sum_h dl_tn w_th [a > 0] scale qn_th,
// then the L2-norm and compression backwards of the indexer keys
// (attn_bwd_finish.hip on the partials written here).
//
// Every sum over channels, blocks or queries is a contraction, and runs on the
// fp32 matrix instruction 16x16x4 (the same precision as the vector units):
// the (query, head) pairs are the 16 columns (rows) of a tile, a query's NIH
// heads side by side, so a tile holds 16 / NIH queries against 16 blocks.
//
// ste_bwd_query_kernel  four waves of 16 / NIH queries share the blocks' key
//   rows, 32 a step, double-buffered in LDS. A^T = K Qn^T leaves 4 blocks of
//   one (query, head) in each lane; the heads' sum is a DPP reduction over
//   adjacent lanes. Pass 1: lse and D with a running maximum; pass 2: dl, dw,
//   and dqn^T += K^T coef^T straight from the accumulator layout.
// ste_bwd_key_kernel    64 key rows (16 per wave, in registers) and a chunk of
//   queries, 32 (query, head) rows a step in LDS. A = Qn K^T leaves the heads
//   of a query in one lane (or two), so the softmax costs one exponential per
//   (query, block); dk += coef^T Qn. The chunk length follows the grid size:
//   long sequences take 512 queries a chunk, short ones as few as 64 so that
//   every compute unit has work.
// ste_scatter_kernel    the slots' values into the dense dsel.
//
// Bound: the fp32 matrix rate (157 TFLOP/s), of 5 products over the visible
// (query, head, block) triples. With one wave per query and 8 keys per thread
// on the vector units (a shuffle reduction per pair) the two kernels took
// 1002 + 921 us at B2 T4096, 4 heads of 64, 1024 blocks; now 178 + 108 us
// (10.8 GFLOP of products: 38 TFLOP/s over the two, the causal imbalance of
// the query kernel's workgroups and one exponential per lane being the rest).

#include "attn_common.h"
#include "kch_csa.h"
#include "kch_kernels.h"

namespace kch {

namespace {

constexpr int KT = 64;   // key rows per key-kernel workgroup
constexpr int KS = 32;   // key rows (query kernel) / (query, head) rows (key kernel) per step
constexpr float kEps = 1e-12f;

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// sum over the aligned groups of NIH adjacent lanes; every lane gets it
template <int NIH>
__device__ __forceinline__ float head_sum(float v) {
  if constexpr (NIH >= 2) v += dppf<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (NIH >= 4) v += dppf<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (NIH >= 8) v += dppf<0x141>(v);  // row_half_mirror: the other quad of the 8
  return v;
}

__device__ __forceinline__ f32x4 mma4(float4 a, const float* b, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], acc, 0, 0, 0);
}

// The gate [a > 0] jumps at zero. The two kernels sum a in the same order (the
// same channels a step; exchanging the operands changes no bit: 0 of 512000
// entries, half of them sums that cancel), so both take the same side. A score
// of unit rows that the matrix sum leaves at rounding level (0 < |qn.k| <
// kNearZero, about one in 10^5) is summed again in one fixed order, CPL-channel
// chains joined by a balanced tree, so that its side does not depend on the
// tiles' order of channels. A sum of exactly 0 stays: zero rows (a padded
// sequence) have nothing else, and summing each of their pairs again took 2380
// us where random rows take 420 (B2 T4096, 4 heads of 64, half of the queries
// zero; whole indexer backward). Raw rows keep the matrix sum.
constexpr float kNearZero = 2e-6f;

// four consecutive stored values as fp32
template <typename T>
__device__ __forceinline__ float4 load4(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const float4*>(p);
  } else {
    typedef T t4 __attribute__((ext_vector_type(4)));
    const t4 v = *reinterpret_cast<const t4*>(p);
    return make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
  }
}

template <int CPL, int N, typename T>
__device__ __forceinline__ float tree_dot(const T* q, float rq, const float* k) {
  if constexpr (N == 1) {
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < CPL; ++e) d = __builtin_fmaf((float)q[e] * rq, k[e], d);
    return d;
  } else {
    return tree_dot<CPL, N / 2, T>(q, rq, k) + tree_dot<CPL, N / 2, T>(q + N / 2 * CPL, rq, k + N / 2 * CPL);
  }
}
// sum of squares of v[0 .. N CPL) in the same order
template <int CPL, int N>
__device__ __forceinline__ float tree_sq(const float* v) {
  if constexpr (N == 1) {
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < CPL; ++e) d = __builtin_fmaf(v[e], v[e], d);
    return d;
  } else {
    return tree_sq<CPL, N / 2>(v) + tree_sq<CPL, N / 2>(v + N / 2 * CPL);
  }
}
// a[e] summed again where it is near but not zero; row(e): the query and key row of a[e]
template <int NIH, int CI, typename T, typename Rows>
__device__ __forceinline__ void settle_zero(f32x4& a, int normalize, Rows rows) {
  unsigned near = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) near |= a[e] != 0.f && fabsf(a[e]) < kNearZero ? 1u << e : 0u;
  if (!normalize) return;
  while (near) {
    const int e = __builtin_ctz(near);
    near &= near - 1;
    const T* q;
    const float* k;
    float rq;
    if (!rows(e, q, rq, k)) continue;
    const float d = tree_dot<CI * NIH / 64, 64 / NIH, T>(q, rq, k);
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = e == i ? d : a[i];
  }
}

template <int NIH, int CI, typename T>
__global__ __launch_bounds__(256) void ste_bwd_query_kernel(SteBwdParams p, int ntile) {
  constexpr int QPW = 16 / NIH, QPB = 4 * QPW;  // queries per wave, per workgroup
  constexpr int LD = CI + 4;                    // padded row: 16 rows' float4 reads free of conflicts
  constexpr int NP = KS * CI / 4 / 256;         // float4 pieces per thread per step
  constexpr int NT = CI / 16;
  __shared__ __attribute__((aligned(16))) float lds[2][KS * LD];
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, q = lane >> 4, n = lane & 15;
  // the latest queries see the most blocks: they start first
  const int b = blockIdx.x % p.B;
  const int t0 = (ntile - 1 - (int)(blockIdx.x / p.B)) * QPB;
  const int t = t0 + wv * QPW + n / NIH, h = n % NIH;
  const bool live = t < p.T;
  const size_t bt = (size_t)b * p.T + (live ? t : 0);
  const int nvis = live ? min((t + 1) / p.m, p.nb) : 0;
  const int nmax = min(min(t0 + QPB, p.T) / p.m, p.nb);  // of the workgroup's last query
  const int nsteps = (nmax + KS - 1) / KS;
  const bool vec = (p.nb & 3) == 0;

  // B operand: qn of this lane's (query, head), channels q CI/4 + j
  const T* qrow = static_cast<const T*>(p.qi) + (bt * NIH + h) * CI;
  float qv[CI / 4];
#pragma unroll
  for (int j = 0; j < CI / 16; ++j) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live) x = load4<T>(qrow + q * (CI / 4) + 4 * j);
    qv[4 * j] = x.x; qv[4 * j + 1] = x.y; qv[4 * j + 2] = x.z; qv[4 * j + 3] = x.w;
  }
  const float ss = tree_sq<CI * NIH / 64, 16 / NIH>(qv);
  const float nrm = sqrtf(colq_sum(ss));
  const float rq = p.normalize ? 1.f / fmaxf(nrm, kEps) : 1.f;
#pragma unroll
  for (int j = 0; j < CI / 4; ++j) qv[j] *= rq;
  const float wh = live ? (float)static_cast<const T*>(p.w)[bt * NIH + h] : 0.f;
  const float* dsel = p.dsel + bt * p.nb;
  const float* kc = p.kc + (size_t)b * p.nb * CI;

  // key rows of step s (rows past the last visible one read as zeros)
  auto fetch = [&](int s, float4 (&v)[NP]) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int pc = tid + 256 * i, row = KS * s + pc / (CI / 4), c = pc % (CI / 4);
      v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row < nmax) v[i] = *reinterpret_cast<const float4*>(kc + (size_t)row * CI + 4 * c);
    }
  };
  auto put = [&](float* buf, const float4 (&v)[NP]) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int pc = tid + 256 * i, row = pc / (CI / 4), c = pc % (CI / 4);
      *reinterpret_cast<float4*>(buf + row * LD + 4 * c) = v[i];
    }
  };
  // dsel of blocks 32 s + 16 u + 4 q + e
  auto load_ds = [&](int s, float (&d)[8]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int n0 = KS * s + 16 * u + 4 * q;
      if (vec) {
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        if (n0 < nvis) x = *reinterpret_cast<const float4*>(dsel + n0);
        d[4 * u] = x.x;
        d[4 * u + 1] = n0 + 1 < nvis ? x.y : 0.f;
        d[4 * u + 2] = n0 + 2 < nvis ? x.z : 0.f;
        d[4 * u + 3] = n0 + 3 < nvis ? x.w : 0.f;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) d[4 * u + e] = n0 + e < nvis ? dsel[n0 + e] : 0.f;
      }
    }
  };
  // a of the staged blocks 16 u + 4 q + e with this lane's (query, head)
  auto scores = [&](const float* buf, int u) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < CI / 16; ++j)
      a = mma4(*reinterpret_cast<const float4*>(buf + (16 * u + n) * LD + q * (CI / 4) + 4 * j), qv + 4 * j, a);
    settle_zero<NIH, CI, T>(a, p.normalize, [&](int e, const T*& qr, float& f, const float*& kr) {
      qr = qrow;
      f = rq;
      kr = buf + (16 * u + 4 * q + e) * LD;
      return live;
    });
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] *= p.scale;
    return a;
  };

  float4 kv[NP];
  float ds[8], dn[8];
  // ---- pass 1: lse and D, a running maximum per lane (merged over the blocks' lanes below) ----
  float m = -INFINITY, l = 0.f, ad = 0.f;
  if (nsteps > 0) {
    fetch(0, kv);
    load_ds(0, dn);
  }
  for (int s = 0; s < nsteps; ++s) {
    float* buf = lds[s & 1];
    put(buf, kv);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) ds[i] = dn[i];
    if (s + 1 < nsteps) {
      fetch(s + 1, kv);
      load_ds(s + 1, dn);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 a = scores(buf, u);
      float lg[4], mx = m;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = head_sum<NIH>(wh * fmaxf(a[e], 0.f));
        lg[e] = KS * s + 16 * u + 4 * q + e < nvis ? x : -INFINITY;
        mx = fmaxf(mx, lg[e]);
      }
      if (mx > m) {
        const float sc = expf(m - mx);  // m = -inf: 0
        l *= sc;
        ad *= sc;
        m = mx;
      }
      if (m > -INFINITY) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float e1 = expf(lg[e] - m);  // not visible: 0
          l += e1;
          ad += e1 * ds[4 * u + e];
        }
      }
    }
  }
  {
    const float mx = colq_max(m);
    const float sc = m > -INFINITY ? expf(m - mx) : 0.f;
    l = colq_sum(l * sc);
    ad = colq_sum(ad * sc);
    m = mx;
  }
  const float lse = l > 0.f ? m + logf(l) : INFINITY;
  const float D = l > 0.f ? ad / l : 0.f;

  // ---- pass 2 ----
  f32x4 dq[NT];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) dq[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float dwh = 0.f;
  if (nsteps > 0) {
    fetch(0, kv);
    load_ds(0, dn);
    __syncthreads();  // pass 1's last reads of lds[0] (one step) are done
  }
  for (int s = 0; s < nsteps; ++s) {
    float* buf = lds[s & 1];
    put(buf, kv);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) ds[i] = dn[i];
    if (s + 1 < nsteps) {
      fetch(s + 1, kv);
      load_ds(s + 1, dn);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4 a = scores(buf, u);
      float coef[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float r = fmaxf(a[e], 0.f);
        const float lg = head_sum<NIH>(wh * r);
        const float dl =
            KS * s + 16 * u + 4 * q + e < nvis ? expf(lg - lse) * (ds[4 * u + e] - D) : 0.f;
        dwh += dl * r;
        coef[e] = a[e] > 0.f ? dl * wh * p.scale : 0.f;
      }
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          dq[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(buf[(16 * u + 4 * q + e) * LD + 16 * tt + n],
                                                        coef[e], dq[tt], 0, 0, 0);
      }
    }
  }
  dwh = colq_sum(dwh);
  // L2-norm backward of the query row (lane: channels 16 tt + 4 q + e)
  f32x4 y[NT];
  float yd = 0.f;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live) x = load4<T>(qrow + 16 * tt + 4 * q);
    y[tt] = f32x4{x.x * rq, x.y * rq, x.z * rq, x.w * rq};
#pragma unroll
    for (int e = 0; e < 4; ++e) yd += y[tt][e] * dq[tt][e];
  }
  yd = colq_sum(yd);
  if (!live) return;
  const bool big = p.normalize && nrm > kEps;
  T* dst = static_cast<T*>(p.dqi) + (bt * NIH + h) * CI;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (big ? dq[tt][e] - y[tt][e] * yd : dq[tt][e]) * rq;
    Store4<T>::run(dst + 16 * tt + 4 * q, f32x4{o[0], o[1], o[2], o[3]}, 1.f);
  }
  if (q == 0) {
    static_cast<T*>(p.dw)[bt * NIH + h] = (T)dwh;
    p.rq[bt * NIH + h] = rq;
    if (h == 0) {
      p.lse[bt] = lse;
      p.dval[bt] = D;
    }
  }
}

template <int NIH, int CI, typename T>
__global__ __launch_bounds__(256) void ste_bwd_key_kernel(SteBwdParams p, int qc, int nchunk) {
  constexpr int LD = CI + 4;
  constexpr int NP = KS * CI / 4 / 256;
  constexpr int NT = CI / 16;
  constexpr int QPS = KS / NIH;                  // queries per step
  constexpr int NQL = NIH >= 4 ? 1 : 4 / NIH;    // queries in a lane's four rows
  __shared__ __attribute__((aligned(16))) float lds[2][KS * LD];
  __shared__ __attribute__((aligned(16))) float sw[2][KS], sl[2][KS], sd[2][KS];  // w, lse, D per row
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, q = lane >> 4, n = lane & 15;
  const int b = blockIdx.y;
  const int tile = blockIdx.x / nchunk, ci = blockIdx.x - tile * nchunk;
  const int r0 = tile * KT;
  const int thi = min(p.T, (ci + 1) * qc);
  const int tvis = (r0 + 1) * p.m - 1;  // the first query that sees row r0
  if (tvis >= thi) return;  // no row of the tile is seen by this chunk (nothing to read back)
  const int ts0 = max(ci * qc, tvis / QPS * QPS);  // chunks are whole steps
  const int rk = r0 + 16 * wv + n;
  const bool rk_ok = rk < p.nb;
  const int tk = rk_ok ? (rk + 1) * p.m - 1 : p.T;   // the first query that sees row rk
  const int twave = (r0 + 16 * wv + 1) * p.m - 1;    // ... any row of this wave

  // B operand: key row rk, channels q CI/4 + j
  float kv[CI / 4];
#pragma unroll
  for (int j = 0; j < CI / 16; ++j) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (rk_ok) x = *reinterpret_cast<const float4*>(p.kc + ((size_t)b * p.nb + rk) * CI + q * (CI / 4) + 4 * j);
    kv[4 * j] = x.x; kv[4 * j + 1] = x.y; kv[4 * j + 2] = x.z; kv[4 * j + 3] = x.w;
  }
  f32x4 dk[NT];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) dk[tt] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Step {
    float4 v[NP];
    float w, l, d;
    float ds[2][NQL];
  };
  auto fetch = [&](int ts, Step& x) {
    const size_t row0 = ((size_t)b * p.T + ts) * NIH;
    const int live = (thi - ts) * NIH;  // rows of queries before thi
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int pc = tid + 256 * i, row = pc / (CI / 4), c = pc % (CI / 4);
      x.v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row < live) {
        const float f = p.rq[row0 + row];
        const float4 y = load4<T>(static_cast<const T*>(p.qi) + (row0 + row) * CI + 4 * c);
        x.v[i] = make_float4(y.x * f, y.y * f, y.z * f, y.w * f);
      }
    }
    x.w = x.l = x.d = 0.f;
    if (tid < KS && tid < live) {
      x.w = (float)static_cast<const T*>(p.w)[row0 + tid];
      x.l = p.lse[(size_t)b * p.T + ts + tid / NIH];
      x.d = p.dval[(size_t)b * p.T + ts + tid / NIH];
    }
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int i = 0; i < NQL; ++i) {
        const int t = ts + (16 * g + 4 * q) / NIH + i;
        x.ds[g][i] = t >= tk && t < thi ? p.dsel[((size_t)b * p.T + t) * p.nb + rk] : 0.f;
      }
  };
  auto put = [&](int k, const Step& x) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int pc = tid + 256 * i, row = pc / (CI / 4), c = pc % (CI / 4);
      *reinterpret_cast<float4*>(&lds[k][row * LD + 4 * c]) = x.v[i];
    }
    if (tid < KS) {
      sw[k][tid] = x.w;
      sl[k][tid] = x.l;
      sd[k][tid] = x.d;
    }
  };

  Step x;
  fetch(ts0, x);
  int k = 0;
  for (int ts = ts0; ts < thi; ts += QPS, k ^= 1) {
    put(k, x);
    __syncthreads();
    float ds[2][NQL];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int i = 0; i < NQL; ++i) ds[g][i] = x.ds[g][i];
    if (ts + QPS < thi) fetch(ts + QPS, x);
    if (ts + QPS > twave) {
      const float* buf = lds[k];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        // rows (query, head) 16 g + 4 q + e against key rk
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < CI / 16; ++j)
          a = mma4(*reinterpret_cast<const float4*>(buf + (16 * g + n) * LD + q * (CI / 4) + 4 * j), kv + 4 * j, a);
        const int r = 16 * g + 4 * q;
        settle_zero<NIH, CI, T>(a, p.normalize, [&](int e, const T*& qr, float& f, const float*& kr) {
          const size_t row = ((size_t)b * p.T + ts) * NIH + r + e;
          const bool ok = rk_ok && ts + (r + e) / NIH < thi;
          qr = static_cast<const T*>(p.qi) + (ok ? row * CI : 0);
          f = ok ? p.rq[row] : 0.f;
          kr = p.kc + ((size_t)b * p.nb + (rk_ok ? rk : 0)) * CI;
          return ok;
        });
        const float4 w4 = *reinterpret_cast<const float4*>(&sw[k][r]);
        const float w[4] = {w4.x, w4.y, w4.z, w4.w};
        float part[4], lg[NQL];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] *= p.scale;
          part[e] = w[e] * fmaxf(a[e], 0.f);
        }
#pragma unroll
        for (int i = 0; i < NQL; ++i) {
          lg[i] = part[i * (4 / NQL)];
#pragma unroll
          for (int e = 1; e < 4 / NQL; ++e) lg[i] += part[i * (4 / NQL) + e];
          if constexpr (NIH == 8) lg[i] += __shfl_xor(lg[i], 16);
        }
        float coef[4];
#pragma unroll
        for (int i = 0; i < NQL; ++i) {
          const int t = ts + r / NIH + i;
          const float dl = t >= tk && t < thi
                               ? expf(lg[i] - sl[k][r + i * NIH]) * (ds[g][i] - sd[k][r + i * NIH])
                               : 0.f;
#pragma unroll
          for (int e = 0; e < 4 / NQL; ++e) {
            const int j = i * (4 / NQL) + e;
            coef[j] = a[j] > 0.f ? dl * w[j] * p.scale : 0.f;
          }
        }
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            dk[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(coef[e], buf[(r + e) * LD + 16 * tt + n], dk[tt], 0, 0, 0);
        }
      }
    }
  }
  // lane: key rows 16 wv + 4 q + e, channels 16 tt + n
  float* out = p.part + (((size_t)b * nchunk + ci) * p.nb) * CI;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = r0 + 16 * wv + 4 * q + e;
    if (r < p.nb) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) out[(size_t)r * CI + 16 * tt + n] = dk[tt][e];
    }
  }
}

// dsel[row, idx[row, j]] += slot[row, j] (idx < 0: unused slot)
__global__ __launch_bounds__(256) void ste_scatter_kernel(const int* idx, const float* slot, float* dsel,
                                                          long long n, int topk, int nb) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int k = idx[i];
  if (k >= 0 && k < nb) unsafeAtomicAdd(dsel + i / topk * nb + k, slot[i]);
}

size_t al256(size_t x) { return (x + 255) & ~size_t(255); }

// Queries per chunk of the key kernel: 512, halved while the grid would leave
// compute units without a workgroup (half of the causal grid is empty).
int ste_chunk(int B, int T, int nb) {
  const int ntile = (nb + KT - 1) / KT;
  int qc = 512;
  while (qc > 64 && (long long)ntile * ((T + qc - 1) / qc) * B < 1024) qc /= 2;
  return qc;
}

template <int NIH, int CI, typename T>
hipError_t launch_ste(const SteBwdParams& p, const BwdFinish& f, hipStream_t s) {
  const int qpb = 64 / NIH, nt = (p.T + qpb - 1) / qpb;
  hipLaunchKernelGGL((ste_bwd_query_kernel<NIH, CI, T>), dim3((unsigned)((long long)nt * p.B)), dim3(256), 0, s, p,
                     nt);
  if (p.nb > 0)
    hipLaunchKernelGGL((ste_bwd_key_kernel<NIH, CI, T>), dim3((p.nb + KT - 1) / KT * f.nchunk, p.B), dim3(256), 0, s,
                       p, f.part_qc, f.nchunk);
  return hipGetLastError();
}

}  // namespace

size_t ste_bwd_ws_bytes(int B, int T, int nIh, int cI, int m) {
  const int nb = T / m, qc = ste_chunk(B, T, nb);
  return 2 * al256((size_t)B * T * 4) + al256((size_t)B * T * nIh * 4) +
         al256((size_t)B * ((T + qc - 1) / qc) * nb * cI * 4) + al256((size_t)B * T * cI * 4) +
         sum_rows_ws_bytes((long long)B * nb, m * cI);
}

hipError_t ste_bwd_dispatch(SteBwdParams p, BwdFinish f, void* ws, hipStream_t stream) {
  char* w = static_cast<char*>(ws);
  const size_t per = al256((size_t)p.B * p.T * 4);
  f.part_qc = ste_chunk(p.B, p.T, p.nb);
  f.nchunk = (p.T + f.part_qc - 1) / f.part_qc;
  p.lse = reinterpret_cast<float*>(w);
  p.dval = reinterpret_cast<float*>(w + per);
  p.rq = reinterpret_cast<float*>(w + 2 * per);
  w += 2 * per + al256((size_t)p.B * p.T * p.nIh * 4);
  p.part = reinterpret_cast<float*>(w);
  f.part_b = p.part;
  w += al256((size_t)p.B * f.nchunk * p.nb * p.cI * 4);
  f.dBp = reinterpret_cast<float*>(w);
  w += al256((size_t)p.B * p.T * p.cI * 4);
  hipError_t e = hipErrorInvalidValue;
#define KCH_STE(NIH, CI)                                                    \
  if (p.nIh == NIH && p.cI == CI)                                           \
    e = p.qdt == DT_BF16  ? launch_ste<NIH, CI, bf16_t>(p, f, stream)       \
        : p.qdt == DT_F16 ? launch_ste<NIH, CI, _Float16>(p, f, stream)     \
                          : launch_ste<NIH, CI, float>(p, f, stream);
  KCH_STE(1, 64) KCH_STE(1, 128) KCH_STE(2, 64) KCH_STE(2, 128) KCH_STE(4, 64) KCH_STE(4, 128)
  KCH_STE(8, 64)
#undef KCH_STE
  // compression and L2-norm backward of the indexer keys
  if (e == hipSuccess) e = bwd_finish_launch(f, p.cI, stream);
  if (e == hipSuccess) e = sum_rows_launch(f.dBp, p.dB, (long long)p.B * p.nb, p.m * p.cI, 1.f, w, stream);
  return e;
}

hipError_t ste_scatter_launch(const int* idx, const float* slot, float* dsel, long long rows, int topk, int nb,
                              hipStream_t s) {
  const long long k = rows * topk;
  if (k == 0) return hipSuccess;
  hipLaunchKernelGGL(ste_scatter_kernel, dim3((unsigned)((k + 255) / 256)), dim3(256), 0, s, idx, slot, dsel, k,
                     topk, nb);
  return hipGetLastError();
}

}  // namespace kch
