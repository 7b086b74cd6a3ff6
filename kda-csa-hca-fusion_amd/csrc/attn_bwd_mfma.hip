// Attention backward on MFMA for gfx950: the gradients of the joint
// softmax over compressed rows (HCA: every causal block; CSA: the selected
// blocks), window rows and the sink, with L2-normalised queries and keys
// (normalize_qk=True, |score| <= scale). Same algebra as the SIMT kernels of
// hca_backward.hip (ops_hca.py:132-194, ops_csa.py:869-1155 under autograd):
//   s = scale qn.k,  p = exp(s - lse),  dp = dout.k,  D = sum p dp,
//   ds = p (dp - D),  dqn = scale sum ds k,  dk += scale ds qn + p dout.
//
// Every operand that is not bf16 already is a two-part bf16 split x = hi + lo
// (2^-16 relative); a product takes the MFMAs hi*hi + hi*lo + lo*hi of the
// parts that exist, accumulated in fp32. Queries and dout enter as they are
// given, with 1/|q| applied to the scores in fp32 (and to ds for dk): bf16
// ones are exact in one part, so a product with a split key takes two MFMAs
// and no split copy of them is ever written; fp16 / fp32 ones are split while
// they are staged. The window rows enter the same way (1/|x| in fp32): with
// bf16 queries and rows their products take one MFMA. The compressed rows,
// fp32 sums, are split once by split_rows_kernel.
//
// attn_bwd_qt_kernel  a workgroup of 4 waves and 8 (bf16) or 4 consecutive
//   queries, all 16 heads as the MFMA columns (MQA: every key row is shared by
//   the heads). The queries' key rows (every visible block, masked by the
//   selection bitmap for CSA, then the window rows) are staged in LDS 32 rows
//   a step, once for the workgroup, double-buffered, and each K fragment read
//   serves the wave's two queries: S^T = K Q^T and dP^T = K dout^T per 16
//   rows. Pass 1: lse and D with a running maximum per lane; pass 2: ds, and
//   dqn^T += K^T ds^T (K^T fragments from the transposing LDS read, ds^T from
//   the accumulators, as the forward's O^T = V^T P^T). Writes dq (after the
//   L2-norm backward), 1/|q|, lse, D, and for CSA each selected block's
//   gradient dotted with its row (dense, dsel) and their sum gsum.
// attn_bwd_q_kernel   CSA over long contexts: one wave per query gathers only
//   the selected rows, 32 a step, into its own LDS stage. Its bound is the L2
//   gather of 512 bytes a row and pass (8.5 TB/s measured), the tile kernel's
//   the matrix cores; see attn_bwd_dense_rows for where the line lies. The
//   slots' values go where they are asked for: slot by slot, or into the
//   query's own row of dsel, which the wave clears first.
// attn_bwd_k_kernel   one workgroup per 64 KG key rows (16 KG per wave, KG 1 or
//   2, key fragments in registers) and chunk of queries; queries are taken in
//   pairs: the pair's q and dout rows (32 rows of (query, head)) are staged in
//   LDS once for the four waves (double-buffered), S = Q K^T and dP = dout K^T
//   per query, then dk += ds^T Q + p^T dout with (query, head) as the
//   contraction (the accumulators of the two queries' S are the A operand in
//   the packed order of the transposing read of Q / dout). Every fragment read
//   serves KG groups of 16 keys. Writes per-chunk partials of the compressed
//   rows and of the window rows; the chunk length follows the grid size.
// The L2-norm and compression backwards follow on these partials
// (attn_bwd_finish.hip).
//
// Measured, 16 heads of 128, window 128, bf16, against one wave per query with
// its own copy of every row and 16 keys per wave on three-MFMA products: HCA
// B2 T8192 (64 blocks) query pass 254 -> 168 us, window keys 233 -> 105,
// compressed keys 625 (32 workgroups) -> 62, splits of q and dout 68 -> 0; CSA
// B2 T4096 top-512 (1024 blocks) query pass 565 -> 305, compressed keys 677 ->
// 253, window keys 197 -> 71. (The window rows in two parts: 211, 150 and 349,
// 114.)

#include "attn_common.h"
#include "kch_csa.h"
#include "kch_kernels.h"

namespace kch {

namespace {

constexpr float kLn2F = 0.6931471805599453f;

__device__ __forceinline__ bf16_t lo_of(float x) { return (bf16_t)(x - (float)(bf16_t)x); }

// acc + a * b with b exactly bf16 (its low part zero): al*bh + ah*bh
__device__ __forceinline__ f32x4 mfma2a(const bf16x8& ah, const bf16x8& al, const bf16x8& bh, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
}
// acc + a * b with a exactly bf16: ah*bl + ah*bh
__device__ __forceinline__ f32x4 mfma2b(const bf16x8& ah, const bf16x8& bh, const bf16x8& bl, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma3(const bf16x8& ah, const bf16x8& al, const bf16x8& bh,
                                       const bf16x8& bl, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
}

// Four consecutive elements at element offset off of a row stored in dt
// (DT_F32 / DT_BF16 / DT_F16), as fp32, and the rounded store of four.
__device__ __forceinline__ float4 load4(const void* base, long long off, int dt) {
  if (dt == DT_F32) return *reinterpret_cast<const float4*>(static_cast<const float*>(base) + off);
  const uint2 r = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + off);
  if (dt == DT_BF16)
    return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u),
                       __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  const h4 h = __builtin_bit_cast(h4, r);
  return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
}
__device__ __forceinline__ void store4(void* base, long long off, float4 v, int dt) {
  if (dt == DT_F32) {
    *reinterpret_cast<float4*>(static_cast<float*>(base) + off) = v;
  } else if (dt == DT_BF16) {
    bf16x4 h = {(bf16_t)v.x, (bf16_t)v.y, (bf16_t)v.z, (bf16_t)v.w};
    *reinterpret_cast<bf16x4*>(static_cast<bf16_t*>(base) + off) = h;
  } else {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    h4 h = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    *reinterpret_cast<h4*>(static_cast<_Float16*>(base) + off) = h;
  }
}

// Rows of HD fp32 values as bf16 hi / lo rows (x = hi + lo): the compressed
// rows, 8 values a lane.
template <int HD>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* x, long long rows, bf16_t* hi, bf16_t* lo) {
  constexpr int LPR = HD / 8;  // lanes per row
  const long long r = (long long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (r >= rows) return;
  const long long o = r * HD + 8 * (threadIdx.x % LPR);
  float v[8];
  Load8<float>::run(x + o, v);
  bf16x8 h, l;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    h[i] = (bf16_t)v[i];
    l[i] = lo_of(v[i]);
  }
  *reinterpret_cast<bf16x8*>(hi + o) = h;
  *reinterpret_cast<bf16x8*>(lo + o) = l;
}

// The window rows' 1 / max(|row|, 1e-12) and, where asked for, the splits of
// the rows as given (hi, lo) and normalised (nhi, nlo). Rows ld elements apart
// in, contiguous out.
template <int HD, typename T>
__global__ __launch_bounds__(256) void window_rows_kernel(const T* x, long long ld, long long rows, float* rl,
                                                          bf16_t* hi, bf16_t* lo, bf16_t* nhi, bf16_t* nlo) {
  constexpr int LPR = HD / 8;
  const long long r = (long long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const int lc = threadIdx.x % LPR;
  const bool act = r < rows;  // no early return: the row sum shuffles
  float v[8];
  Load8<T>::run(x + (act ? r : 0) * ld + 8 * lc, v);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss += v[i] * v[i];
#pragma unroll
  for (int m = LPR / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
  if (!act) return;
  const float f = l2_inv(ss);
  if (lc == 0) rl[r] = f;
  auto split = [&](bf16_t* h, bf16_t* l, float g) {
    bf16x8 a, b;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i] = (bf16_t)(v[i] * g);
      b[i] = lo_of(v[i] * g);
    }
    *reinterpret_cast<bf16x8*>(h + r * HD + 8 * lc) = a;
    *reinterpret_cast<bf16x8*>(l + r * HD + 8 * lc) = b;
  };
  if (hi) split(hi, lo, 1.f);
  if (nhi) split(nhi, nlo, f);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// sum over the 16 lanes of a DPP row; every lane of the row gets the total
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f<0x141>(v);  // row_half_mirror: the other quad of the 8
  v += dpp_f<0x140>(v);  // row_mirror: the other 8 of the row
  return v;
}

// Eight stored values of a query or dout row as bf16 parts: one (exact) for
// bf16, hi + lo for fp16 and fp32.
template <typename QT>
struct Parts {
  static constexpr bool one = std::is_same<QT, bf16_t>::value;
};
template <typename QT>
__device__ __forceinline__ void load_parts(const QT* p, bool ok, bf16x8& h, bf16x8& l, float& ss) {
  float v[8];
  if (ok) {
    Load8<QT>::run(p, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ss += v[i] * v[i];
    h[i] = (bf16_t)v[i];
    if constexpr (!Parts<QT>::one) l[i] = lo_of(v[i]);
  }
}
// acc + k * x, k split (kh, kl), x in one part (exact) or two
template <bool ONE>
__device__ __forceinline__ f32x4 mma_kx(const bf16x8& kh, const bf16x8& kl, const bf16x8& xh, const bf16x8& xl,
                                        f32x4 acc) {
  if constexpr (ONE) return mfma2a(kh, kl, xh, acc);
  else return mfma3(kh, kl, xh, xl, acc);
}
// acc + x * k
template <bool ONE>
__device__ __forceinline__ f32x4 mma_xk(const bf16x8& xh, const bf16x8& xl, const bf16x8& kh, const bf16x8& kl,
                                        f32x4 acc) {
  if constexpr (ONE) return mfma2b(xh, kh, kl, acc);
  else return mfma3(xh, xl, kh, kl, acc);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int HD>
struct QWave {
  static constexpr int NS = HD / 32, NT = HD / 16;
  static constexpr int TPR = HD / 8, RPI = 64 / TPR, NLI = 32 / RPI;
  struct Rows {
    u32x4 h[NLI], l[NLI];
  };
};

// The end of a query's pass: the L2-norm backward of qn and the stores of dq,
// lse, D, 1/|q| and the sink term (lane: head n, dims 16 tt + 4 q + e).
template <int HD>
__device__ __forceinline__ void finish_query(const HcaBwdParams& p, size_t bt, int n, int q, f32x4 (&dq)[HD / 16],
                                             float rq, float lse2, float D, float sk2) {
  constexpr int NT = HD / 16;
  float qv[NT][4];
  float yd = 0.f;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (n < p.nh) x = load4(p.q, (bt * p.nh + n) * HD + 16 * tt + 4 * q, p.qdt);
    qv[tt][0] = x.x * rq; qv[tt][1] = x.y * rq; qv[tt][2] = x.z * rq; qv[tt][3] = x.w * rq;
#pragma unroll
    for (int e = 0; e < 4; ++e) yd += qv[tt][e] * dq[tt][e];
  }
  yd = colq_sum(yd);
  if (n < p.nh) {
    // rq = 1 / max(|q|, eps): for |q| <= eps the norm is the constant eps
    const bool big = rq < 1e12f;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (big ? dq[tt][e] - qv[tt][e] * yd : dq[tt][e]) * rq;
      store4(p.dq, (bt * p.nh + n) * HD + 16 * tt + 4 * q, make_float4(o[0], o[1], o[2], o[3]), p.qdt);
    }
  }
  if (q == 0) {
    p.lse[bt * 16 + n] = lse2;
    p.dval[bt * 16 + n] = D;
    p.rq[bt * 16 + n] = n < p.nh ? rq : 0.f;
    if (p.sink_part && n < p.nh) p.sink_part[bt * p.nh + n] = p.sink ? fast_exp2(sk2 - lse2) * D : 0.f;
  }
}

// gsum = sum over the heads of dssel qn + psel dout (dims 32 s + 8 q + i). The
// rows are read again: kept as fp32 across the passes they spill.
template <int HD, typename QT>
__device__ __forceinline__ void store_gsum(const HcaBwdParams& p, size_t bt, int n, int q, float psel, float dssel,
                                           float rq) {
  psel = colq_sum(psel);
  dssel = colq_sum(dssel) * rq;
  const bool ok = n < p.nh;
  const size_t ro = ok ? (bt * p.nh + n) * HD + 8 * q : 0;
#pragma unroll
  for (int s = 0; s < HD / 32; ++s) {
    float qv[8], dv[8], gv[8];
    Load8<QT>::run(static_cast<const QT*>(p.q) + ro + 32 * s, qv);
    Load8<QT>::run(static_cast<const QT*>(p.dout) + ro + 32 * s, dv);
#pragma unroll
    for (int i = 0; i < 8; ++i) gv[i] = row16_sum(ok ? dssel * qv[i] + psel * dv[i] : 0.f);
    if (n == 0) {
      float* dst = p.gsum + bt * HD + 32 * s + 8 * q;
      *reinterpret_cast<float4*>(dst) = make_float4(gv[0], gv[1], gv[2], gv[3]);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(gv[4], gv[5], gv[6], gv[7]);
    }
  }
}

// lse (log2 units) and D of a head from its four lanes' running m, l, ad and the sink
struct Soft {
  float lse2, D, sk2;
};
__device__ __forceinline__ Soft close_softmax(const HcaBwdParams& p, int n, float m, float l, float ad) {
  const float mx = colq_max(m);
  const float f = m > -INFINITY ? fast_exp2(m - mx) : 0.f;
  l = colq_sum(l * f);
  ad = colq_sum(ad * f);
  m = mx;
  Soft r;
  r.sk2 = -INFINITY;
  if (p.sink && n < p.nh) r.sk2 = p.sink[n] * kLog2eF;
  if (r.sk2 > -INFINITY) {
    const float mn = fmaxf(m, r.sk2);
    const float a = fast_exp2(m - mn);
    l = l * a + fast_exp2(r.sk2 - mn);
    ad *= a;
    m = mn;
  }
  const bool live = n < p.nh && l > 0.f;
  r.lse2 = live ? m + __log2f(l) : INFINITY;
  r.D = live ? ad / l : 0.f;
  return r;
}
// one step of eight scores (log2 units, -inf: masked) and dp into m, l, ad
__device__ __forceinline__ void soft_step(const float (&s8)[8], const float (&d8)[8], float& m, float& l, float& ad) {
  float mx = s8[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s8[e]);
  if (mx > m) {
    const float a = fast_exp2(m - mx);  // m = -inf: a = 0
    l *= a;
    ad *= a;
    m = mx;
  }
  if (m > -INFINITY) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float pe = fast_exp2(s8[e] - m);  // masked: 0
      l += pe;
      ad += pe * d8[e];
    }
  }
}

// --------------------------------------------------- query pass, rows in tiles
// KX: the window rows are exact in one part (bf16 rows and queries).
template <int HD, typename QT, bool SEL, bool KX>
__global__ __launch_bounds__(256, 2) void attn_bwd_qt_kernel(HcaBwdParams p, int ntile) {
  constexpr bool ONE = Parts<QT>::one;
  constexpr int QW = ONE ? 2 : 1;             // queries per wave
  constexpr int NS = HD / 32, NT = HD / 16;
  constexpr int TILE = 32 * HD, CPR = HD / 8;
  constexpr int LPT = 2 * TILE / 8 / 256;     // 16-byte pieces per thread per step
  __shared__ __attribute__((aligned(16))) bf16_t lds[2][2 * TILE];  // hi, lo
  __shared__ __attribute__((aligned(16))) float srl[2][32];         // the rows' factors: 1, or 1/|x| (window)
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, q = lane >> 4, n = lane & 15;
  // the latest queries see the most blocks: they start first
  const int b = blockIdx.x % p.B;
  const int t0 = (ntile - 1 - (int)(blockIdx.x / p.B)) * 4 * QW;
  const int tlast = min(t0 + 4 * QW, p.T) - 1;
  const int t1 = t0 + wv * QW;                // this wave's queries t1 .. t1 + QW - 1
  const TileOffsets<HD> to;

  // B operands: q and dout of head n, dims 32s + 8q .. (16 heads, padded rows zero)
  bf16x8 qh[QW][NS], ql[QW][ONE ? 1 : NS], dh[QW][NS], dl[QW][ONE ? 1 : NS];
  float rq[QW], scq[QW];
  int nv[QW];
#pragma unroll
  for (int i = 0; i < QW; ++i) {
    const bool ok = t1 + i < p.T && n < p.nh;
    const size_t ro = ok ? (((size_t)b * p.T + t1 + i) * p.nh + n) * HD + 8 * q : 0;
    float ss = 0.f, unused = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      load_parts<QT>(static_cast<const QT*>(p.q) + ro + 32 * s, ok, qh[i][s], ql[i][ONE ? 0 : s], ss);
      load_parts<QT>(static_cast<const QT*>(p.dout) + ro + 32 * s, ok, dh[i][s], dl[i][ONE ? 0 : s], unused);
    }
    rq[i] = l2_inv(colq_sum(ss));
    scq[i] = rq[i] * p.scale * kLog2eF;  // raw score -> log2 units
    nv[i] = min((t1 + i + 1) / p.m2, p.nb);
  }
  const int nvm = SEL && p.topk == 0 ? 0 : min((tlast + 1) / p.m2, p.nb);
  const int nsc = (nvm + 31) / 32;
  // window steps start at whole 32-row groups: the rows summed together, and so
  // the bits, do not depend on how many queries share the workgroup
  const int w0 = max(0, t0 - p.win + 1) & ~31;
  const int nwin = p.win > 0 ? tlast - w0 + 1 : 0;
  const int nsteps = nsc + (nwin + 31) / 32;
  const int nw = (p.nb + 31) / 32;

  // the 32 rows of step m (hi and lo planes; rows past the end read as zeros)
  struct Rows {
    u32x4 v[LPT];
    float f;
  };
  auto fetch = [&](int m, Rows& x) {
    const bool comp = m < nsc;
    const int r0 = comp ? 32 * m : 32 * (m - nsc);
    const int lim = comp ? nvm : nwin;
    const size_t base = comp ? (size_t)b * p.nb : (size_t)b * p.T + w0;
    const long long ld = comp ? HD : p.ldl;
    const bf16_t* hi = comp ? p.kc_hi : p.kl_hi;
    const bf16_t* lo = comp ? p.kc_lo : p.kl_lo;
#pragma unroll
    for (int k = 0; k < LPT; ++k) {
      const int pc = tid + 256 * k, w = pc % (32 * CPR), row = w / CPR, c = w % CPR;
      if (KX && k >= LPT / 2 && !comp) break;  // the rows' low parts are zero
      const bf16_t* src = pc < 32 * CPR ? hi : lo;
      x.v[k] = u32x4{0, 0, 0, 0};
      if (r0 + row < lim) x.v[k] = *reinterpret_cast<const u32x4*>(src + (base + r0 + row) * ld + 8 * c);
    }
    x.f = 1.f;
    if (tid < 32 && !comp) x.f = r0 + tid < lim ? p.rl[base + r0 + tid] : 0.f;
  };
  auto put = [&](int k2, int m, const Rows& x) {
#pragma unroll
    for (int k = 0; k < LPT; ++k) {
      const int pc = tid + 256 * k, w = pc % (32 * CPR), row = w / CPR, c = w % CPR;
      if (KX && k >= LPT / 2 && m >= nsc) break;
      *reinterpret_cast<u32x4*>(lds[k2] + (pc / (32 * CPR)) * TILE + row * HD + 8 * (c ^ tile_swz<HD>(row & 15))) =
          x.v[k];
    }
    if (tid < 32) srl[k2][tid] = x.f;
  };
  // the selection's word of step m (uniform per query)
  auto load_word = [&](int m, uint32_t (&w)[QW]) {
#pragma unroll
    for (int i = 0; i < QW; ++i)
      w[i] = m < nsc && t1 + i < p.T ? p.sel[((size_t)b * p.T + t1 + i) * nw + m] : 0u;
  };
  // S^T (log2 units, masked) and dP^T of the staged rows of step m (comp: block
  // rows, else window rows): keys 4q+e, 16+4q+e of head n
  auto scores = [&](auto comp_, int m, const uint32_t (&sw)[QW], float (&s8)[QW][8], float (&d8)[QW][8]) {
    constexpr bool comp = decltype(comp_)::value;
    const bf16_t* kt = lds[m & 1];
    const int r0 = comp ? 32 * m : 32 * (m - nsc);
    const int lim = comp ? nvm : nwin;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 sa[QW], da[QW];
#pragma unroll
      for (int i = 0; i < QW; ++i) sa[i] = da[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      // (rows past the last query's, or before the first query's window)
      if (r0 + 16 * half < lim && (comp || w0 + r0 + 16 * half + 15 > t0 - p.win)) {
        const bf16_t* kr = kt + 16 * HD * half;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const bf16x8 kh = *reinterpret_cast<const bf16x8*>(kr + to.key(s));
          if constexpr (KX && !comp) {
#pragma unroll
            for (int i = 0; i < QW; ++i) {
              sa[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, qh[i][s], sa[i], 0, 0, 0);
              da[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kh, dh[i][s], da[i], 0, 0, 0);
            }
          } else {
            const bf16x8 kl = *reinterpret_cast<const bf16x8*>(kr + TILE + to.key(s));
#pragma unroll
            for (int i = 0; i < QW; ++i) {
              sa[i] = mma_kx<ONE>(kh, kl, qh[i][s], ql[i][ONE ? 0 : s], sa[i]);
              da[i] = mma_kx<ONE>(kh, kl, dh[i][s], dl[i][ONE ? 0 : s], da[i]);
            }
          }
        }
      }
      float f[4] = {1.f, 1.f, 1.f, 1.f};
      if constexpr (!comp) {
        const float4 f4 = *reinterpret_cast<const float4*>(&srl[m & 1][16 * half + 4 * q]);
        f[0] = f4.x; f[1] = f4.y; f[2] = f4.z; f[3] = f4.w;
      }
#pragma unroll
      for (int i = 0; i < QW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = r0 + 16 * half + 4 * q + e;
          bool ok;
          if (comp) ok = SEL ? (sw[i] >> (16 * half + 4 * q + e)) & 1u : j < nv[i];
          else ok = (w0 + j <= t1 + i) & (w0 + j > t1 + i - p.win);
          s8[i][4 * half + e] = ok ? sa[i][e] * (scq[i] * f[e]) : -INFINITY;
          d8[i][4 * half + e] = da[i][e] * f[e];
        }
    }
  };

  Rows pv;
  uint32_t sw[QW] = {}, swn[QW] = {};
  // the staged rows of step m to LDS, the next step's requested
  auto begin = [&](int m) {
    put(m & 1, m, pv);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < QW; ++i) sw[i] = swn[i];
    if (m + 1 < nsteps) {
      fetch(m + 1, pv);
      if constexpr (SEL) load_word(m + 1, swn);
    }
  };
  typedef std::integral_constant<bool, true> Comp;
  typedef std::integral_constant<bool, false> Win;
  float m_[QW], l_[QW], ad_[QW];
#pragma unroll
  for (int i = 0; i < QW; ++i) {
    m_[i] = -INFINITY;
    l_[i] = ad_[i] = 0.f;
  }
  // ---- pass 1: lse and D ----
  if (nsteps > 0) {
    fetch(0, pv);
    if constexpr (SEL) load_word(0, swn);
  }
  auto pass1 = [&](auto comp_, int m) {
    begin(m);
    float s8[QW][8], d8[QW][8];
    scores(comp_, m, sw, s8, d8);
#pragma unroll
    for (int i = 0; i < QW; ++i) soft_step(s8[i], d8[i], m_[i], l_[i], ad_[i]);
  };
  for (int m = 0; m < nsc; ++m) pass1(Comp{}, m);
  for (int m = nsc; m < nsteps; ++m) pass1(Win{}, m);
  Soft sf[QW];
#pragma unroll
  for (int i = 0; i < QW; ++i) sf[i] = close_softmax(p, n, m_[i], l_[i], ad_[i]);

  // ---- pass 2: ds, dqn^T += K^T ds^T, the selected rows' terms ----
  f32x4 dq[QW][NT];
#pragma unroll
  for (int i = 0; i < QW; ++i)
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) dq[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float psel[QW] = {}, dssel[QW] = {};  // sums over the selected rows (gsum)
  if (nsteps > 0) {
    fetch(0, pv);
    if constexpr (SEL) load_word(0, swn);
    __syncthreads();  // pass 1's last reads are done
  }
  auto pass2 = [&](auto comp_, int m) {
    constexpr bool comp = decltype(comp_)::value;
    begin(m);
    float s8[QW][8], d8[QW][8];
    scores(comp_, m, sw, s8, d8);
    const bf16_t* kt = lds[m & 1];
    bf16x8 bh[QW], bl[QW];  // ds^T, times the rows' factors
    float f[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
    if constexpr (!comp) {
      const float4 x = *reinterpret_cast<const float4*>(&srl[m & 1][4 * q]);
      const float4 y = *reinterpret_cast<const float4*>(&srl[m & 1][16 + 4 * q]);
      f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w;
      f[4] = y.x; f[5] = y.y; f[6] = y.z; f[7] = y.w;
    }
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      float pe[8], dse[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pe[e] = fast_exp2(s8[i][e] - sf[i].lse2);  // masked or dead head: 0
        dse[e] = pe[e] * (d8[i][e] - sf[i].D) * p.scale;
        const float x = dse[e] * f[e];
        bh[i][e] = (bf16_t)x;
        bl[i][e] = lo_of(x);
      }
      if constexpr (SEL && comp) {
        if (p.dsel || p.gsum) {
          // sum over the heads of p ((dp - D) s + dp): the row's gradient dotted with the row
          float g[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float sraw = s8[i][e] > -INFINITY ? s8[i][e] * kLn2F : 0.f;  // scale qn.k
            g[e] = row16_sum(pe[e] * ((d8[i][e] - sf[i].D) * sraw + d8[i][e]));
            psel[i] += pe[e];
            dssel[i] += dse[e];
          }
          if (p.dsel && n == 0 && t1 + i < p.T) {
            float* dst = p.dsel + ((size_t)b * p.T + t1 + i) * p.nb;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              const int j = 32 * m + 16 * half + 4 * q;
              // (added: calls for further groups of heads add theirs)
              if ((p.nb & 3) == 0 && !p.dsel_add) {
                if (j < p.nb) *reinterpret_cast<float4*>(dst + j) =
                    make_float4(g[4 * half], g[4 * half + 1], g[4 * half + 2], g[4 * half + 3]);
              } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  if (j + e < p.nb) dst[j + e] = g[4 * half + e] + (p.dsel_add ? dst[j + e] : 0.f);
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      const bf16x8 vh = MqaWave<HD>::vt_frag(kt, to, tt);
      if constexpr (KX && !comp) {
#pragma unroll
        for (int i = 0; i < QW; ++i) dq[i][tt] = mfma2b(vh, bh[i], bl[i], dq[i][tt]);
      } else {
        const bf16x8 vl = MqaWave<HD>::vt_frag(kt + TILE, to, tt);
#pragma unroll
        for (int i = 0; i < QW; ++i) dq[i][tt] = mfma3(vh, vl, bh[i], bl[i], dq[i][tt]);
      }
    }
  };
  for (int m = 0; m < nsc; ++m) pass2(Comp{}, m);
  for (int m = nsc; m < nsteps; ++m) pass2(Win{}, m);
#pragma unroll
  for (int i = 0; i < QW; ++i) {
    if (t1 + i >= p.T) break;  // whole waves
    const size_t bt = (size_t)b * p.T + t1 + i;
    finish_query<HD>(p, bt, n, q, dq[i], rq[i], sf[i].lse2, sf[i].D, sf[i].sk2);
    if constexpr (SEL) {
      if (p.gsum) store_gsum<HD, QT>(p, bt, n, q, psel[i], dssel[i], rq[i]);
      // the blocks that no query of the workgroup sees
      if (p.dsel && !p.dsel_add)
        for (int j = 32 * nsc + lane; j < p.nb; j += 64) p.dsel[bt * p.nb + j] = 0.f;
    }
  }
}

// -------------------------------------------- query pass, selected rows gathered
template <int HD, typename QT>
__global__ __launch_bounds__(256, 2) void attn_bwd_q_kernel(HcaBwdParams p) {
  constexpr bool ONE = Parts<QT>::one;
  using W = QWave<HD>;
  constexpr int NS = W::NS, NT = W::NT, TPR = W::TPR, RPI = W::RPI, NLI = W::NLI;
  constexpr int TILE = 32 * HD;  // bf16 per 32-row tile
  __shared__ __attribute__((aligned(16))) bf16_t lds[4 * 2 * TILE];
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, q = lane >> 4, n = lane & 15;
  bf16_t* sth = lds + wv * 2 * TILE;  // this wave's hi and lo tiles
  bf16_t* stl = sth + TILE;
  const int tiles_per_b = (p.T + 3) / 4;
  const int b = blockIdx.x / tiles_per_b;
  const int t = (blockIdx.x - b * tiles_per_b) * 4 + wv;
  if (t >= p.T) return;  // whole waves: no workgroup barrier below
  const size_t bt = (size_t)b * p.T + t;
  const TileOffsets<HD> to;

  // B operands: q and dout of head n, dims 32s + 8q .. (16 heads, padded rows zero)
  bf16x8 qh[NS], ql[NS], dh[NS], dl[NS];
  float ss = 0.f;
  {
    const bool ok = n < p.nh;
    const size_t ro = ok ? (bt * p.nh + n) * HD + 8 * q : 0;
    float unused = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      load_parts<QT>(static_cast<const QT*>(p.q) + ro + 32 * s, ok, qh[s], ql[s], ss);
      load_parts<QT>(static_cast<const QT*>(p.dout) + ro + 32 * s, ok, dh[s], dl[s], unused);
    }
  }
  const float rq = l2_inv(colq_sum(ss));
  const int nsel = p.topk;
  const int i0 = p.win > 0 ? max(0, p.win - 1 - t) : 0;
  const int nwin = p.win > 0 ? p.win - i0 : 0;
  const int wpos0 = t - p.win + 1 + i0;
  // The compressed rows are padded to whole 32-row steps (masked), so that a
  // step reads only compressed or only window rows, each through a buffer
  // resource over this batch row's rows (hi and lo planes): an offset past its
  // end reads zeros, so a row address is one multiply-add and masked slots
  // need no readable default. Rows are taken in the score layout of
  // MqaWave::chunk_sl: slot k of lane group q is row row_sl(k, q) of the
  // step, whose scores the lane holds, so each lane masks its own scores
  // from the indices it loaded.
  using MW = MqaWave<HD>;
  constexpr int ROWB = HD * 2;
  const int nsel_pad = p.nb > 0 ? (nsel + 31) & ~31 : 0;
  const int nsteps = (nsel_pad + nwin + 31) / 32;
  const int lane_off = 16 * (lane % TPR);
  const int hmask = (TPR == 8 && ((lane >> 3) & 1)) ? -1 : 0;  // HD 64: slot i + 4
  auto rsrc = [](const bf16_t* base, long long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), 0, (int)bytes, 0x00020000);
  };
  const long long cbytes = (long long)p.nb * ROWB, wbytes = nwin > 0 ? (long long)p.T * ROWB : 0;
  const __amdgpu_buffer_rsrc_t rs_ch = rsrc(p.kc_hi + (size_t)b * p.nb * HD, cbytes);
  const __amdgpu_buffer_rsrc_t rs_cl = rsrc(p.kc_lo + (size_t)b * p.nb * HD, cbytes);
  const __amdgpu_buffer_rsrc_t rs_wh = rsrc(nwin > 0 ? p.kn_hi + (size_t)b * p.T * HD : p.kc_hi, wbytes);
  const __amdgpu_buffer_rsrc_t rs_wl = rsrc(nwin > 0 ? p.kn_lo + (size_t)b * p.T * HD : p.kc_lo, wbytes);
  const bool has_idx = nsel > 0;
  const __amdgpu_buffer_rsrc_t rs_idx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int*>(has_idx ? p.idx + bt * p.topk : nullptr), 0, has_idx ? nsel * 4 : 0, 0x00020000);
  const bool idx16 = (nsel & 3) == 0;  // 16-byte index loads never straddle the end
  float* const drow = p.dsel ? p.dsel + bt * p.nb : nullptr;
  if (drow && !p.dsel_add) {
    // the query's row of dsel, cleared while pass 1 runs
    if ((p.nb & 3) == 0)
      for (int j = 4 * lane; j < p.nb; j += 256) *reinterpret_cast<float4*>(drow + j) = make_float4(0.f, 0.f, 0.f, 0.f);
    else
      for (int j = lane; j < p.nb; j += 64) drow[j] = 0.f;
  }
  const float sc = rq * p.scale * kLog2eF;  // raw score -> log2 units

  // the row indices of step m: selected or causal block, or window position
  struct Sel {
    int v[8];
  };
  auto load_sel = [&](int m, Sel& sl) {
    const int j0 = 32 * m;
    if (__builtin_amdgcn_readfirstlane(j0 < nsel_pad ? 1 : 0)) {
      if (idx16) {
        typedef int i32x4 __attribute__((ext_vector_type(4)));
        const i32x4 x = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_idx, (j0 + 4 * q) * 4, 0, 0));
        const i32x4 y = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_idx, (j0 + 16 + 4 * q) * 4, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sl.v[e] = x[e];
          sl.v[4 + e] = y[e];
        }
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          sl.v[k] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_idx, (j0 + MW::row_sl(k, q)) * 4, 0, 0);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) sl.v[k] = wpos0 + (j0 - nsel_pad) + MW::row_sl(k, q);
    }
  };
  // gather the 32 rows of step m (hi and lo planes); ok[k]: slot k is a key
  auto gather = [&](int m, const Sel& sl, typename W::Rows& rr, bool (&ok)[8]) {
    const int j0 = 32 * m;
    const int ms = __builtin_amdgcn_readfirstlane(j0 < nsel_pad ? 1 : 0);
    const __amdgpu_buffer_rsrc_t rh = ms ? rs_ch : rs_wh;
    const __amdgpu_buffer_rsrc_t rl = ms ? rs_cl : rs_wl;
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
      // (a select of values, not an indexed read: that would put sl in scratch memory)
      const int v = TPR == 8 ? sl.v[i] ^ ((sl.v[i] ^ sl.v[(i + 4) & 7]) & hmask) : sl.v[i];
      const int off = (int)((unsigned)v * ROWB + lane_off);
      rr.h[i] = __builtin_amdgcn_raw_buffer_load_b128(rh, off, 0, 0);
      rr.l[i] = __builtin_amdgcn_raw_buffer_load_b128(rl, off, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int j = j0 + MW::row_sl(k, q);
      const bool okc = (j < nsel) & ((unsigned)sl.v[k] < (unsigned)p.nb);
      const bool okw = j - nsel_pad < nwin;
      ok[k] = ms ? okc : okw;
    }
  };
  auto stage = [&](const typename W::Rows& rr) {
    wave_lds_sync();  // the previous step's reads are done
#pragma unroll
    for (int i = 0; i < NLI; ++i) {
      const int r = MW::row_sl(MW::slot_sl(i), q), c = lane % TPR;
      const int off = r * HD + 8 * (c ^ tile_swz<HD>(r & 15));
      *reinterpret_cast<u32x4*>(sth + off) = rr.h[i];
      *reinterpret_cast<u32x4*>(stl + off) = rr.l[i];
    }
    wave_lds_sync();
  };
  // S^T (log2 units) and dP^T of the staged 32 rows: sc8 / dp8 for keys 4q+e, 16+4q+e of head n
  auto scores = [&](const bool (&ok)[8], float (&s8)[8], float (&d8)[8]) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 sa = {0.f, 0.f, 0.f, 0.f}, da = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const bf16x8 kh = *reinterpret_cast<const bf16x8*>(sth + 16 * HD * half + to.key(s));
        const bf16x8 kl = *reinterpret_cast<const bf16x8*>(stl + 16 * HD * half + to.key(s));
        sa = mma_kx<ONE>(kh, kl, qh[s], ql[s], sa);
        da = mma_kx<ONE>(kh, kl, dh[s], dl[s], da);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s8[4 * half + e] = ok[4 * half + e] ? sa[e] * sc : -INFINITY;
        d8[4 * half + e] = da[e];
      }
    }
  };

  // ---- pass 1: lse (log2 units) and D = sum p dp, running maximum per head ----
  float m = -INFINITY, l = 0.f, ad = 0.f;
  {
    typename W::Rows rr;
    Sel sl;
    bool okn[8];
    if (nsteps > 0) {
      load_sel(0, sl);
      gather(0, sl, rr, okn);
      load_sel(1, sl);
    }
    for (int st = 0; st < nsteps; ++st) {
      stage(rr);
      bool ok[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) ok[k] = okn[k];
      if (st + 1 < nsteps) {
        gather(st + 1, sl, rr, okn);
        load_sel(st + 2, sl);
      }
      float s8[8], d8[8];
      scores(ok, s8, d8);
      soft_step(s8, d8, m, l, ad);
    }
  }
  const Soft sf = close_softmax(p, n, m, l, ad);
  const float lse2 = sf.lse2, D = sf.D;

  // ---- pass 2: ds, dqn^T += K^T ds^T, the slot terms ----
  f32x4 dq[NT];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) dq[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float psel = 0.f, dssel = 0.f;  // sums over the selected slots (gsum)
  if (drow) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // its zeros are written before any value
  {
    typename W::Rows rr;
    Sel sl;
    bool okn[8];
    if (nsteps > 0) {
      load_sel(0, sl);
      gather(0, sl, rr, okn);
      load_sel(1, sl);
    }
    for (int st = 0; st < nsteps; ++st) {
      stage(rr);
      bool ok[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) ok[k] = okn[k];
      if (st + 1 < nsteps) {
        gather(st + 1, sl, rr, okn);
        load_sel(st + 2, sl);
      }
      float s8[8], d8[8];
      scores(ok, s8, d8);
      float pe[8], dse[8];
      bf16x8 bh, bl;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pe[e] = fast_exp2(s8[e] - lse2);  // masked or dead head: 0
        dse[e] = pe[e] * (d8[e] - D) * p.scale;
        bh[e] = (bf16_t)dse[e];
        bl[e] = lo_of(dse[e]);
      }
      if (32 * st < nsel_pad) {
        if (p.gsum) {
          // this head's p and ds sums over the selected rows (unused slots: 0)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            psel += pe[e];
            dssel += dse[e];
          }
        }
        if (drow || p.slot_grad) {
          // sum over the heads of p ((dp - D) s + dp), the row's gradient dotted
          // with the row; slot e of the lane group to its lane n = e
          const int j = 32 * st + MW::row_sl(n & 7, q);
          const int at = has_idx ? (int)__builtin_amdgcn_raw_buffer_load_b32(rs_idx, j * 4, 0, 0) : -1;
          float mine = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float sraw = s8[e] > -INFINITY ? s8[e] * kLn2F : 0.f;  // scale qn.k
            const float g = row16_sum(pe[e] * ((d8[e] - D) * sraw + d8[e]));
            if (n == e) mine = g;
          }
          if (n < 8 && j < nsel && (unsigned)at < (unsigned)p.nb) {
            // (no block is selected twice: one writer an element)
            if (p.slot_grad) p.slot_grad[bt * p.topk + j] += mine;
            if (drow) drow[at] = mine + (p.dsel_add ? drow[at] : 0.f);
          }
        }
      }
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        const bf16x8 vh = MqaWave<HD>::vt_frag(sth, to, tt);
        const bf16x8 vl = MqaWave<HD>::vt_frag(stl, to, tt);
        dq[tt] = mfma3(vh, vl, bh, bl, dq[tt]);
      }
    }
  }
  finish_query<HD>(p, bt, n, q, dq, rq, lse2, D, sf.sk2);
  if (p.gsum) store_gsum<HD, QT>(p, bt, n, q, psel, dssel, rq);
}

// ------------------------------------------------------------------ key pass
// MODE 0: compressed rows (HCA: visible when n < (t+1) / m2; CSA: selected),
// chunk ci of part_qc queries; MODE 1: window rows (row u seen by t in
// [u, u + win)), chunk ci of win_qc of the queries that see the tile.
// KX (MODE 1): the window rows are exact in one part (bf16 rows and queries).
template <int HD, int MODE, typename QT, int KG, bool KX>
__global__ __launch_bounds__(256, 2) void attn_bwd_k_kernel(HcaBwdParams p, int nchunk) {
  constexpr bool ONE = Parts<QT>::one;
  constexpr int NS = HD / 32, NT = HD / 16;
  constexpr int TILE = 32 * HD;
  constexpr int PL = ONE ? 1 : 2;             // planes of q and of dout
  constexpr int CPR = HD / 8;                 // 8-element chunks per row
  constexpr int LPT = 2 * TILE / 8 / 256;     // chunks per thread per pair (q and dout)
  constexpr int KTR = 64 * KG;                // key rows per workgroup
  __shared__ __attribute__((aligned(16))) bf16_t lds[2][2 * PL * TILE];  // q (hi, lo), dout (hi, lo)
  __shared__ __attribute__((aligned(16))) float sl[2][32], sd[2][32], sr[2][32];  // lse, D, 1/|q| per row
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, q = lane >> 4, n = lane & 15;
  const int b = blockIdx.y;
  const int nrows = MODE == 0 ? p.nb : p.T;
  const int tile = blockIdx.x / nchunk, ci = blockIdx.x - tile * nchunk;
  const int r0 = tile * KTR;
  int tlo, thi;
  if constexpr (MODE == 0) {
    tlo = max(ci * p.part_qc, (r0 + 1) * p.m2 - 1);
    thi = min(p.T, (ci + 1) * p.part_qc);
    if (tlo >= thi) return;  // no row of the tile is seen by this chunk (nothing is read back)
  } else {
    tlo = r0 + ci * p.win_qc;
    thi = min(min(p.T, r0 + KTR + p.win - 1), tlo + p.win_qc);
  }
  // the queries that see any row of this wave: the others are only staged
  const int rw = r0 + 16 * KG * wv;
  const int wlo = MODE == 0 ? (rw + 1) * p.m2 - 1 : rw;
  const int whi = MODE == 0 ? p.T : rw + 16 * KG - 1 + p.win;
  const TileOffsets<HD> to;

  // key fragments (B operand of S = Q K^T): rows rw + 16 g + n, dims 32s + 8q ..
  bf16x8 kh[KG][NS], kl[KG][KX ? 1 : NS];
  float rk1[KG];  // the row's factor: 1, or 1/|x| (window)
  f32x4 dk[KG][NT];
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    const int rk = rw + 16 * g + n;
    const bool ok = rk < nrows;
    const size_t row = (size_t)b * nrows + (ok ? rk : 0);
    const size_t ro = row * (MODE == 0 ? HD : p.ldl) + 8 * q;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      kh[g][s] = *reinterpret_cast<const bf16x8*>((MODE == 0 ? p.kc_hi : p.kl_hi) + ro + 32 * s);
      if (!ok) kh[g][s] = bf16x8{};
      if constexpr (!KX) {
        kl[g][s] = *reinterpret_cast<const bf16x8*>((MODE == 0 ? p.kc_lo : p.kl_lo) + ro + 32 * s);
        if (!ok) kl[g][s] = bf16x8{};
      }
    }
    rk1[g] = MODE == 0 ? 1.f : p.rl[row];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) dk[g][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // staging of a query pair (t, t + 1): rows 16 i + h = head h of query t + i of
  // q (the thread's first chunks) and dout
  struct alignas(16) Raw {
    QT v[8];
  };
  struct Pair {
    Raw x[LPT];
    float l, d, r;
  };
  auto fetch = [&](int tp, Pair& v) {
#pragma unroll
    for (int k = 0; k < LPT; ++k) {
      const int pc = tid + 256 * k, w = pc % (32 * CPR), row = w / CPR, c = w % CPR;
      const int tq = tp + (row >> 4), h = row & 15;
      const QT* src = static_cast<const QT*>(pc < 32 * CPR ? p.q : p.dout);
      const bool ok = tq < p.T && h < p.nh;
      const QT* at = src + (ok ? (((size_t)b * p.T + tq) * p.nh + h) * HD + 8 * c : 0);
      if (ok) {
#pragma unroll
        for (int i = 0; i < (int)sizeof(Raw) / 16; ++i)
          reinterpret_cast<u32x4*>(v.x[k].v)[i] = reinterpret_cast<const u32x4*>(at)[i];
      } else {
#pragma unroll
        for (int i = 0; i < (int)sizeof(Raw) / 16; ++i) reinterpret_cast<u32x4*>(v.x[k].v)[i] = u32x4{0, 0, 0, 0};
      }
    }
    v.l = INFINITY;
    v.d = v.r = 0.f;
    if (tid < 32 && tp + (tid >> 4) < p.T) {
      const size_t li = ((size_t)b * p.T + tp + (tid >> 4)) * 16 + (tid & 15);
      v.l = p.lse[li];
      v.d = p.dval[li];
      v.r = p.rq[li];
    }
  };
  auto put = [&](int k2, const Pair& v) {
#pragma unroll
    for (int k = 0; k < LPT; ++k) {
      const int pc = tid + 256 * k, w = pc % (32 * CPR), row = w / CPR, c = w % CPR;
      bf16_t* dst = lds[k2] + (pc / (32 * CPR)) * PL * TILE + row * HD + 8 * (c ^ tile_swz<HD>(row & 15));
      if constexpr (ONE) {
        *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(v.x[k].v);
      } else {
        bf16x8 h, l;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float f = (float)v.x[k].v[i];
          h[i] = (bf16_t)f;
          l[i] = lo_of(f);
        }
        *reinterpret_cast<bf16x8*>(dst) = h;
        *reinterpret_cast<bf16x8*>(dst + TILE) = l;
      }
    }
    if (tid < 32) {
      sl[k2][tid] = v.l;
      sd[k2][tid] = v.d;
      sr[k2][tid] = v.r;
    }
  };
  const int nw = (p.nb + 31) / 32;
  auto visible = [&](int tq, int rk) -> bool {
    if (tq >= thi || rk >= nrows) return false;  // (the pair's second query may lie past the chunk)
    if constexpr (MODE == 1) return tq >= rk && tq < rk + p.win;
    if (p.sel) return (p.sel[((size_t)b * p.T + tq) * nw + (rk >> 5)] >> (rk & 31)) & 1u;
    return rk < (tq + 1) / p.m2;
  };

  Pair pv;
  if (tlo < thi) {
    fetch(tlo, pv);
    put(0, pv);
  }
  __syncthreads();
  int buf = 0;
  for (int tp = tlo; tp < thi; tp += 2) {
    const bool more = tp + 2 < thi;
    if (more) fetch(tp + 2, pv);
    if (tp + 1 >= wlo && tp < whi) {
      const bf16_t* xq = lds[buf];
      const bf16_t* xd = lds[buf] + PL * TILE;
      bf16x8 ash[KG], asl[KG], aph[KG], apl[KG];  // ds^T / |q| and p^T: key n, slots (query i, heads 4q .. 4q+3)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int tq = tp + i;
        f32x4 sa[KG], da[KG];
#pragma unroll
        for (int g = 0; g < KG; ++g) sa[g] = da[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const int ko = 16 * HD * i + to.key(s);
          const bf16x8 xh = *reinterpret_cast<const bf16x8*>(xq + ko);
          const bf16x8 yh = *reinterpret_cast<const bf16x8*>(xd + ko);
          bf16x8 xl = xh, yl = yh;
          if constexpr (!ONE) {
            xl = *reinterpret_cast<const bf16x8*>(xq + TILE + ko);
            yl = *reinterpret_cast<const bf16x8*>(xd + TILE + ko);
          }
#pragma unroll
          for (int g = 0; g < KG; ++g) {
            if constexpr (KX) {
              sa[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, kh[g][s], sa[g], 0, 0, 0);
              da[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yh, kh[g][s], da[g], 0, 0, 0);
            } else {
              sa[g] = mma_xk<ONE>(xh, xl, kh[g][s], kl[g][s], sa[g]);
              da[g] = mma_xk<ONE>(yh, yl, kh[g][s], kl[g][s], da[g]);
            }
          }
        }
        // lane: heads 4q .. 4q+3 of query tq, keys rw + 16 g + n
        const float4 L4 = *reinterpret_cast<const float4*>(&sl[buf][16 * i + 4 * q]);
        const float4 D4 = *reinterpret_cast<const float4*>(&sd[buf][16 * i + 4 * q]);
        const float4 R4 = *reinterpret_cast<const float4*>(&sr[buf][16 * i + 4 * q]);
        const float Ls[4] = {L4.x, L4.y, L4.z, L4.w}, Ds[4] = {D4.x, D4.y, D4.z, D4.w};
        const float Rs[4] = {R4.x, R4.y, R4.z, R4.w};
#pragma unroll
        for (int g = 0; g < KG; ++g) {
          const bool vis = visible(tq, rw + 16 * g + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float pe = vis ? fast_exp2(sa[g][e] * (Rs[e] * (rk1[g] * p.scale * kLog2eF)) - Ls[e]) : 0.f;
            const float dse = pe * (da[g][e] * rk1[g] - Ds[e]) * p.scale * Rs[e];
            ash[g][4 * i + e] = (bf16_t)dse;
            asl[g][4 * i + e] = lo_of(dse);
            aph[g][4 * i + e] = (bf16_t)pe;
            apl[g][4 * i + e] = lo_of(pe);
          }
        }
      }
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        const bf16x8 bq = MqaWave<HD>::vt_frag(xq, to, tt);
        const bf16x8 bd = MqaWave<HD>::vt_frag(xd, to, tt);
        bf16x8 bql = bq, bdl = bd;
        if constexpr (!ONE) {
          bql = MqaWave<HD>::vt_frag(xq + TILE, to, tt);
          bdl = MqaWave<HD>::vt_frag(xd + TILE, to, tt);
        }
#pragma unroll
        for (int g = 0; g < KG; ++g) {
          dk[g][tt] = mma_kx<ONE>(ash[g], asl[g], bq, bql, dk[g][tt]);
          dk[g][tt] = mma_kx<ONE>(aph[g], apl[g], bd, bdl, dk[g][tt]);
        }
      }
    }
    if (more) put(buf ^ 1, pv);
    __syncthreads();
    buf ^= 1;
  }
  // dk tile tt: rows (keys) rw + 16 g + 4q + e, column (dim) 16 tt + n
  float* out = MODE == 0 ? p.part_b + (((size_t)b * nchunk + ci) * p.nb) * HD
                         : p.part_w + ((size_t)ci * p.B + b) * p.T * HD;
#pragma unroll
  for (int g = 0; g < KG; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = rw + 16 * g + 4 * q + e;
      if (r < nrows) {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) out[(size_t)r * HD + 16 * tt + n] = dk[g][tt][e];
      }
    }
}

// slot[row, j] += dsel[row, idx[row, j]] (idx < 0: unused slot)
__global__ __launch_bounds__(256) void slot_gather_kernel(const int* idx, const float* dsel, float* slot,
                                                          long long n, int topk, int nb) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int k = idx[i];
  if (k >= 0 && k < nb) slot[i] += dsel[i / topk * nb + k];
}

// The key passes' grids: groups of 16 keys per wave, queries per chunk.
struct KeyPlan {
  int kg, qc, nchunk;    // compressed rows
  int wqc, wnc;          // window rows
};
KeyPlan key_plan(int B, int T, int nb, int win) {
  KeyPlan k;
  // two groups of 16 keys per wave halve the LDS reads per product; one group
  // where two would leave waves without keys
  k.kg = nb > 64 ? 2 : 1;
  const long long ntile = (nb + 64 * k.kg - 1) / (64 * k.kg);
  // chunks of 512 queries, halved (to 64) while the grid, half of which the
  // causal rule leaves empty, would give the 256 compute units less than two
  // workgroups each
  k.qc = 512;
  while (k.qc > 64 && ntile * ((T + k.qc - 1) / k.qc) * B < 1024) k.qc /= 2;
  k.nchunk = (T + k.qc - 1) / k.qc;
  // window: a tile of 128 rows is seen by 127 + win queries, in up to 4 chunks
  const long long wt = (long long)B * ((T + 127) / 128);
  k.wnc = 1;
  while (k.wnc < 4 && wt * k.wnc < 512 && (127 + win) / k.wnc > 64) k.wnc *= 2;
  k.wqc = ((127 + win + k.wnc - 1) / k.wnc + 1) & ~1;
  return k;
}

}  // namespace

bool attn_bwd_mfma_supported(const HcaBwdParams& p) {
  return p.normalize && (p.c == 64 || p.c == 128) && p.nh >= 1 && p.nh <= 16;
}

// CSA: whether the query pass takes every visible block in tiles (true) or
// gathers the selected rows. The tiles' cost grows with the visible blocks
// (nb / 2 on average), the gather's with topk. Whole core backward with the
// surrogate, about 8192 queries, 16 heads of 128, window 128, bf16, tiles /
// gather in ms: topk 512, nb 1024 1.04 / 1.11, 1536 1.10 / 1.08, 2048 1.74 /
// 1.62; topk 256, nb 512 0.69 / 0.73, 768 0.71 / 0.71, 1024 1.03 / 0.98; topk
// 128, nb 256 0.54 / 0.57, 384 0.61 / 0.61, 512 0.68 / 0.67; topk 64, nb 128 0.48
// / 0.51, 256 0.53 / 0.54, 512 0.68 / 0.64.
static bool attn_bwd_dense_rows(int nb, int topk) { return nb <= 3 * topk; }

static size_t al256m(size_t x) { return (x + 255) & ~size_t(255); }

size_t attn_bwd_mfma_ws_bytes(int B, int T, int c, int m2, int win, int topk, bool slots) {
  const size_t BT = (size_t)B * T;
  const int nb = T / m2;
  const KeyPlan k = key_plan(B, T, nb, win);
  size_t z = 3 * al256m(BT * 16 * 4);                  // lse, D, 1/|q| (16 heads)
  z += 2 * al256m((size_t)B * nb * c * 2);              // compressed rows hi / lo
  // window rows: factors, the splits of the rows and of the normalised rows
  if (win > 0) z += al256m(BT * 4) + 4 * al256m(BT * c * 2);
  z += al256m((size_t)B * k.nchunk * nb * c * 4);       // compressed-row partials
  if (win > 0) z += al256m(BT * k.wnc * c * 4);         // window-row partials
  if (topk > 0) {
    z += al256m(BT * ((nb + 31) / 32) * 4);              // selection bitmap
    // the tiled query pass's values by block, for the slots (at most 3 topk a query)
    if (slots && attn_bwd_dense_rows(nb, topk)) z += al256m(BT * nb * 4);
  }
  return z;
}

hipError_t sel_bitmap_launch(const int* idx, uint32_t* sel, long long nq, int topk, int nw, hipStream_t s);

template <int HD, typename QT, bool KX>
static void launch_passes(const HcaBwdParams& p, const KeyPlan& k, hipStream_t s) {
  const int tq = Parts<QT>::one ? 8 : 4;  // queries per workgroup of the tiled query pass
  const int nt = (p.T + tq - 1) / tq;
  const dim3 qg((unsigned)((long long)p.B * nt));
  if (!p.sparse)
    hipLaunchKernelGGL((attn_bwd_qt_kernel<HD, QT, false, KX>), qg, dim3(256), 0, s, p, nt);
  else if (attn_bwd_dense_rows(p.nb, p.topk))
    hipLaunchKernelGGL((attn_bwd_qt_kernel<HD, QT, true, KX>), qg, dim3(256), 0, s, p, nt);
  else
    hipLaunchKernelGGL((attn_bwd_q_kernel<HD, QT>), dim3((unsigned)(p.B * ((p.T + 3) / 4))), dim3(256), 0, s, p);
  if (p.nb > 0 && !(p.sparse && p.topk == 0)) {
    const dim3 g((p.nb + 64 * k.kg - 1) / (64 * k.kg) * k.nchunk, p.B);
    if (k.kg == 2)
      hipLaunchKernelGGL((attn_bwd_k_kernel<HD, 0, QT, 2, false>), g, dim3(256), 0, s, p, k.nchunk);
    else
      hipLaunchKernelGGL((attn_bwd_k_kernel<HD, 0, QT, 1, false>), g, dim3(256), 0, s, p, k.nchunk);
  }
  if (p.win > 0)
    hipLaunchKernelGGL((attn_bwd_k_kernel<HD, 1, QT, 2, KX>), dim3((p.T + 127) / 128 * k.wnc, p.B), dim3(256), 0, s,
                       p, k.wnc);
}

// The window rows' factors and splits: the rows as given unless they are used in
// place (ldl = f.ldl), the normalised rows for the gathering query pass.
template <int HD, typename T>
static void launch_window_rows(const HcaBwdParams& p, const BwdFinish& f, hipStream_t s) {
  constexpr int rpb = 256 / (HD / 8);
  const long long BT = (long long)p.B * p.T;
  hipLaunchKernelGGL((window_rows_kernel<HD, T>), dim3((unsigned)((BT + rpb - 1) / rpb)), dim3(256), 0, s,
                     static_cast<const T*>(f.lsrc), f.ldl, BT, const_cast<float*>(p.rl),
                     p.kl_lo ? const_cast<bf16_t*>(p.kl_hi) : nullptr, const_cast<bf16_t*>(p.kl_lo),
                     const_cast<bf16_t*>(p.kn_hi), const_cast<bf16_t*>(p.kn_lo));
}

template <int HD>
static hipError_t run_passes(const HcaBwdParams& p, const BwdFinish& f, const KeyPlan& k, hipStream_t s) {
  constexpr int rpb = 256 / (HD / 8);  // rows per workgroup
  const long long bn = (long long)p.B * p.nb;
  if (bn > 0)
    hipLaunchKernelGGL((split_rows_kernel<HD>), dim3((unsigned)((bn + rpb - 1) / rpb)), dim3(256), 0, s, f.kc, bn,
                       const_cast<bf16_t*>(p.kc_hi), const_cast<bf16_t*>(p.kc_lo));
  if (p.win > 0) {
    if (f.cdt == DT_BF16) launch_window_rows<HD, bf16_t>(p, f, s);
    else if (f.cdt == DT_F16) launch_window_rows<HD, _Float16>(p, f, s);
    else launch_window_rows<HD, float>(p, f, s);
  }
  if (p.qdt == DT_BF16) {
    if (p.win > 0 && !p.kl_lo) launch_passes<HD, bf16_t, true>(p, k, s);
    else launch_passes<HD, bf16_t, false>(p, k, s);
  } else if (p.qdt == DT_F16) {
    launch_passes<HD, _Float16, false>(p, k, s);
  } else {
    launch_passes<HD, float, false>(p, k, s);
  }
  return hipGetLastError();
}

hipError_t attn_bwd_mfma_dispatch(HcaBwdParams p, BwdFinish f, void* ws, hipStream_t s) {
  const int HD = p.c;
  const size_t BT = (size_t)p.B * p.T;
  const KeyPlan k = key_plan(p.B, p.T, p.nb, p.win);
  char* w = static_cast<char*>(ws);
  auto take = [&](size_t bytes) {
    char* r = w;
    w += al256m(bytes);
    return r;
  };
  p.lse = reinterpret_cast<float*>(take(BT * 16 * 4));
  p.dval = reinterpret_cast<float*>(take(BT * 16 * 4));
  p.rq = reinterpret_cast<float*>(take(BT * 16 * 4));
  p.kc_hi = reinterpret_cast<bf16_t*>(take((size_t)p.B * p.nb * HD * 2));
  p.kc_lo = reinterpret_cast<bf16_t*>(take((size_t)p.B * p.nb * HD * 2));
  const bool tiled = !p.sparse || attn_bwd_dense_rows(p.nb, p.topk);
  if (p.win > 0) {
    p.rl = reinterpret_cast<float*>(take(BT * 4));
    if (f.cdt == DT_BF16 && p.qdt == DT_BF16) {
      p.kl_hi = static_cast<const bf16_t*>(f.lsrc);
      p.ldl = f.ldl;
    } else {
      p.kl_hi = reinterpret_cast<bf16_t*>(take(BT * HD * 2));
      p.kl_lo = reinterpret_cast<bf16_t*>(take(BT * HD * 2));
      p.ldl = HD;
    }
    if (!tiled) {
      p.kn_hi = reinterpret_cast<bf16_t*>(take(BT * HD * 2));
      p.kn_lo = reinterpret_cast<bf16_t*>(take(BT * HD * 2));
    }
  }
  p.part_b = reinterpret_cast<float*>(take((size_t)p.B * k.nchunk * p.nb * HD * 4));
  p.part_w = p.win > 0 ? reinterpret_cast<float*>(take(BT * k.wnc * HD * 4)) : nullptr;
  p.part_qc = k.qc;
  p.win_qc = k.wqc;
  if (p.idx && p.topk > 0) {
    const int nw = (p.nb + 31) / 32;
    uint32_t* sel = reinterpret_cast<uint32_t*>(take(BT * nw * 4));
    const hipError_t e = sel_bitmap_launch(p.idx, sel, (long long)BT, p.topk, nw, s);
    if (e != hipSuccess) return e;
    p.sel = sel;
    if (tiled && p.slot_grad && !p.dsel) {
      p.dsel = reinterpret_cast<float*>(take(BT * p.nb * 4));
      p.dsel_add = 0;
    }
  }
  hipError_t e = HD == 64 ? run_passes<64>(p, f, k, s) : run_passes<128>(p, f, k, s);
  if (e != hipSuccess) return e;
  if (p.slot_grad && p.idx && tiled) {
    const long long ns = (long long)BT * p.topk;
    hipLaunchKernelGGL(slot_gather_kernel, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, s, p.idx, p.dsel,
                       p.slot_grad, ns, p.topk, p.nb);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (p.nb > 0 && p.sparse && p.topk == 0) {
    // no selection: the compressed rows receive nothing
    e = fill_u32(p.part_b, (long long)p.B * k.nchunk * p.nb * HD, 0u, s);
    if (e != hipSuccess) return e;
  }
  f.part_b = p.part_b;
  f.part_w = p.part_w;
  f.rl = p.rl;
  f.nchunk = k.nchunk;
  f.part_qc = k.qc;
  f.win_nc = k.wnc;
  return bwd_finish_launch(f, HD, s);
}

}  // namespace kch
