// Manifold-constrained hyper-connection (mHC) mixing with the Sinkhorn normalisation fused in (gfx950).
//
// The reference configures the DeepSeek residual hyper-connections (hc_mult = 4 streams,
// hc_sinkhorn_iters = 20, hc_eps; baseline/indexer.py:48-50) and ships their 4x4 Sinkhorn projection as
// an operator of its own (baseline/sinkhorn.py; mhc = 4 there).  A layer with hc_mult = n keeps n residual
// streams x[t] in R^{n x C} per token; from logits computed on the flattened, normalised streams it forms
//   H_pre  = sigmoid(pre logits)        (n)       the layer input   h = H_pre x            (ks_mhc_pre)
//   H_post = 2 sigmoid(post logits)     (n)       the residual update
//   H_res  = Sinkhorn(res logits)       (n x n)   x' = H_res x + H_post^T f(h)            (ks_mhc_post)
// with the Sinkhorn of baseline/sinkhorn.py:13-19 (softmax + eps, column pass, then repeat - 1 row /
// column passes).  Here the Sinkhorn runs inside its consumer: ks_mhc_post normalises each token's 4x4
// logits in registers (a quad of lanes, one row per lane) and applies the doubly stochastic matrix to the
// streams in the same pass, so the matrices never reach memory and no Sinkhorn launch is needed.
//
// Work decomposition (both kernels HBM-bound streams): one wave per token; every quad of the wave
// computes the token's matrix (the DPP reductions keep the quads independent), lanes then gather the four
// rows by quad broadcasts, and the wave streams the token's columns in 16-byte chunks (8 bf16) with fully
// coalesced loads of the n stream rows and of f, fp32 arithmetic, and RNE bf16 stores.
#include "common.h"
#include "sinkhorn_quad.h"

namespace ks {
namespace {

constexpr int kMhcWaves = 4;  // tokens (waves) per workgroup
constexpr int kMhcN = 4;      // hc_mult

// Value of lane (lane & ~3) + SRC of the quad (DPP quad_perm [SRC, SRC, SRC, SRC]).
template <int SRC>
__device__ __forceinline__ float quad_bcast(float v) {
  constexpr int ctrl = SRC | (SRC << 2) | (SRC << 4) | (SRC << 6);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, false));
}

__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ __forceinline__ void unpack8(uint4 u, float (&v)[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    v[2 * p] = bf16_to_f32(static_cast<uint16_t>(w[p] & 0xFFFFu));
    v[2 * p + 1] = bf16_to_f32(static_cast<uint16_t>(w[p] >> 16));
  }
}

__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    w[p] = cvt_pk_bf16(v[2 * p], v[2 * p + 1]);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// out[t, i, :] = sum_j H_res[t][i][j] x[t, j, :] + H_post[t][i] f[t, :]   (out may alias x: each lane reads
// its columns of all four streams before writing them)
__global__ __launch_bounds__(64 * kMhcWaves) void mhc_post_kernel(const uint16_t *x, const uint16_t *__restrict__ f,
                                                                 const float *__restrict__ res_logits,
                                                                 const float *__restrict__ post_logits, uint16_t *out,
                                                                 int64_t N, int64_t C8, int repeat, float eps) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kMhcWaves + wave;
  if (t >= N) return;  // uniform per wave
  const int r = lane & 3;
  // the token's Sinkhorn: lane r of every quad normalises row r (all lanes active for the DPP exchanges)
  float4 row = reinterpret_cast<const float4 *>(res_logits + t * 16)[r];
  const float4 pl = reinterpret_cast<const float4 *>(post_logits + t * 4)[0];
  row = sinkhorn_quad_row(row, repeat, eps);
  float M[kMhcN][kMhcN];
  {
    const float rc[4] = {row.x, row.y, row.z, row.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      M[0][j] = quad_bcast<0>(rc[j]);
      M[1][j] = quad_bcast<1>(rc[j]);
      M[2][j] = quad_bcast<2>(rc[j]);
      M[3][j] = quad_bcast<3>(rc[j]);
    }
  }
  const float p[4] = {2.f * sigmoid(pl.x), 2.f * sigmoid(pl.y), 2.f * sigmoid(pl.z), 2.f * sigmoid(pl.w)};
  const int64_t C = C8 * 8;
  const uint4 *xs = reinterpret_cast<const uint4 *>(x + t * kMhcN * C);
  const uint4 *fs = reinterpret_cast<const uint4 *>(f + t * C);
  uint4 *os = reinterpret_cast<uint4 *>(out + t * kMhcN * C);
  for (int64_t c = lane; c < C8; c += 64) {
    uint4 xu[kMhcN];
#pragma unroll
    for (int j = 0; j < kMhcN; ++j) xu[j] = xs[j * C8 + c];
    const uint4 fu = fs[c];
    float xv[kMhcN][8], fv[8];
#pragma unroll
    for (int j = 0; j < kMhcN; ++j) unpack8(xu[j], xv[j]);
    unpack8(fu, fv);
#pragma unroll
    for (int i = 0; i < kMhcN; ++i) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float acc = M[i][0] * xv[0][e];
        acc = __builtin_fmaf(M[i][1], xv[1][e], acc);
        acc = __builtin_fmaf(M[i][2], xv[2][e], acc);
        acc = __builtin_fmaf(M[i][3], xv[3][e], acc);
        o[e] = __builtin_fmaf(p[i], fv[e], acc);
      }
      os[i * C8 + c] = pack8(o);
    }
  }
}

// h[:] = sum_j g[j] x[j, :] of one token, by one wave
__device__ __forceinline__ void mix_streams(const uint16_t *__restrict__ x, const float (&g)[4],
                                            uint16_t *__restrict__ h, int64_t C8, int lane) {
  const uint4 *xs = reinterpret_cast<const uint4 *>(x);
  uint4 *hs = reinterpret_cast<uint4 *>(h);
  for (int64_t c = lane; c < C8; c += 64) {
    uint4 xu[kMhcN];
#pragma unroll
    for (int j = 0; j < kMhcN; ++j) xu[j] = xs[j * C8 + c];
    float xv[kMhcN][8], o[8];
#pragma unroll
    for (int j = 0; j < kMhcN; ++j) unpack8(xu[j], xv[j]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float acc = g[0] * xv[0][e];
      acc = __builtin_fmaf(g[1], xv[1][e], acc);
      acc = __builtin_fmaf(g[2], xv[2][e], acc);
      o[e] = __builtin_fmaf(g[3], xv[3][e], acc);
    }
    hs[c] = pack8(o);
  }
}

// h[t, :] = sum_j sigmoid(pre_logits[t][j]) x[t, j, :]
__global__ __launch_bounds__(64 * kMhcWaves) void mhc_pre_kernel(const uint16_t *__restrict__ x,
                                                                const float *__restrict__ pre_logits,
                                                                uint16_t *__restrict__ h, int64_t N, int64_t C8) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kMhcWaves + wave;
  if (t >= N) return;
  const float4 pl = reinterpret_cast<const float4 *>(pre_logits + t * 4)[0];
  const float g[4] = {sigmoid(pl.x), sigmoid(pl.y), sigmoid(pl.z), sigmoid(pl.w)};
  mix_streams(x + t * kMhcN * C8 * 8, g, h + t * C8 * 8, C8, lane);
}

// ---------------------------------------------------------------- logits of the streams, fused into the layer input
// logits[t] = alpha * (x_norm[t] @ phi) + base with x_norm the RMS-normalised flattened streams (K = 4 C values) and
// phi fp32 [K, 24].  The normalisation is one factor per token, so the contraction runs on the bf16 streams as they
// are, on the MFMA:
//   x phi = x phi_hi + x phi_mid + x phi_lo,  phi split exactly into three bf16 values by truncation (8 significant
// bits each), every product exact and summed in fp32; sum(x^2) is the diagonal of one more MFMA of the tile with
// itself.  Splitting phi in registers (rather than in a pass of its own) costs ~130 VALU per 32 rows and 16 TT tokens,
// under a fifth of the time that the tokens' x needs to arrive.
//   workgroup  16 TT tokens x one of `splits` ranges of K, its 4 waves taking a quarter each; the waves' sums meet in
//              LDS and leave as one partial [split][token][32] (24 products, sum of squares, padding)
//   columns    tiles [hi 0..15], [mid 0..15], [lo 0..15], [hi 16..23 | mid 16..23], [lo 16..23 | 0]
// Bound by the read of x.  At N 4096, C 4096 (134 MB) it takes 37.3 us, 3.6 TB/s, where the torch sequence it replaces
// (widening, square, mean, scale, fp32 GEMM, slices) took 417 us.  x one step ahead instead of three: 41 us; a grid of
// one and a half rounds of workgroups (2048 -> 3072 waves aimed at): 46 us; one wave per SIMD (no register cap): 59 us.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                  0, 0, 0);
}

constexpr int kLogits = 24;      // 4 pre, 4 post, 16 res
constexpr int kPartCols = 32;    // floats per token of a partial: 24 products, sum of squares, 7 unused
constexpr int kProjWaves = 4;
constexpr int kProjMaxSplits = 64;

// Truncation of eight fp32 values to bf16, packed; v keeps the exact remainders (zero where nothing is left, which
// also keeps an infinity out of inf - inf; a NaN stays one).
__device__ __forceinline__ uint4 take_bf16(float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v[2 * p]), b = __builtin_bit_cast(uint32_t, v[2 * p + 1]);
    w[p] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // high halves: a low, b high
    const float ah = __builtin_bit_cast(float, a & 0xFFFF0000u), bh = __builtin_bit_cast(float, b & 0xFFFF0000u);
    v[2 * p] = v[2 * p] == ah ? 0.f : v[2 * p] - ah;
    v[2 * p + 1] = v[2 * p + 1] == bh ? 0.f : v[2 * p + 1] - bh;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

template <int TT>
__global__ __launch_bounds__(64 * kProjWaves, TT == 4 ? 2 : 3) void mhc_proj_kernel(const uint16_t *__restrict__ x,
                                                                  const float *__restrict__ phi,
                                                                  float *__restrict__ part, int64_t N, int64_t K,
                                                                  int splits, int steps_per_wave) {
  constexpr int TOK = 16 * TT;
  __shared__ float red[kProjWaves][TOK][kPartCols + 1];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int split = blockIdx.x % splits;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x / splits) * TOK;
  const int nstep = static_cast<int>(K / 32);  // C % 8 == 0, so K % 32 == 0
  const int s0 = (split * kProjWaves + wave) * steps_per_wave;
  const int s1 = s0 + steps_per_wave < nstep ? s0 + steps_per_wave : nstep;

  // A-fragments: token 16 tt + l16, k = 32 step + 8 g .. + 7 (tokens past N read the last one; not stored)
  const uint16_t *xr[TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    const int64_t t = t0 + 16 * tt + l16;
    xr[tt] = x + (t < N ? t : N - 1) * K + 8 * g;
  }
  const float *pr = phi + static_cast<int64_t>(8 * g) * kLogits;
  const int c1 = 16 + (l16 & 7);
  auto load_x = [&](int s, uint4 (&a)[TT]) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) a[tt] = *reinterpret_cast<const uint4 *>(xr[tt] + 32 * static_cast<int64_t>(s));
  };
  auto load_phi = [&](int s, float (&p0)[8], float (&p1)[8]) {
    const float *ps = pr + static_cast<int64_t>(s) * 32 * kLogits;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p0[i] = ps[i * kLogits + l16];
      p1[i] = ps[i * kLogits + c1];
    }
  };
  f32x4_t acc[TT][6];  // five column tiles and the tile's Gram matrix
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[tt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto step = [&](const uint4 (&a)[TT], float (&p0)[8], float (&p1)[8]) {
    uint4 b[5];
    b[0] = take_bf16(p0);
    b[1] = take_bf16(p0);
    b[2] = take_bf16(p0);
    const uint4 h = take_bf16(p1), m = take_bf16(p1), l = take_bf16(p1);
    const bool lowc = l16 < 8;
    b[3] = make_uint4(lowc ? h.x : m.x, lowc ? h.y : m.y, lowc ? h.z : m.z, lowc ? h.w : m.w);
    b[4] = make_uint4(lowc ? l.x : 0u, lowc ? l.y : 0u, lowc ? l.z : 0u, lowc ? l.w : 0u);
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
      for (int c = 0; c < 5; ++c) acc[tt][c] = mfma16(a[tt], b[c], acc[tt][c]);
      acc[tt][5] = mfma16(a[tt], a[tt], acc[tt][5]);
    }
  };
  if (s0 < s1) {
    // x runs kAhead steps ahead (it comes from memory), phi one step ahead (from L2), phi's loads of a step issued in
    // front of x's: loads return in order, so the wait for the next phi leaves the later x loads in flight
    constexpr int kAhead = 3, kRing = kAhead + 1;
    uint4 a[kRing][TT];
    float p0[2][8], p1[2][8];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      load_x(s0 + i < s1 ? s0 + i : s1 - 1, a[i]);
      if (i == 0) load_phi(s0, p0[0], p1[0]);
    }
    for (int s = s0; s < s1; s += kRing) {
#pragma unroll
      for (int i = 0; i < kRing; ++i) {
        if (s + i >= s1) break;  // uniform
        load_phi(s + i + 1 < s1 ? s + i + 1 : s1 - 1, p0[(i + 1) & 1], p1[(i + 1) & 1]);
        load_x(s + i + kAhead < s1 ? s + i + kAhead : s1 - 1, a[(i + kAhead) % kRing]);
        step(a[i], p0[i & 1], p1[i & 1]);
      }
    }
  }
  // lane (column l16, g): tokens 4 g + r of each tile
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float *d = red[wave][16 * tt + 4 * g + r];
      const float hm = acc[tt][3][r];  // lanes 0..7 the high, 8..15 the mid parts of columns 16..23
      const float other = __builtin_bit_cast(float, lane_xor<8>(__builtin_bit_cast(uint32_t, hm)));
      d[l16] = (acc[tt][2][r] + acc[tt][1][r]) + acc[tt][0][r];
      if (l16 < 8) d[16 + l16] = (acc[tt][4][r] + other) + hm;
      if (l16 == 4 * g + r) d[kLogits] = acc[tt][5][r];
    }
  __syncthreads();
  for (int e = threadIdx.x; e < TOK * kPartCols; e += 64 * kProjWaves) {
    const int tk = e / kPartCols, c = e % kPartCols;
    if (t0 + tk < N && c <= kLogits) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < kProjWaves; ++w) v += red[w][tk][c];
      part[(static_cast<int64_t>(split) * N + t0 + tk) * kPartCols + c] = v;
    }
  }
}

// x phi of one token with x normalised first, for the tokens whose products of plain values leave the fp32 range (values
// past 2^60 or so against large weights): one wave, lane c < 24 receives column c.  Rare, so written for few registers.
__device__ float normalised_product(const uint16_t *__restrict__ x, const float *__restrict__ phi, float rn, int64_t K,
                                    int lane) {
  float z = 0.f;
#pragma unroll 1
  for (int c = 0; c < kLogits; ++c) {
    float acc = 0.f;
#pragma unroll 1
    for (int64_t k = lane; k < K; k += 64) acc = __builtin_fmaf(bf16_to_f32(x[k]) * rn, phi[k * kLogits + c], acc);
#pragma unroll
    for (int m = 1; m < 64; m *= 2) acc += __shfl_xor(acc, m, 64);
    z = lane == c ? acc : z;
  }
  return z;
}

// The logits from the partials, then h as mhc_pre_kernel: one wave per token.  post and res logits are stored for
// the residual update.
__global__ __launch_bounds__(64 * kMhcWaves) void mhc_input_kernel(const uint16_t *__restrict__ x,
                                                                  const float *__restrict__ part,
                                                                  const float *__restrict__ phi,
                                                                  const float *__restrict__ alpha,
                                                                  const float *__restrict__ base,
                                                                  uint16_t *__restrict__ h, float *__restrict__ post,
                                                                  float *__restrict__ res, int64_t N, int64_t C8,
                                                                  int splits, float norm_eps) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kMhcWaves + wave;
  if (t >= N) return;
  const int c = lane & 31;
  const int cc = c <= kLogits ? c : 0;  // the unused columns of a partial are not written
  const int cl = c < kLogits ? c : 0;
  const float al = alpha[cl < 4 ? 0 : cl < 8 ? 1 : 2], bs = base[cl];
  float z = 0.f;
#pragma unroll 4
  for (int s = lane >> 5; s < splits; s += 2) z += part[(static_cast<int64_t>(s) * N + t) * kPartCols + cc];
  z += __builtin_bit_cast(float, lane_xor<32>(__builtin_bit_cast(uint32_t, z)));
  const float ss = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, z), kLogits));
  const float rn = 1.0f / sqrtf(ss / static_cast<float>(C8 * 32) + norm_eps);
  float zn = z * rn;
  // a product or the sum of squares past the fp32 range (uniform; not finite on any of the 25 lanes)
  if (__builtin_amdgcn_ballot_w64(lane <= kLogits && !(fabsf(z) < __builtin_inff())) != 0ull)
    zn = normalised_product(x + t * kMhcN * C8 * 8, phi, rn, C8 * 32, lane);
  const float lg = al * zn + bs;
  if (lane >= 4 && lane < 8) post[t * 4 + lane - 4] = lg;
  if (lane >= 8 && lane < kLogits) res[t * 16 + lane - 8] = lg;
  const float gate = sigmoid(lg);
  float gt[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    gt[j] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, gate), j));
  mix_streams(x + t * kMhcN * C8 * 8, gt, h + t * C8 * 8, C8, lane);
}

int check_mhc(const void *x, int64_t N, int64_t C, const char *what) {
  KS_CHECK_ARG(N >= 0 && N < (int64_t(1) << 31), "%s: N=%lld out of range", what, (long long)N);
  KS_CHECK_ARG(C >= 8 && C % 8 == 0, "%s: C=%lld must be a positive multiple of 8", what, (long long)C);
  KS_CHECK_ARG(N == 0 || x != nullptr, "%s: null pointer", what);
  return KS_OK;
}

// Token tiles per workgroup and ranges of K: 64 tokens share each split of phi's rows where the tokens are enough to
// fill the device that way; ranges until about kProjTargetWaves waves run (one round at two per SIMD), each wave with at least two
// 32-wide steps (one 128-byte line of every row).
constexpr int64_t kProjTargetWaves = 2048;
struct ProjPlan {
  int tt, splits, steps;  // token tiles, ranges, steps per wave
};
inline ProjPlan proj_plan(int64_t N, int64_t C) {
  const int tt = N <= 16 ? 1 : N <= 32 ? 2 : 4;
  const int64_t groups = ceil_div(N, 16 * tt), nstep = 4 * C / 32;
  int64_t splits = ceil_div(kProjTargetWaves, groups * kProjWaves);
  const int64_t most = ceil_div(nstep, 2 * kProjWaves);
  splits = splits > most ? most : splits;
  splits = splits > kProjMaxSplits ? kProjMaxSplits : splits < 1 ? 1 : splits;
  const int64_t steps = ceil_div(nstep, splits * kProjWaves);
  return ProjPlan{tt, static_cast<int>(ceil_div(nstep, steps * kProjWaves)), static_cast<int>(steps)};
}

}  // namespace
}  // namespace ks

extern "C" size_t ks_mhc_input_workspace_size(int64_t N, int64_t C) {
  if (N <= 0 || C < 8 || C % 8 != 0) return 0;  // sizes that ks_mhc_input refuses (or, N = 0, does nothing for)
  return static_cast<size_t>(ks::proj_plan(N, C).splits) * N * ks::kPartCols * sizeof(float);
}

extern "C" int ks_mhc_input(const uint16_t *x, const float *phi, const float *alpha, const float *base, uint16_t *h,
                            float *post_logits, float *res_logits, int64_t N, int64_t C, float norm_eps,
                            void *workspace, size_t workspace_bytes, void *stream) {
  ks::last_error().clear();
  int rc = ks::check_mhc(x, N, C, "ks_mhc_input");
  if (rc != KS_OK) return rc;
  KS_CHECK_ARG(C < (int64_t(1) << 32), "ks_mhc_input: C=%lld out of range", (long long)C);  // 32-bit step counts
  if (N == 0) return KS_OK;
  KS_CHECK_ARG(phi && alpha && base && h && post_logits && res_logits, "ks_mhc_input: null pointer");
  KS_CHECK_ARG(ks::aligned(x, 16) && ks::aligned(h, 16) && ks::aligned(phi, 4) && ks::aligned(alpha, 4) &&
                   ks::aligned(base, 4) && ks::aligned(post_logits, 4) && ks::aligned(res_logits, 4),
               "ks_mhc_input: x and h must be 16-byte aligned, the fp32 buffers 4-byte aligned");
  const size_t need = ks_mhc_input_workspace_size(N, C);
  KS_CHECK_ARG(workspace != nullptr && workspace_bytes >= need && ks::aligned(workspace, 4),
               "ks_mhc_input: workspace of %zu bytes required, %zu given", need, workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const ks::ProjPlan p = ks::proj_plan(N, C);
  const int64_t wgs = ks::ceil_div(N, 16 * p.tt) * p.splits;
  KS_CHECK_ARG(wgs < (int64_t(1) << 31), "ks_mhc_input: N=%lld out of range", (long long)N);
  float *part = static_cast<float *>(workspace);
  const dim3 grid(static_cast<unsigned>(wgs)), block(64 * ks::kProjWaves);
  if (p.tt == 1)
    hipLaunchKernelGGL(ks::mhc_proj_kernel<1>, grid, block, 0, st, x, phi, part, N, 4 * C, p.splits, p.steps);
  else if (p.tt == 2)
    hipLaunchKernelGGL(ks::mhc_proj_kernel<2>, grid, block, 0, st, x, phi, part, N, 4 * C, p.splits, p.steps);
  else
    hipLaunchKernelGGL(ks::mhc_proj_kernel<4>, grid, block, 0, st, x, phi, part, N, 4 * C, p.splits, p.steps);
  KS_CHECK_LAUNCH("mhc_proj_kernel");
  hipLaunchKernelGGL(ks::mhc_input_kernel, dim3(static_cast<unsigned>(ks::ceil_div(N, ks::kMhcWaves))),
                     dim3(64 * ks::kMhcWaves), 0, st, x, part, phi, alpha, base, h, post_logits, res_logits, N, C / 8,
                     p.splits, norm_eps);
  KS_CHECK_LAUNCH("mhc_input_kernel");
  return KS_OK;
}

extern "C" int ks_mhc_pre(const uint16_t *x, const float *pre_logits, uint16_t *h, int64_t N, int64_t C,
                          void *stream) {
  ks::last_error().clear();
  int rc = ks::check_mhc(x, N, C, "ks_mhc_pre");
  if (rc != KS_OK) return rc;
  if (N == 0) return KS_OK;
  KS_CHECK_ARG(pre_logits && h, "ks_mhc_pre: null pointer");
  KS_CHECK_ARG(ks::aligned(x, 16) && ks::aligned(h, 16) && ks::aligned(pre_logits, 16),
               "ks_mhc_pre: x and h must be 16-byte aligned, pre_logits 16-byte aligned");
  hipLaunchKernelGGL(ks::mhc_pre_kernel, dim3(static_cast<unsigned>(ks::ceil_div(N, ks::kMhcWaves))),
                     dim3(64 * ks::kMhcWaves), 0, static_cast<hipStream_t>(stream), x, pre_logits, h, N, C / 8);
  KS_CHECK_LAUNCH("mhc_pre_kernel");
  return KS_OK;
}

extern "C" int ks_mhc_post(const uint16_t *x, const uint16_t *f, const float *res_logits, const float *post_logits,
                           uint16_t *out, int64_t N, int64_t C, int32_t sinkhorn_iters, float eps, void *stream) {
  ks::last_error().clear();
  int rc = ks::check_mhc(x, N, C, "ks_mhc_post");
  if (rc != KS_OK) return rc;
  KS_CHECK_ARG(sinkhorn_iters >= 1, "ks_mhc_post: sinkhorn_iters must be >= 1");
  if (N == 0) return KS_OK;
  KS_CHECK_ARG(f && res_logits && post_logits && out, "ks_mhc_post: null pointer");
  KS_CHECK_ARG(ks::aligned(x, 16) && ks::aligned(f, 16) && ks::aligned(out, 16) && ks::aligned(res_logits, 16) &&
                   ks::aligned(post_logits, 16),
               "ks_mhc_post: every buffer must be 16-byte aligned");
  hipLaunchKernelGGL(ks::mhc_post_kernel, dim3(static_cast<unsigned>(ks::ceil_div(N, ks::kMhcWaves))),
                     dim3(64 * ks::kMhcWaves), 0, static_cast<hipStream_t>(stream), x, f, res_logits, post_logits, out,
                     N, C / 8, static_cast<int>(sinkhorn_iters), eps);
  KS_CHECK_LAUNCH("mhc_post_kernel");
  return KS_OK;
}
