// Indexer score kernel (gfx950): bf16 MFMA q.k^T, exact bf16 rounding of every dot, ReLU, head-weighted
// reduction in the canonical order, causal mask.
//
// Semantics: baseline/indexer.py:176-193 (einsum -> relu_ -> * weights -> sum over heads -> -inf mask),
// replacing the reference megakernel optimized/indexer_project/op_kernel/fused_indexer_qk_reduce.asc:1-24,
// 368-428 (cube GEMM + vector head reduction).  Bit-exact contract (include/kswift.h): each dot is the
// exact real dot product rounded once to bf16; heads are summed in four groups g = (h/4) % 4, each in
// increasing h with fma (fp32 weights), then (G0 + G1) + (G2 + G3).
//
// Work decomposition: a 512-lane workgroup = 8 waves = 8 queries x a block of 256 keys.  The key block is
// staged once in LDS (64 KiB; rows past T unused) behind the kernel's only barrier; from there each wave runs
// independently.  A wave keeps its query's rows in VGPRs as MFMA A-fragments and walks the block in
// 16-key tiles with v_mfma_f32_16x16x32_bf16 (M = 16 heads, N = 16 keys, 4 k-steps), issuing the next
// tile's MFMAs before the current tile's epilogue.  LDS rows use a 16-byte XOR swizzle (chunk c of row r
// at c ^ (r & 15)), so 16 lanes reading one chunk of 16 rows hit 16 distinct bank groups.  In the MFMA
// output layout lane l holds heads 16m + 4(l/16) + r (r = 0..3) of key l % 16, i.e. exactly the canonical
// head group g = l/16, so the head sum runs in-lane and two permlane swaps finish ((G0+G1)+(G2+G3)).
//
// Exactness: the MFMA fp32 sum A differs from the exact dot by at most the half-width
//   delta = C * 2^-23 * (||q_h|| + 2^-122)(max_t ||k_t|| + 2^-122) + 2^-144   (C = score_bound_c(D): 13 for
//   D = 128, 9 for D = 64),
// derived from the instruction's accumulation (see dot_halfwidth), so the relu'd bf16 value is exact when
// RNE(A - delta) and RNE(A + delta) agree after the ReLU (one packed convert and one packed max per pair of
// dots and interval end).  Keys with a disagreeing ("near-tie") dot are deferred: both interval ends of all
// their head groups go to a per-wave LDS list, and when the list fills (and at the end) the near-tie dots
// are recomputed exactly, 16 at a time with 4 lanes per dot, and the affected scores rewritten.  Per-row
// spans from the statistics pass prove every partial sum of the exact dot representable in a double
// (span_q + span_k <= 52); up to 84 a hi/lo split keeps both halves exact; beyond that an integer
// accumulator (exact_dot_wide_bf16) computes the dot.  A wave whose norms could overflow inside the MFMA
// ((||q|| ||k|| >= 2^126) treats every dot as a near tie.
//
// Bound mode (BOUND, bounded_scores) writes an approximate score and a bound U on its distance from the exact one, for a
// selection that needs only the scores of its top k exactly; with few queries a batch (FEW) the waves of a workgroup
// share the keys of one query.
//
// FP8 keys (F8, bound mode): k holds e4m3 codes with one fp32 scale per row, read directly (half the bytes of
// bf16 rows) and dequantised in registers to the bf16 rows the contract defines, bf16(fp32(value * scale)), before
// the key block is staged in LDS; the rest of the kernel is the bf16 one.  (q arrives dequantised: each query's
// rows are read by every key block's workgroup, T / 256 of them, so they are converted once, by the statistics
// pass, while a key block is read by S / 8 workgroups.)
#include "common.h"
#include "indexer_common.h"
#include "indexer_exact.h"

#include <type_traits>

namespace ks {
namespace {


constexpr int kQW = 8;        // queries (= waves) per workgroup
constexpr int kThreads = kQW * 64;
constexpr int kKR = kScoreKeyBlock;  // keys per workgroup
constexpr int64_t kFewQueries = 4;       // queries a batch up to which the few-queries form runs
constexpr int64_t kFewTargetWgs = 2048;  // its workgroups, about
constexpr int kEntCap = 32;   // deferred key entries per wave (flushed before another 16 could overflow them)
static_assert(kEntCap >= 16, "16 listed keys are resolved at a time");
static_assert(4 * kEntCap <= 255, "list entries hold the (entry, group) pair in 8 bits");
constexpr int kDotCap = 256;  // near-tie dots listed at a time per wave

// Context of one key whose score depends on a near-tie dot: for the four head groups, the relu'd bf16
// values of the two interval ends (packed pairs, 2 HT per group; they differ exactly at the near-tie slots).
// Sized by the head count, so that fewer heads leave LDS for a second workgroup per CU.
template <int HT>
struct alignas(16) KeyEntry {
  uint32_t pl[4][2 * HT];
  uint32_t ph[4][2 * HT];
  int32_t key;
  int32_t pad[3];
};

template <int KD, int HT>
struct ScoresLds {
  uint4 k[kKR * KD / 8];             // swizzled key block of this workgroup (KD / 8 16-byte chunks per key)
  uint16_t kstep[HT == 1 ? kKR : 0][KD / 8];  // 16 heads: per key, the step exponents of |k| (step_exponent_pow2 of
                                              // each 16-byte chunk: a chunk is one accumulation step)
  uint8_t klist[kQW][kKR];           // per wave: block rows of the keys holding a near-tie dot (a wave's tiles
                                     // defer at most every key of the block)
  KeyEntry<HT> ent[HT == 1 ? 0 : kQW][kEntCap];  // 16 heads: the resolution keeps its keys' values in registers
  uint32_t dots[kQW][kDotCap];       // near-tie dots: head << 24 | key row << 16 | pair << 4 | slot,
                                     // pair = 4 entry + group
  int32_t kspan[kKR];                // row statistics of the key block and of each wave's query rows, for
  float knorm[kKR];                  // the exact recomputation (no global loads there)
  int32_t qspan[kQW][64];
  float qnorm[kQW][64];
  float dl[kQW][64];                 // each wave's interval half-widths, one per head
  float w[kQW][64];                  // each wave's head weights (fp32)
};

// Canonical sum of one lane's head group (heads 16 m + 4 g + r, m = 0 .. HT - 1, r = 0 .. 3, in that order) from
// the relu'd bf16 values word(2 m + r / 2) (packed pairs): fp32 weights, G = fma(r_h, w_h, G); bf16 weights,
// G = G + bf16(r_h w_h), the two products of a pair rounded together by one v_cvt_pk_bf16_f32 (RNE, the same
// results as the software rounding for every non-NaN value) and added in head order.
template <int HT, bool WBF, typename Word>
__device__ __forceinline__ float group_sum(Word word, const float (&wv)[HT][4]) {
  float G = 0.f;
#pragma unroll
  for (int m = 0; m < HT; ++m)
#pragma unroll
    for (int rp = 0; rp < 2; ++rp) {
      const uint32_t p2 = word(2 * m + rp);
      if constexpr (WBF) {
        const uint32_t pr = cvt_pk_bf16(unpack_lo(p2) * wv[m][2 * rp], unpack_hi(p2) * wv[m][2 * rp + 1]);
        G = G + unpack_lo(pr);
        G = G + unpack_hi(pr);
      } else {
        G = __builtin_fmaf(unpack_lo(p2), wv[m][2 * rp], G);
        G = __builtin_fmaf(unpack_hi(p2), wv[m][2 * rp + 1], G);
      }
    }
  return G;
}

// Exclusive prefix sum over the 64 lanes of a wave of values below 2^NB, and the wave's total: one ballot per bit
// and the count of the lanes below (mbcnt), with no data moved between lanes.
template <int NB>
__device__ __forceinline__ uint32_t wave_excl_scan_bits(uint32_t v, uint32_t &total) {
  uint32_t pre = 0, tot = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const uint64_t m = __builtin_amdgcn_ballot_w64((v >> b) & 1u);
    pre += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u))
           << b;
    tot += static_cast<uint32_t>(__builtin_popcountll(m)) << b;
  }
  total = tot;
  return pre;
}

// A score's bf16 rounding (bf16 weights) with the hardware conversion: RNE, the same as the software rounding for
// every non-NaN value.
__device__ __forceinline__ float round_score_bf16(float x) { return unpack_lo(cvt_pk_bf16(x, x)); }

// Near-tie slot bits (16 per head group) of an entry: positions where the two interval ends differ.
template <int HT>
__device__ __forceinline__ uint32_t entry_mask(const KeyEntry<HT> &en, int gg) {
  uint32_t m = 0;
#pragma unroll
  for (int p = 0; p < 2 * HT; ++p) {
    const uint32_t x = en.pl[gg][p] ^ en.ph[gg][p];
    m |= ((x & 0xFFFFu) ? 1u : 0u) << (2 * p);
    m |= ((x >> 16) ? 1u : 0u) << (2 * p + 1);
  }
  return m;
}

// The exact value (RNE to bf16, before the ReLU) of the dot of head h's q row and key row kl of the block,
// computed by a quad of lanes (this lane: quarter `sub`); every lane of the wave calls it together (the path
// choices are ballots).  16 heads: quarter `sub` takes the 16-byte chunks 4c + sub, which lane h + 16 sub holds as
// its A-fragment qa[0][c] (read with ds_bpermute); more heads: the chunks kLC sub + c, read from global memory
// (L2-resident).  scur: the span sum that decided the path (> 84: the integer accumulator).
template <int HT, int KD>
__device__ __forceinline__ uint16_t quad_exact_dot(ScoresLds<KD, HT> &L, int wave, int sub, int h, int kl,
                                                   const uint16_t *__restrict__ q, QSplit qsp,
                                                   const uint4 (&qa)[HT][KD / 32], int64_t qrow0, int &scur) {
  constexpr int kC = KD / 8, kLC = KD / 32;  // 16-byte chunks per key row; chunks per lane
  // the q rows this lane reads from memory: its quarter (elements KD/4 sub ..) lies wholly on one side of a
  // split (QSplit boundaries are 32-aligned)
  const uint16_t *qsrc = (qsp.rot != nullptr && (KD / 4) * sub >= qsp.lo && (KD / 4) * sub < qsp.hi) ? qsp.rot : q;
  uint4 qcur[kLC], kcur[kLC];
  if constexpr (HT == 1) {
    const int src = 4 * (h + 16 * sub);
    auto bp = [&](uint32_t v) { return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(v))); };
#pragma unroll
    for (int c = 0; c < kLC; ++c) {
      qcur[c] = make_uint4(bp(qa[0][c].x), bp(qa[0][c].y), bp(qa[0][c].z), bp(qa[0][c].w));
      kcur[c] = L.k[kl * kC + ((4 * c + sub) ^ (kl & (kC - 1)))];
    }
  } else {
    const uint4 *qp = reinterpret_cast<const uint4 *>(qsrc + (qrow0 + h) * KD + (KD / 4) * sub);
#pragma unroll
    for (int c = 0; c < kLC; ++c) qcur[c] = qp[c];
#pragma unroll
    for (int c = 0; c < kLC; ++c) kcur[c] = L.k[kl * kC + ((kLC * sub + c) ^ (kl & (kC - 1)))];
  }
  scur = L.qspan[wave][h] + L.kspan[kl];
  uint16_t r;
  if (__builtin_amdgcn_ballot_w64(scur > 52) == 0ull) {
    // every partial sum is a multiple of the smallest product LSB and below 2^53 of it: exact doubles
    // in any order
    double a0 = 0.0, a1 = 0.0;
#pragma unroll
    for (int c = 0; c < kLC; ++c) {
      const uint32_t qw[4] = {qcur[c].x, qcur[c].y, qcur[c].z, qcur[c].w};
      const uint32_t kw[4] = {kcur[c].x, kcur[c].y, kcur[c].z, kcur[c].w};
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        a0 = __builtin_fma(static_cast<double>(unpack_lo(qw[p])), static_cast<double>(unpack_lo(kw[p])), a0);
        a1 = __builtin_fma(static_cast<double>(unpack_hi(qw[p])), static_cast<double>(unpack_hi(kw[p])), a1);
      }
    }
    const double sum = quad_sum_f64(a0 + a1);
    const bool outside = sum != 0.0 && !(fabs(sum) >= 0x1p-126 && fabs(sum) < 0x1p127);
    if (__builtin_amdgcn_ballot_w64(outside) == 0ull) {
      r = round_to_bf16_fast(sum);
    } else {
      r = round_dir_to_bf16(sum, 0);
    }
  } else {
    // wide dynamic range: products above / below 2^(top - 38) accumulate separately, each exactly
    const int span_sum = scur;
    const int top_sum = frexp_exp(L.qnorm[wave][h]) + frexp_exp(L.knorm[kl]);
    const bool split = span_sum > 52;
    const double thr = split ? ldexp(1.0, top_sum - 38) : 0.0;
    double hi = 0.0, lo = 0.0;
    // rare path, kept register-light: one dword of q and k per step, re-read from memory
    const uint32_t *q32 = reinterpret_cast<const uint32_t *>(qsrc + (qrow0 + h) * KD + (KD / 4) * sub);
#pragma unroll 1
    for (int j = 0; j < 4 * kLC; ++j) {
      const uint32_t qw = q32[j];
      const uint32_t kw =
          reinterpret_cast<const uint32_t *>(&L.k[kl * kC + ((kLC * sub + (j >> 2)) ^ (kl & (kC - 1)))])[j & 3];
      const double p0 = static_cast<double>(unpack_lo(qw)) * static_cast<double>(unpack_lo(kw));
      const double p1 = static_cast<double>(unpack_hi(qw)) * static_cast<double>(unpack_hi(kw));
      if (!split || fabs(p0) >= thr) hi += p0; else lo += p0;
      if (!split || fabs(p1) >= thr) hi += p1; else lo += p1;
    }
    r = round2_to_bf16(quad_sum_f64(hi), quad_sum_f64(lo));
  }
  if (scur > 84) {
    // wider still (the whole quad takes this branch): the integer accumulator, any range
    const uint32_t *q32 = reinterpret_cast<const uint32_t *>(qsrc + (qrow0 + h) * KD);  // part `sub` of it
    r = exact_dot_wide_bf16<KD, 4>(
        [&](int j) { return q32[j]; },
        [&](int j) {
          return reinterpret_cast<const uint32_t *>(&L.k[kl * kC + ((j >> 2) ^ (kl & (kC - 1)))])[j & 3];
        },
        sub);
  }
  return r;
}

// Exact recomputation of the deferred near-tie dots of one wave, then of the affected scores.
template <int HT, int KD, bool WBF>
__device__ void flush_entries(ScoresLds<KD, HT> &L, int wave, int lane, int nent, const uint16_t *__restrict__ q,
                              const uint4 (&qa)[HT][KD / 32], int64_t qrow0, float *orow, int64_t limit, int T, int kb0,
                              const float (&wv)[HT][4], uint32_t &n_exact, uint32_t &n_unres, QSplit qsp) {
  KeyEntry<HT> *E = L.ent[wave];
  uint32_t *D = L.dots[wave];
  const int g = lane >> 4, l16 = lane & 15;
  // 1. near-tie masks of the (entry, group) pairs, pair = 4 * entry + group; taken before any patching
  const int npairs = 4 * nent;
  auto key_row = [&](int pair) {  // row of the entry's key in the LDS block (entries hold keys of the block)
    return static_cast<uint32_t>(min(max(E[pair >> 2].key - kb0, 0), kKR - 1));
  };
  // pairs are taken 64 at a time: pair 64 i + lane in set i
  constexpr int kSets = (4 * kEntCap + 63) / 64;
  uint32_t mset[kSets], rset[kSets], cset[kSets], first[kSets];
  uint32_t ndots_u = 0;
#pragma unroll
  for (int i = 0; i < kSets; ++i) {
    const int pair = 64 * i + lane;
    mset[i] = pair < npairs ? entry_mask<HT>(E[pair >> 2], pair & 3) : 0u;
    rset[i] = pair < npairs ? key_row(pair) : 0u;
    cset[i] = __builtin_popcount(mset[i]);  // at most 4 HT near-tie slots per pair
    uint32_t tot;
    first[i] = ndots_u + wave_excl_scan_bits<HT == 1 ? 3 : HT == 2 ? 4 : 5>(cset[i], tot);  // list position of the
    ndots_u += tot;                                                                       // pair's first dot
  }
  const int ndots = static_cast<int>(ndots_u);
  n_exact += ndots_u;
  // 2. the dot list, kDotCap at a time: exact dots, 16 per pass, 4 lanes per dot (lane quarter `sub` owns
  //    elements KD/4 sub .. KD/4 (sub + 1) - 1); the exact relu'd value replaces the pl value of its slot.
  //    List entry: head (slot s of pair (entry, group gg) is head 16 (s >> 2) + 4 gg + (s & 3)), key row,
  //    pair and slot, so that one LDS read locates both operands.
  constexpr int kC = KD / 8, kLC = KD / 32;  // 16-byte chunks per key row; chunks per lane
  auto pack = [](uint32_t pair, uint32_t row, int bit) {
    const uint32_t h = 16u * (bit >> 2) + 4u * (pair & 3u) + (bit & 3);
    return (h << 24) | (row << 16) | (pair << 4) | static_cast<uint32_t>(bit);
  };
  for (int base = 0; base < ndots; base += kDotCap) {
#pragma unroll
    for (int i = 0; i < kSets; ++i) {
      uint32_t mm = mset[i];
      int pos = static_cast<int>(first[i]) - base;
      while (mm) {
        const int bit = __builtin_ctz(mm);
        mm &= mm - 1;
        if (pos >= 0 && pos < kDotCap) D[pos] = pack(static_cast<uint32_t>(64 * i + lane), rset[i], bit);
        ++pos;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int nd = min(kDotCap, ndots - base);
    const int dq = lane >> 2, sub = lane & 3;
    for (int b0 = 0; b0 < nd; b0 += 16) {
      // list entry of this quad (idle quads repeat the last one; the result is identical)
      const uint32_t dcur = D[min(b0 + dq, nd - 1)];
      const int h = static_cast<int>(dcur >> 24), kl = static_cast<int>((dcur >> 16) & 255u);
      const int pr = static_cast<int>((dcur >> 4) & 255u), slot = static_cast<int>(dcur & 15u);
      int scur;
      const uint16_t r = quad_exact_dot<HT, KD>(L, wave, sub, h, kl, q, qsp, qa, qrow0, scur);
      const uint32_t rv = (r & 0x8000) ? 0u : r;  // ReLU (also maps -0 to +0)
      if (sub == 0 && b0 + dq < nd) {
        uint16_t *half = reinterpret_cast<uint16_t *>(&E[pr >> 2].pl[pr & 3][slot >> 1]) + (slot & 1);
        *half = static_cast<uint16_t>(rv);
        if (scur > 84) ++n_unres;  // counted: dots that needed the integer accumulator
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // 3. scores of the deferred keys from the corrected values: lane (row g, column e) sums group g of entry
  //    e with this lane's own head weights, the rows combine as in the main loop
  for (int eb = 0; eb < nent; eb += 16) {
    const int e = min(eb + l16, nent - 1);
    const float G = group_sum<HT, WBF>([&](int i) { return E[e].pl[g][i]; }, wv);
    const float tot = combine_groups(G);
    const int key = E[e].key;
    if (g == 0 && eb + l16 < nent && key < T) orow[key] = (key < limit) ? (WBF ? round_score_bf16(tot) : tot) : -INFINITY;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Shared memory of the bound-emitting form: the key block (few queries: the query's rows instead), and the head weights
// of each wave's query (few: of the one query) as bf16 values: high part, low part, upper bound of |w|, zero.
template <int KD, bool FEW>
struct ScoresLdsBound {
  uint4 k[(FEW ? 64 : kKR) * KD / 8];
  uint16_t wf[FEW ? 1 : kQW][4][64];
};

// Waves per SIMD a kernel form is built for.  The bound kernel runs grids of several workgroups per CU: at
// up to 128 VGPRs and 70 KiB of LDS two of them share a CU, so that one's prologue loads overlap the other's tiles (64
// queries x 32768 keys: 40.7 us, against 49.1 at 147 VGPRs with the next tile's MFMAs issued a tile ahead).  The exact
// kernel at 16 heads of 64 dims (the drop-in shape: 4 dots per lane and tile, a tile one chain of dependent steps) at
// up to 128 VGPRs and 57 KiB of LDS does the same: four waves per SIMD hide each other's tile latency.
template <int HT, int KD, bool BOUND, bool FEW>
constexpr int score_waves() { return BOUND ? (FEW ? 2 : 4) : (!BOUND && HT == 1 && KD == 64) ? 4 : 1; }

// e4m3 key chunks of the staging loop, dequantised to the contract's bf16 rows: 16 codes per load, rows past nk zero.
template <int KD, int NV>
__device__ __forceinline__ void stage_fp8_keys(uint4 *kl, const uint4 (&kv)[NV], const float (&ksv)[NV], int tid, int nk) {
  constexpr int kC = KD / 8;
  // one conversion form for the whole wave: the one-instruction form when every scale it holds allows it
  bool p2 = true;
#pragma unroll
  for (int it = 0; it < NV; ++it) p2 = p2 & fp8_scale_pow2(ksv[it]);  // no short-circuit: no branches
  p2 = __builtin_amdgcn_ballot_w64(!p2) == 0ull;
  auto stage = [&](auto POW2) {
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int lin = it * kThreads + tid;
      const int kr = lin / (kC / 2), ch = 2 * (lin % (kC / 2));
      const uint32_t msk = kr < nk ? 0xFFFFFFFFu : 0u;
      const uint4 lo = fp8_dequant8<decltype(POW2)::value>(make_uint2(kv[it].x, kv[it].y), ksv[it]);
      const uint4 hi = fp8_dequant8<decltype(POW2)::value>(make_uint2(kv[it].z, kv[it].w), ksv[it]);
      kl[kr * kC + (ch ^ (kr & (kC - 1)))] = make_uint4(lo.x & msk, lo.y & msk, lo.z & msk, lo.w & msk);
      kl[kr * kC + ((ch + 1) ^ (kr & (kC - 1)))] = make_uint4(hi.x & msk, hi.y & msk, hi.z & msk, hi.w & msk);
    }
  };
  if (p2)
    stage(std::true_type{});
  else
    stage(std::false_type{});
}

// Sum of a value over the 64 lanes (the same bits in every lane: each exchange adds the same two values).
__device__ __forceinline__ float wave_sum_f32(float x) {
#define KS_ADD(S_) x += __builtin_bit_cast(float, lane_xor<S_>(__builtin_bit_cast(uint32_t, x)));
  KS_ADD(32) KS_ADD(16) KS_ADD(8) KS_ADD(4) KS_ADD(2) KS_ADD(1)
#undef KS_ADD
  return x;
}

// What a row's bounds are made of (the derivation is below): bf16 parts of the head weights, U = kC1 sum(w_up p) +
// (the dots' own errors) + kC2 |S|, and the store of 64 keys' scores and bounds.
struct WeightParts {
  float up;  // w_up
  uint16_t hi, lo, up16;
};
template <bool WBF>
__device__ __forceinline__ WeightParts weight_parts(float w) {
  WeightParts p;
  p.up16 = w == 0.f ? 0 : max(bf16_abs_round_up(w), static_cast<uint16_t>(17 << 7));  // 2^-110
  p.up = bf16_to_f32(p.up16);
  const float hi = bf16_to_f32(static_cast<uint16_t>(cvt_pk_bf16(w, w) & 0xFFFFu));
  p.hi = static_cast<uint16_t>(__builtin_bit_cast(uint32_t, hi) >> 16);
  p.lo = WBF ? 0 : static_cast<uint16_t>(cvt_pk_bf16(w - hi, 0.f) & 0xFFFFu);
  return p;
}
template <bool WBF>
__device__ __forceinline__ void store_bounded(float *__restrict__ orow, float *__restrict__ urow, int key, bool in,
                                              bool live, f32x4_t sums, float dsum, bool forced) {
  constexpr float kC1 = WBF ? (0x1p-7f + 0x1p-8f) * 1.0625f : 0x1p-7f * 1.0625f;
  constexpr float kC2 = WBF ? 0x1p-8f * 1.0625f : 0x1p-21f;
  float sc = sums[0] + sums[1];
  float u = __builtin_fmaf(kC2, fabsf(sc), __builtin_fmaf(kC1, sums[2], dsum)) + 0x1p-120f;
  if (forced || !(fabsf(sc) + u < 3e38f)) {  // no statement about the score: it is always recomputed
    sc = 0.f;
    u = __builtin_inff();
  }
  if (in) {
    orow[static_cast<uint32_t>(key)] = live ? sc : -INFINITY;
    urow[static_cast<uint32_t>(key)] = live ? u : 0.f;
  }
}
// The head-sum A operand of tile j: the lanes of rows 4 j .. 4 j + 3 keep wa (row l16 holds part l16 & 3 of the weights),
// the others are zero.  Made in the loop: hoisted, the four forms would take 32 registers.
__device__ __forceinline__ uint4 tile_weights(uint4 wa, int j) {
  uint64_t rows = 0x000F000F000F000Full << (4 * j);
  asm volatile("" : "+s"(rows));
  const bool in = __builtin_amdgcn_inverse_ballot_w64(rows);
  return make_uint4(in ? wa.x : 0u, in ? wa.y : 0u, in ? wa.z : 0u, in ? wa.w : 0u);
}
// wa for heads 32 hh + 4 g + 0 .. 3 and 16 above (the k-slots 8 g .. 8 g + 7 of the relu'd dots packed per lane)
__device__ __forceinline__ uint4 head_weights(const uint16_t (&wf)[4][64], int hh, int l16, int g) {
  const uint32_t *wr = reinterpret_cast<const uint32_t *>(wf[l16 & 3]);
  const int h0 = 32 * hh + 4 * g, h1 = h0 + 16;
  return make_uint4(wr[h0 / 2], wr[h0 / 2 + 1], wr[h1 / 2], wr[h1 / 2 + 1]);
}
// sums += the weighted relu'd bf16 dots of one 16-key tile (tile j of its four), from the tile's MFMA sums
__device__ __forceinline__ f32x4_t add_tile(const f32x4_t (&acc)[4], const uint4 (&wa)[2], int j, f32x4_t sums) {
  uint32_t p[8];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int rp = 0; rp < 2; ++rp) p[2 * m + rp] = cvt_relu_pk(acc[m][2 * rp], acc[m][2 * rp + 1]);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
    sums = mfma16(tile_weights(wa[hh], j), make_uint4(p[4 * hh], p[4 * hh + 1], p[4 * hh + 2], p[4 * hh + 3]), sums);
  return sums;
}
__device__ __forceinline__ uint32_t row_scale(float upqn, float kns) {  // the same bits in every lane and workgroup
  return __builtin_bit_cast(uint32_t, wave_sum_f32(upqn) * wave_max_f32(kns)) & 0x7FFFFFFFu;
}

// The bound-emitting form (64 heads): per (query, key) a score S and a bound U with |exact score - S| <= U, for a
// selection that computes exactly only the scores that can reach its top k.  No dot is certified here: with A the MFMA
// sum of a dot, p = max(bf16(A), 0) is within one bf16 rounding of each side of the exact relu'd value r (at most 2^-8 of
// the value, or, below 2^-126, half a step of 2^-133),
//   |p - r| <= delta + 2^-8 |A| + 2^-8 (|A| + delta) + 2 2^-134 <= 2^-7 (1 + 2^-7) p + (1 + 2^-7) delta + 2^-132
// (delta: dot_halfwidth; for A <= 0, p = 0 and r <= (1 + 2^-8) delta + 2^-134), so that
//   S = sum_h w_h p_h,   U = c1 sum_h w_up p_h + sum_h w_up (delta_h + 2^-132) + c2 |S|,
// w_up a bf16 value >= |w_h| (and >= 2^-110 where w_h != 0, so that the low part of a tiny weight, lost below the bf16
// range, stays under 2^-24 w_up).  The head sums run on the MFMA too: p packs into the B operand as it is (lane (key, g)
// holds the heads of k-slots 8 g .. + 7), and the A operand's rows hold w's high and low bf16 parts and w_up.  Products
// are exact and the sums lose under 2^-19 of w_up p; w - hi - lo is under 2^-16 |w|.
//   c1 = 2^-7 (1 + 2^-4) covers (1 + 2^-7) with those and the canonical sum's own roundings (2^-18 of |w| r);
//   bf16 weights: each product and the score are rounded to bf16, 2^-8 of |w| r and of |S| + U more:
//   c1 = (2^-7 + 2^-8)(1 + 2^-4), c2 = 2^-8 (1 + 2^-4) in place of c2 = 2^-21 (the ends S -/+ U may be rounded).
// Four 16-key tiles share one accumulator: tile j's A operand holds the weight rows at 4 j .. 4 j + 2 and zeros
// elsewhere, so that lane (l16, g) ends with the sums of key 16 g + l16 and the epilogue serves 64 keys at once.
// Against certifying every dot (two interval ends per dot, a rounding test and the canonical sum in VALU: ~105 VALU
// instructions per tile, VALU-bound: 71.9 us at 64 queries x 32768 keys), this takes ~45; 40.7 us, 844 TFLOP/s, the
// matrix cores busy ~45% of it (18 MFMAs per tile, 17.7 us of them) and the rest the workgroups' prologues (the block's
// 64 KiB of keys and 128 KiB of query rows).  128 queries x 4096 keys, one workgroup per CU: 23.7 -> 21.0 us.
template <bool WBF, bool F8>
__device__ __forceinline__ void bounded_scores(ScoresLdsBound<128, false> &L, const uint16_t *__restrict__ q,
                                               const uint16_t *__restrict__ k, const void *__restrict__ w,
                                               const float *__restrict__ qn, const float *__restrict__ kn,
                                               float *__restrict__ scores, int64_t S, int T, int64_t kbs, int64_t kns_stride, int causal,
                                               int64_t start_pos, int ratio, float bound_c, float *__restrict__ bounds,
                                               uint32_t *__restrict__ row_state, const float *__restrict__ ksc, int kblk,
                                               int qgrp) {
  constexpr int KD = 128, HT = 4, H = 64, kC = KD / 8;
  const uint8_t *__restrict__ k8 = reinterpret_cast<const uint8_t *>(k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t b = blockIdx.z;
  const int kb0 = kblk * kKR;
  const int nk = min(kKR, T - kb0);
  const int64_t s = static_cast<int64_t>(qgrp) * kQW + wave;
  const bool s_ok = s < S;
  const int64_t krow0 = b * kbs + kb0;  // first key row of this workgroup

  // Every prologue load goes out before the first wait, the key block ahead of every q load of the workgroup (the
  // memory pipeline serves a CU's loads in issue order); indices are clamped, values masked afterwards.
  const int64_t qrow0 = (b * S + (s_ok ? s : 0)) * H;
  const float *__restrict__ knb = kn + b * kns_stride + kb0;
  float kn4[kKR / 64];
#pragma unroll
  for (int j = 0; j < kKR / 64; ++j) {
    const int kj = lane + 64 * j;
    kn4[j] = knb[static_cast<uint32_t>(kj < nk ? kj : nk - 1)];
  }
  // 64 norms spread over the batch's keys: the scale of the row's histogram (the same for every key block)
  const float kns = (kn + b * kns_stride)[static_cast<uint32_t>((static_cast<int64_t>(lane) * T) >> 6)];
  const float qn_v = (qn + qrow0)[static_cast<uint32_t>(lane)];
  const float w_v = WBF ? bf16_to_f32((static_cast<const uint16_t *>(w) + qrow0)[static_cast<uint32_t>(lane)])
                        : (static_cast<const float *>(w) + qrow0)[static_cast<uint32_t>(lane)];
  constexpr int kKL = kKR * kC / kThreads;  // 16-byte key chunks per thread (F8: kKL / 2 loads of 16 codes)
  constexpr int kKV = F8 ? kKL / 2 : kKL;
  uint4 kv[kKV];
  float ksv[F8 ? kKV : 1];
#pragma unroll
  for (int it = 0; it < kKV; ++it) {
    const int lin = it * kThreads + tid;
    if constexpr (F8) {
      const int kr = lin / (kC / 2), ch2 = lin % (kC / 2);
      const int64_t row = krow0 + (kr < nk ? kr : nk - 1);
      kv[it] = *reinterpret_cast<const uint4 *>(k8 + row * KD + ch2 * 16);
      ksv[it] = ksc[row];
    } else {
      const int kr = lin / kC, ch = lin % kC;
      kv[it] = *reinterpret_cast<const uint4 *>(k + krow0 * KD + static_cast<uint32_t>((kr < nk ? kr : nk - 1) * KD + ch * 8));
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  uint4 qa[HT][KD / 32];  // query rows as MFMA A-fragments, loaded in the order the first tile uses them
#pragma unroll
  for (int kk = 0; kk < KD / 32; ++kk)
#pragma unroll
    for (int m = 0; m < HT; ++m)
      qa[m][kk] = *reinterpret_cast<const uint4 *>(q + qrow0 * KD + static_cast<uint32_t>((16 * m + l16) * KD + 32 * kk + 8 * g));

  float knm = 0.f;
#pragma unroll
  for (int j = 0; j < kKR / 64; ++j) knm = fmaxf(knm, lane + 64 * j < nk ? kn4[j] : 0.f);
  knm = wave_max_f32(knm);
  // lane h: head h's weight parts and its share of the row's bound
  const WeightParts wp = weight_parts<WBF>(w_v);
  L.wf[wave][0][lane] = wp.hi;
  L.wf[wave][1][lane] = wp.lo;
  L.wf[wave][2][lane] = wp.up16;
  L.wf[wave][3][lane] = 0;
  const float dl = dot_halfwidth(qn_v, knm, bound_c);
  const bool forced = __builtin_amdgcn_ballot_w64(dl == __builtin_inff()) != 0ull;
  // sum_h w_up (delta_h + 2^-132), (1 + 2^-7) and the fp32 sums covered
  const float dsum = wave_sum_f32(wp.up * (dl + 0x1p-132f)) * 1.03125f;
  const uint32_t mrow = row_scale(wp.up * qn_v, kns);

  if constexpr (F8) {
    stage_fp8_keys<KD>(L.k, kv, ksv, tid, nk);
  } else {
    // rows past T are zeroed: with the loaded values used only by the LDS stores, the compiler would sink their loads
    // below the q loads and the load-ordering barrier (a CPU test checks the placement in the compiled code)
#pragma unroll
    for (int it = 0; it < kKL; ++it) {
      const int lin = it * kThreads + tid;
      const int kr = lin / kC, ch = lin % kC;
      const uint32_t msk = kr < nk ? 0xFFFFFFFFu : 0u;
      L.k[kr * kC + (ch ^ (kr & (kC - 1)))] = make_uint4(kv[it].x & msk, kv[it].y & msk, kv[it].z & msk, kv[it].w & msk);
    }
  }
  // the only barrier past the load ordering: LDS writes done, no wait for the q loads
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (!s_ok) return;
  if (kblk == 0 && lane == 0) row_state[2 * (b * S + s) + 1] = mrow;

  const int64_t limit = causal ? (start_pos + s + 1) / ratio : INT64_MAX;
  float *orow = scores + (b * S + s) * T;
  float *urow = bounds + (b * S + s) * T;
  const int64_t lim_rel = limit - kb0;
  const int nlk = lim_rel <= 0 ? 0 : (lim_rel < nk ? static_cast<int>(lim_rel) : nk);  // live keys of the block
  const int nlive = (nlk + 15) / 16;

  const uint4 wa[2] = {head_weights(L.wf[wave], 0, l16, g), head_weights(L.wf[wave], 1, l16, g)};
  auto tile_b = [&](int t, uint4(&bv)[KD / 32]) {
    const int key_l = 16 * t + l16;
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk) bv[kk] = L.k[key_l * kC + ((4 * kk + g) ^ (key_l & (kC - 1)))];
  };
  auto tile_mfma = [&](const uint4(&bv)[KD / 32], f32x4_t(&acc)[HT]) {
#pragma unroll
    for (int m = 0; m < HT; ++m) acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk)
#pragma unroll
      for (int m = 0; m < HT; ++m) acc[m] = mfma16(qa[m][kk], bv[kk], acc[m]);
  };
  if (nlive > 0) {
    // tiles past the last live one repeat it (their keys are masked)
    const int last = nlive - 1;
    uint4 bv[KD / 32];
    tile_b(0, bv);
    for (int t0 = 0; t0 < nlive; t0 += 4) {
      f32x4_t sums = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + j;
        f32x4_t acc[HT];
        tile_mfma(bv, acc);
        tile_b(t + 1 < nlive ? t + 1 : last, bv);
        sums = add_tile(acc, wa, j, sums);
      }
      const int key_l = 16 * t0 + lane;
      store_bounded<WBF>(orow, urow, kb0 + key_l, key_l < nk, key_l < nlk, sums, dsum, forced);
    }
  }
  // keys past the last group of live tiles (at or past the causal limit)
  for (int key_l = 64 * ((nlive + 3) / 4) + lane; key_l < nk; key_l += 64) {
    orow[static_cast<uint32_t>(kb0 + key_l)] = -INFINITY;
    urow[static_cast<uint32_t>(kb0 + key_l)] = 0.f;
  }
}

// Few queries per batch (generation: one new token a sequence): a workgroup takes one query, and its 8 waves take 64-key
// groups of their own, so that no wave idles (with a query per wave, one query would leave seven of eight idle).  No key
// is used twice, so key fragments are read from memory as they are, each tile's registers refilled with the next group's
// tile once its MFMAs are issued; the query's rows are staged once in LDS for the workgroup.  Scores and bounds as above
// (the dots' error from the largest norm of the group's 64 keys).
// 16 single queries over 16382 keys each: 23.5 us (67 MB of keys, 2.9 TB/s), where the exact kernel with a query per wave
// took 176 us.
template <bool WBF, bool F8>
__device__ __forceinline__ void bounded_scores_few(ScoresLdsBound<128, true> &L, const uint16_t *__restrict__ q,
                                                   const uint16_t *__restrict__ k, const void *__restrict__ w,
                                                   const float *__restrict__ qn, const float *__restrict__ kn,
                                                   float *__restrict__ scores, int64_t S, int T, int64_t kbs, int64_t kns_stride,
                                                   int causal, int64_t start_pos, int ratio, float bound_c,
                                                   float *__restrict__ bounds, uint32_t *__restrict__ row_state,
                                                   const float *__restrict__ ksc) {
  constexpr int KD = 128, HT = 4, H = 64, kC = KD / 8;
  const uint8_t *__restrict__ k8 = reinterpret_cast<const uint8_t *>(k);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t b = blockIdx.z, s = blockIdx.y, row = b * S + s;
  const int ngrp = (T + 63) / 64, gstep = 8 * gridDim.x;  // group of this wave: wave + 8 blockIdx.x, then every gstep
  const int64_t limit = causal ? (start_pos + s + 1) / ratio : INT64_MAX;
  const int nlk = limit <= 0 ? 0 : (limit < T ? static_cast<int>(limit) : T);  // live keys of the row
  float *orow = scores + row * T;
  float *urow = bounds + row * T;
  const int64_t qrow0 = row * H;

  // the first group's keys (rows past T read the last one), the query's rows and head data: all in flight together
  uint4 bv[4][KD / 32];
  uint2 bc[F8 ? 4 : 1][KD / 32];
  float bs[F8 ? 4 : 1];
  auto load_tile = [&](int grp, int j) {
    const int key = 64 * grp + 16 * j + l16;
    const int64_t kr = b * kbs + (key < T ? key : T - 1);
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk) {
      if constexpr (F8)
        bc[j][kk] = *reinterpret_cast<const uint2 *>(k8 + kr * KD + 32 * kk + 8 * g);
      else
        bv[j][kk] = *reinterpret_cast<const uint4 *>(k + kr * KD + 32 * kk + 8 * g);
    }
    if constexpr (F8) bs[j] = ksc[kr];
  };
  auto load_norm = [&](int grp) {
    const int key = 64 * grp + lane;
    return kn[b * kns_stride + (key < T ? key : T - 1)];
  };
  int grp = wave + 8 * static_cast<int>(blockIdx.x);
  const int grp0 = grp < ngrp ? grp : ngrp - 1;
  uint4 qv[H * kC / kThreads];
#pragma unroll
  for (int i = 0; i < H * kC / kThreads; ++i) {
    const int idx = tid + i * kThreads;
    qv[i] = *reinterpret_cast<const uint4 *>(q + (qrow0 + idx / kC) * KD + 8 * (idx % kC));
  }
  const float qn_v = (qn + qrow0)[static_cast<uint32_t>(lane)];
  const float w_v = WBF ? bf16_to_f32((static_cast<const uint16_t *>(w) + qrow0)[static_cast<uint32_t>(lane)])
                        : (static_cast<const float *>(w) + qrow0)[static_cast<uint32_t>(lane)];
  const float kns = (kn + b * kns_stride)[static_cast<uint32_t>((static_cast<int64_t>(lane) * T) >> 6)];
  float kg = load_norm(grp0);
#pragma unroll
  for (int j = 0; j < 4; ++j) load_tile(grp0, j);
  __builtin_amdgcn_sched_barrier(0);  // keep the key loads above the staging's waits

#pragma unroll
  for (int i = 0; i < H * kC / kThreads; ++i) {
    const int idx = tid + i * kThreads, h = idx / kC, c = idx % kC;
    L.k[h * kC + (c ^ (h & (kC - 1)))] = qv[i];
  }
  const WeightParts wp = weight_parts<WBF>(w_v);
  L.wf[0][0][lane] = wp.hi;  // every wave writes the same values
  L.wf[0][1][lane] = wp.lo;
  L.wf[0][2][lane] = wp.up16;
  L.wf[0][3][lane] = 0;
  // sum_h w_up (delta_h + 2^-132) = bound_c 2^-23 (knm + pad) sum(w_up (qn + pad)) + (2^-144 + 2^-132) sum(w_up), per
  // group's knm
  const float a1 = wave_sum_f32(wp.up * (qn_v + 0x1p-122f)) * bound_c * 0x1p-23f * 1.03125f;
  const float a2 = wave_sum_f32(wp.up) * 0x1.08p-132f;
  const float qpmax = wave_max_f32(qn_v) + 0x1p-122f;
  const uint32_t mrow = row_scale(wp.up * qn_v, kns);
  if (blockIdx.x == 0 && tid == 0) row_state[2 * row + 1] = mrow;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // LDS writes done, no wait for the key loads
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  uint4 qa[HT][KD / 32];
#pragma unroll
  for (int kk = 0; kk < KD / 32; ++kk)
#pragma unroll
    for (int m = 0; m < HT; ++m) qa[m][kk] = L.k[(16 * m + l16) * kC + ((4 * kk + g) ^ l16)];
  const uint4 wa[2] = {head_weights(L.wf[0], 0, l16, g), head_weights(L.wf[0], 1, l16, g)};

  for (; grp < ngrp; grp += gstep) {
    const int nxt = grp + gstep < ngrp ? grp + gstep : grp;
    const int key = 64 * grp + lane;
    if (64 * grp >= nlk) {  // uniform: every key of the group is masked (and so are the later ones)
      if (key < T) {
        orow[key] = -INFINITY;
        urow[key] = 0.f;
      }
      continue;
    }
    const float kp = wave_max_f32(kg) + 0x1p-122f;
    kg = load_norm(nxt);
    const bool forced = !(qpmax * kp < 0x1p126f);
    const float dsum = __builtin_fmaf(a1, kp, a2);
    f32x4_t sums = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (F8) {
        if (__builtin_amdgcn_ballot_w64(!fp8_scale_pow2(bs[j])) == 0ull) {
#pragma unroll
          for (int kk = 0; kk < KD / 32; ++kk) bv[j][kk] = fp8_dequant8<true>(bc[j][kk], bs[j]);
        } else {
#pragma unroll
          for (int kk = 0; kk < KD / 32; ++kk) bv[j][kk] = fp8_dequant8<false>(bc[j][kk], bs[j]);
        }
      }
      f32x4_t acc[HT];
#pragma unroll
      for (int m = 0; m < HT; ++m) acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KD / 32; ++kk)
#pragma unroll
        for (int m = 0; m < HT; ++m) acc[m] = mfma16(qa[m][kk], bv[j][kk], acc[m]);
      load_tile(nxt, j);
      sums = add_tile(acc, wa, j, sums);
    }
    store_bounded<WBF>(orow, urow, key, key < T, key < nlk, sums, dsum, forced);
  }
}

template <int HT, int KD, bool WBF, bool BOUND, bool FEW = false, bool F8 = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(score_waves<HT, KD, BOUND, FEW>()))) void
indexer_scores_kernel(
    const uint16_t *__restrict__ q, const uint16_t *__restrict__ k, const void *__restrict__ w,
    const float *__restrict__ qn, const int32_t *__restrict__ qsp, const float *__restrict__ kn,
    const int32_t *__restrict__ ksp, float *__restrict__ scores, int64_t S, int T, int64_t kbs, int64_t kns_stride,
    int causal, int64_t start_pos, int ratio, float bound_c, uint32_t *__restrict__ stats, int xcd_pk,
    float *__restrict__ bounds, uint32_t *__restrict__ row_state, const float *__restrict__ ksc, float bound_r, const uint16_t *__restrict__ qsplit_rot, int qsplit_lo,
    int qsplit_hi) {
  constexpr int H = HT * 16;
  constexpr int kC = KD / 8;  // 16-byte chunks per key row
  static_assert(!BOUND || (HT == 4 && KD == 128), "the bound-emitting form is built for 64 heads of 128 dims");
  static_assert(BOUND || !FEW, "the few-queries form emits bounds");
  static_assert(!F8 || BOUND, "FP8 keys are read by the bound-emitting variant");
  // per-dot interval half-widths (step_halfwidth_scale: the step-weighted magnitude sum and the step exponents, on
  // the MFMA) instead of the per-head bound_c 2^-23 ||q_h|| max ||k||: under half as wide on typical rows, so
  // under half the near ties and their exact recomputation, for three more MFMAs per 16-key tile (D = 64).  Built
  // where the registers allow it (16 heads).
  constexpr bool PDD = HT == 1;
  constexpr int kSteps = KD / 8;  // accumulation steps of a dot
  __shared__ std::conditional_t<BOUND, ScoresLdsBound<KD, FEW>, ScoresLds<KD, HT>> L;
  if constexpr (FEW) {
    bounded_scores_few<WBF, F8>(L, q, k, w, qn, kn, scores, S, T, kbs, kns_stride, causal, start_pos, ratio, bound_c,
                                bounds, row_state, ksc);
    return;
  } else {
  // the wave index is uniform per wave; readfirstlane lets the compiler keep the query row, the causal limit
  // and the tile loop in scalar registers
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  // XCD-aware placement: workgroup i of a batch slice runs on XCD i % 8 (the slice holds a multiple of 8
  // workgroups when xcd_pk > 0).  XCD j takes a (gridDim.y / Pq) x (gridDim.x / Pk) tile of (query
  // group, key block) pairs with Pk = xcd_pk, Pq = 8 / Pk, so its L2 holds Pk-th of the queries' rows and
  // Pq-th of the keys instead of every query group.
  int kblk = blockIdx.x, qgrp = blockIdx.y;
  if (xcd_pk > 0) {
    const int wg = blockIdx.y * gridDim.x + blockIdx.x, xcd = wg & 7, l = wg >> 3;
    const int gxk = gridDim.x / xcd_pk, gyq = gridDim.y / (8 / xcd_pk);
    qgrp = (xcd / xcd_pk) * gyq + l / gxk;
    kblk = (xcd % xcd_pk) * gxk + l % gxk;
  }
  const int64_t b = blockIdx.z;
  const int kb0 = kblk * kKR;
  const int nk = min(kKR, T - kb0);
  const int64_t s = static_cast<int64_t>(qgrp) * kQW + wave;
  const bool s_ok = s < S;
  const int64_t kbrow0 = b * kbs;        // first key row of batch b
  const int64_t krow0 = kbrow0 + kb0;    // first key row of this workgroup
  // A workgroup whose queries all see none of its keys (causal limits at or below the block; the last query
  // has the largest limit) only writes the mask: no staging, no statistics (uniform over the workgroup, so
  // every wave leaves before the barrier).  Its key block's norm maximum is then read by no query.
  if (causal) {
    const int64_t s_last = static_cast<int64_t>(qgrp) * kQW + kQW - 1 < S - 1 ? static_cast<int64_t>(qgrp) * kQW + kQW - 1
                                                                             : S - 1;
    if ((start_pos + s_last + 1) / ratio <= kb0) {
      if (s_ok) {
        float *orow_m = scores + (b * S + s) * T;
        for (int i = lane; i < nk; i += 64) orow_m[kb0 + i] = -INFINITY;
      }
      return;
    }
  }
  if constexpr (BOUND) {  // a body of its own; the rest is the exact kernel
    bounded_scores<WBF, F8>(L, q, k, w, qn, kn, scores, S, T, kbs, kns_stride, causal, start_pos, ratio, bound_c, bounds,
                            row_state, ksc, kblk, qgrp);
    return;
  } else {

  // Every prologue load is issued before the first wait (loads complete in order, so each later wait is a
  // partial one): the key statistics and this wave's query statistics and head weights, then the key
  // block, then the q fragments.  Indices are clamped into range and the values masked afterwards, so no
  // load sits behind a branch or a loop-carried wait.
  // Statistics slots are written unconditionally: threads t and t + kKR (and lanes l and l + H) load and
  // write the same entry, so no store (and no load the compiler could sink next to it) is behind a branch.
  static_assert(kKR <= kThreads && (kKR & (kKR - 1)) == 0, "key statistics: a power-of-two block");
  const int64_t qrow0 = (b * S + (s_ok ? s : 0)) * H;
  const int kt = tid & (kKR - 1);
  const bool kin = kt < nk;
  const int kst = kin ? kt : nk - 1;  // nk >= 1: the grid covers T with key blocks
  // (loads at 32-bit unsigned offsets from workgroup-uniform bases: one address instruction each)
  const float *__restrict__ knb = kn + krow0;
  const float kn_v = knb[static_cast<uint32_t>(kst)];
  const int32_t ks_v = (ksp + krow0)[static_cast<uint32_t>(kst)];
  // every wave reads the whole block's key norms (keys lane + 64 j), so that it forms the block's norm maximum,
  // and with it the interval half-widths, without waiting for the other waves
  float kn4[kKR / 64];
#pragma unroll
  for (int j = 0; j < kKR / 64; ++j) {
    const int kj = lane + 64 * j;
    kn4[j] = knb[static_cast<uint32_t>(kj < nk ? kj : nk - 1)];
  }
  const int hl = lane & (H - 1);
  const uint32_t hlu = static_cast<uint32_t>(hl);
  const float qn_v = (qn + qrow0)[hlu];
  const int32_t qs_v = (qsp + qrow0)[hlu];
  const float w_v = WBF ? bf16_to_f32((static_cast<const uint16_t *>(w) + qrow0)[hlu])
                        : (static_cast<const float *>(w) + qrow0)[hlu];
  constexpr int kKL = kKR * kC / kThreads;  // 16-byte key chunks per thread
  uint4 kv[kKL];
#pragma unroll
  for (int it = 0; it < kKL; ++it) {
    const int lin = it * kThreads + tid;
    const int kr = lin / kC, ch = lin % kC;
    kv[it] = *reinterpret_cast<const uint4 *>(k + krow0 * KD + static_cast<uint32_t>((kr < nk ? kr : nk - 1) * KD + ch * 8));
  }
  // Every wave's key-block loads are queued ahead of every q load: the memory pipeline serves a CU's loads in
  // issue order, and the waves that issued last would otherwise wait behind the others' q rows (8 x 16 KiB)
  // for their share of the key block, which the barrier below waits for.  (The scheduling barriers keep every
  // load on its side of the barrier.)
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // query rows as MFMA A-fragments (rows of query 0 for a wave past S, which leaves after the barrier); the
  // barrier below waits for the key block only, so these arrive under it and the first tile's MFMAs
  // (issued in the order the first tile's MFMAs use them, k-step by k-step, so that they can start on the first
  // k-step's fragments while the rest arrive)
  uint4 qa[HT][KD / 32];
#pragma unroll
  for (int kk = 0; kk < KD / 32; ++kk)
#pragma unroll
    for (int m = 0; m < HT; ++m)
    {
      // (the exact kernel may read its q rows from two buffers, QSplit: the rotated dims from qsplit_rot)
      const uint16_t *qsrc =
          (qsplit_rot != nullptr && 32 * kk >= qsplit_lo && 32 * kk < qsplit_hi) ? qsplit_rot : q;
      qa[m][kk] = *reinterpret_cast<const uint4 *>(qsrc + qrow0 * KD + static_cast<uint32_t>((16 * m + l16) * KD + 32 * kk + 8 * g));
    }
  auto abs8 = [](uint4 v) {  // |x| of 8 packed bf16
    return make_uint4(v.x & 0x7FFF7FFFu, v.y & 0x7FFF7FFFu, v.z & 0x7FFF7FFFu, v.w & 0x7FFF7FFFu);
  };
  // max key norm over this workgroup's range (the error bound uses it for every key)
  L.knorm[kt] = kin ? kn_v : 0.f;
  L.kspan[kt] = kin ? ks_v : 0;
  float knm = 0.f;
#pragma unroll
  for (int j = 0; j < kKR / 64; ++j) knm = fmaxf(knm, lane + 64 * j < nk ? kn4[j] : 0.f);
  knm = wave_max_f32(knm);
  L.qspan[wave][hl] = qs_v;
  L.qnorm[wave][hl] = qn_v;
  // per-head data formed once per head (lane h), not by each of the 16 lanes that use it.  PDD (the exact kernel
  // at 16 heads): per-dot half-widths from the MFMA sum of the magnitudes, dl then holds their additive part
  L.dl[wave][hl] = PDD ? step_halfwidth_add(qn_v, knm, bound_r) : dot_halfwidth(qn_v, knm, bound_c);
  L.w[wave][hl] = w_v;
  // the workgroup's whole key block into LDS
  {
    // Rows past T hold copies of the last key, loaded from the clamped row: finite operands whose columns are
    // neither stored nor listed.  The 32- and 64-head kernels still zero them: with the loaded values used only by
    // the LDS stores, the compiler sinks their loads below the q loads (and the load-ordering barrier above),
    // which the mask's use of them prevents (a CPU test checks the placement in the compiled code).
    constexpr bool kMask = HT > 1;
#pragma unroll
    for (int it = 0; it < kKL; ++it) {
      const int lin = it * kThreads + tid;
      const int kr = lin / kC, ch = lin % kC;
      const uint32_t msk = (!kMask || kr < nk) ? 0xFFFFFFFFu : 0u;
      L.k[kr * kC + (ch ^ (kr & (kC - 1)))] = make_uint4(kv[it].x & msk, kv[it].y & msk, kv[it].z & msk, kv[it].w & msk);
      if constexpr (PDD) L.kstep[kr][ch] = static_cast<uint16_t>(step_exponent_pow2(kv[it]));
    }
  }
  // the only barrier (from here on every wave runs independently): LDS writes done, no wait for the q loads
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (!s_ok) return;
  float wv[HT][4], dl[HT][4];
#pragma unroll
  for (int m = 0; m < HT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int h = 16 * m + 4 * g + r;
      wv[m][r] = L.w[wave][h];
      dl[m][r] = L.dl[wave][h];
    }
  // a half-width of +inf (norms that could overflow inside the MFMA): every dot of the wave is a near tie
  bool any_inf = false;
#pragma unroll
  for (int m = 0; m < HT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) any_inf = any_inf || dl[m][r] == __builtin_inff();
  const bool forced = __builtin_amdgcn_ballot_w64(any_inf) != 0ull;
  const int64_t limit = causal ? (start_pos + s + 1) / ratio : INT64_MAX;
  const int limit32 = static_cast<int>(limit < INT32_MAX ? limit : INT32_MAX);  // keys are below T < 2^31
  float *orow = scores + (b * S + s) * T;
  uint32_t n_exact = 0, n_unres = 0;
  int nent = 0;
  // tiles of 16 keys; tiles at or past the causal limit are masked without MFMA work
  const int ntiles = (nk + 15) / 16;
  const int64_t lim_rel = limit - kb0;
  const int nlive = lim_rel <= 0 ? 0 : (lim_rel >= 16 * ntiles ? ntiles : static_cast<int>((lim_rel + 15) / 16));

  // PDD: accs holds V >= W + 8 M of the per-dot half-width (step_halfwidth_scale): the step-weighted magnitudes of
  // q (qw, formed once: fragment kk of this lane is step 4 kk + g, weight 2^j >= kSteps + 1 - step) against |k|,
  // then one MFMA of the step exponents: aprime holds 8 A'_s of this lane's head in k-slots 8 g .. 8 g + 7 (steps
  // 8 g ..; zeros past the last step), gathered through the wave's dot-list LDS (unused until the first flush);
  // the keys' B'_s are staged with the key block.
  uint4 qw[HT][KD / 32];
  uint4 aprime = make_uint4(0, 0, 0, 0);
  if constexpr (PDD) {
    uint16_t *sq = reinterpret_cast<uint16_t *>(L.dots[wave]);  // [16 heads][kSteps]: 8 A'_s
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk) {
      const int st = 4 * kk + g;
      qw[0][kk] = step_weighted_q(qa[0][kk], step_weight_log2(kSteps, st));
      const uint32_t p = step_exponent_pow2(qa[0][kk]);
      sq[l16 * kSteps + st] = static_cast<uint16_t>(p == 0u ? 0u : p + (3u << 7));  // 8 A'_s: exponent + 3
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint4 t = reinterpret_cast<const uint4 *>(sq)[(l16 * kSteps + 8 * (g % (kSteps / 8))) / 8];
    aprime = g < kSteps / 8 ? t : make_uint4(0, 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // the MFMAs of 16 keys, lane l16 holding block row key_l (a tile: 16 t + l16; or rows from the deferred list)
  // (every LDS read first; PDD: the magnitude chain starts with the step exponents, so that its dependent MFMAs
  // alternate with the independent ones of the dot)
  auto tile_mfma = [&](int key_l, f32x4_t(&acc)[HT], f32x4_t(&accs)[HT]) {
    uint4 bv[KD / 32];
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk) bv[kk] = L.k[key_l * kC + ((4 * kk + g) ^ (key_l & (kC - 1)))];
#pragma unroll
    for (int m = 0; m < HT; ++m) acc[m] = accs[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (PDD) {
      // the step exponents: lane (key row, g) reads the key's B'_s of steps 8 g .. (lanes past the last step read
      // the first ones: their A' slots are zero, so those products leave the sum unchanged)
      const uint4 bp = *reinterpret_cast<const uint4 *>(&L.kstep[key_l][8 * (g % (kSteps / 8))]);
      accs[0] = mfma16(aprime, bp, accs[0]);
    }
#pragma unroll
    for (int kk = 0; kk < KD / 32; ++kk) {
#pragma unroll
      for (int m = 0; m < HT; ++m) acc[m] = mfma16(qa[m][kk], bv[kk], acc[m]);
      if constexpr (PDD) {
        const uint4 ba = abs8(bv[kk]);
#pragma unroll
        for (int m = 0; m < HT; ++m) accs[m] = mfma16(qw[m][kk], ba, accs[m]);
      }
    }
  };

  const float dsc = PDD ? step_halfwidth_scale(bound_r) : 0.f;
  // the exact kernel's interval test (the tile epilogue's, below) on the 16 keys of a resolution round: pl, ph and the
  // ballot of the lanes holding a near-tie dot.
  auto interval_ends = [&](const f32x4_t(&acc)[HT], const f32x4_t(&accs)[HT], uint32_t(&pl)[2 * HT],
                           uint32_t(&ph)[2 * HT]) {
    uint64_t anyr = 0;
#pragma unroll
    for (int m = 0; m < HT; ++m)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        const float A0 = acc[m][2 * rp], A1 = acc[m][2 * rp + 1];
        const float d0 = PDD ? __builtin_fmaf(accs[m][2 * rp], dsc, dl[m][2 * rp]) : dl[m][2 * rp];
        const float d1 = PDD ? __builtin_fmaf(accs[m][2 * rp + 1], dsc, dl[m][2 * rp + 1]) : dl[m][2 * rp + 1];
        pl[2 * m + rp] = cvt_relu_pk(A0 - d0, A1 - d1);
        ph[2 * m + rp] = cvt_relu_pk(A0 + d0, A1 + d1);
        anyr |= __builtin_amdgcn_ballot_w64(pl[2 * m + rp] != ph[2 * m + rp]);
      }
    if (forced) {
#pragma unroll
      for (int p = 0; p < 2 * HT; ++p) {
        pl[p] = 0u;
        ph[p] = 0x7F807F80u;
      }
      anyr = ~0ull;
    }
    return anyr;
  };
  // the key mask (bit = key column) of a ballot over the four head-group rows
  auto key_mask = [](uint64_t r) { return static_cast<uint32_t>((r | (r >> 16) | (r >> 32) | (r >> 48)) & 0xFFFFull); };
  // returns the mask of this tile's keys (bit = key column) that hold a near-tie dot (in the exact kernel, before
  // the causal limit: a key past it keeps the -inf stored here); pl / ph keep the interval ends.
  // FULL (the exact kernel's tiles before its last live one): every key of the tile is in range and before the
  // causal limit, so the tile needs no per-lane key tests.  PAIR (the exact kernel): the lane's group sum is
  // returned in gsum, and store_pair combines two tiles' sums at once; otherwise the tile stores its own scores.
  auto tile_epilogue = [&](auto FC, auto FULL, auto PAIR, int t, const f32x4_t(&acc)[HT], const f32x4_t(&accs)[HT],
                           uint32_t(&pl)[2 * HT], uint32_t(&ph)[2 * HT], float &gsum) {
    const bool fcd = decltype(FC)::value;
    constexpr bool full = decltype(FULL)::value;
    const int key_l = 16 * t + l16;
    const int key = kb0 + key_l;
    const bool kvalid = full || key_l < nk;
    // interval test: RNE(A - delta) == RNE(A + delta) (after ReLU) <=> the exact dot rounds to the same
    // relu'd bf16 value; pl holds that value for the head sum
    uint64_t anyr = 0;
#pragma unroll
    for (int m = 0; m < HT; ++m)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        const float A0 = acc[m][2 * rp], A1 = acc[m][2 * rp + 1];
        const float d0 = PDD ? __builtin_fmaf(accs[m][2 * rp], dsc, dl[m][2 * rp]) : dl[m][2 * rp];
        const float d1 = PDD ? __builtin_fmaf(accs[m][2 * rp + 1], dsc, dl[m][2 * rp + 1]) : dl[m][2 * rp + 1];
        pl[2 * m + rp] = cvt_relu_pk(A0 - d0, A1 - d1);
        ph[2 * m + rp] = cvt_relu_pk(A0 + d0, A1 + d1);
        anyr |= __builtin_amdgcn_ballot_w64(pl[2 * m + rp] != ph[2 * m + rp]);
      }
    if (fcd) {  // wave-uniform and rare: A may not even be finite; the exact values replace everything
#pragma unroll
      for (int p = 0; p < 2 * HT; ++p) {
        pl[p] = 0u;
        ph[p] = 0x7F807F80u;
      }
      anyr = ~0ull;
    }
    // canonical head sum of this lane's group, then ((G0+G1)+(G2+G3)) across the rows
    float G = 0.f;
    if constexpr (WBF) {
      G = group_sum<HT, WBF>([&](int i) { return pl[i]; }, wv);
    } else {
#pragma unroll
      for (int m = 0; m < HT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t p2 = pl[2 * m + (r >> 1)];
          const float rv = (r & 1) ? unpack_hi(p2) : unpack_lo(p2);
          G = __builtin_fmaf(rv, wv[m][r], G);
        }
    }
    float tot = 0.f, outv = 0.f;
    if constexpr (decltype(PAIR)::value) {
      gsum = G;
    } else {
      tot = combine_groups(G);
      outv = WBF ? round_score_bf16(tot) : tot;
      if (g == 0 && kvalid) orow[key] = (full || key < limit32) ? outv : -INFINITY;
    }
    // keys past T are not stored and keys past the causal limit are -inf: neither is deferred
    if constexpr (!full) anyr &= __builtin_amdgcn_ballot_w64(kvalid && key < limit32);
    return key_mask(anyr);
  };
  // software pipeline: the MFMAs of the next tile are in flight during the current tile's epilogue.
  f32x4_t acc[HT], nxt[HT];
  {
    // the tile loop only lists the keys holding a near-tie dot (their block rows, in LDS); the
    // listed keys are resolved after it.  Nothing of the recomputation is live in the loop, so the loop keeps its
    // pipeline in few registers.  The next tile's MFMAs past the last live tile repeat that tile (results unused).
    // Two tiles per iteration alternate the accumulator sets (no copies between them); the loop is built twice,
    // for forced waves (every key listed) and the others, so that the tile epilogue carries no select for it.
    f32x4_t accs[HT], nxts[HT];
    uint8_t *klist = L.klist[wave];
    int nlist = 0;
    // Tiles before the last live one are full (every key in range and before the limit).
    auto epilogue = [&](auto FC, auto FULL, auto PAIR, int t, const f32x4_t(&a)[HT], const f32x4_t(&as)[HT]) {
      uint32_t pl[2 * HT], ph[2 * HT];
      float gs = 0.f;
      const uint32_t km = tile_epilogue(FC, FULL, PAIR, t, a, as, pl, ph, gs);
      if (km != 0u) {  // wave-uniform
        if (g == 0 && ((km >> l16) & 1u))
          klist[nlist + __builtin_popcount(km & ((1u << l16) - 1u))] = static_cast<uint8_t>(16 * t + l16);
        nlist += __builtin_popcount(km);
      }
      return gs;
    };
    // The scores of tiles t and t + 1 from their lanes' group sums ga, gb: ((G0 + G1) + (G2 + G3)) of both tiles
    // with one exchange of each kind (combine_groups with two different registers in place of one copied twice):
    // after the row-pair swap, rows 0 / 2 hold tile t's pair sums and rows 1 / 3 tile t + 1's; after the half swap
    // row 0 holds tile t's score and row 1 tile t + 1's.  PB: tile t + 1 is the last live tile (key tests).
    auto store_pair = [&](auto PB, int t, float ga, float gb) {
      float a = ga, b = gb;
      asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
      float c = a + b, d = c;
      asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(c), "+v"(d));
      const float tot = c + d;
      const float outv = WBF ? round_score_bf16(tot) : tot;
      const int key_l = 16 * (t + (g & 1)) + l16;
      if constexpr (decltype(PB)::value) {
        if (g == 0 || (g == 1 && key_l < nk)) orow[kb0 + key_l] = (g == 0 || kb0 + key_l < limit32) ? outv : -INFINITY;
      } else {
        if (g < 2) orow[static_cast<uint32_t>(kb0 + key_l)] = outv;
      }
    };
    const int last = nlive - 1;
    if (nlive > 0 && !forced) {
      const std::true_type full, pair;
      const std::false_type fc, partial, single;
      tile_mfma(l16, acc, accs);
      int t = 0;
      for (; t + 2 <= last; t += 2) {
        tile_mfma(16 * (t + 1) + l16, nxt, nxts);
        const float ga = epilogue(fc, full, pair, t, acc, accs);
        tile_mfma(16 * (t + 2) + l16, acc, accs);
        const float gb = epilogue(fc, full, pair, t + 1, nxt, nxts);
        store_pair(std::false_type{}, t, ga, gb);
      }
      if (t < last) {
        tile_mfma(16 * last + l16, nxt, nxts);
        const float ga = epilogue(fc, full, pair, t, acc, accs);
        const float gb = epilogue(fc, partial, pair, last, nxt, nxts);
        store_pair(std::true_type{}, t, ga, gb);
      } else {
        (void)epilogue(fc, partial, single, last, acc, accs);
      }
    } else if (nlive > 0) {
      // a forced wave lists every key (its interval ends are not used)
      for (int t = 0; t < nlive; ++t) (void)epilogue(std::true_type{}, std::false_type{}, std::false_type{}, t, acc, accs);
    }
    // resolution, 16 listed keys at a time: the same MFMAs and interval test on their rows (the same operands, so
    // the same interval ends)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if constexpr (HT == 1) {
      // 16 heads: each round keeps its 16 keys' interval ends in registers (lane (g, l16): heads 4 g .. 4 g + 3 of
      // key l16), lists the round's near-tie dots (lane and head bit, 16 bits each; at most 256) in the wave's dot list,
      // computes them exactly 16 at a time, patches the exact relu'd values (through the list's patch slots, one
      // per lane and head bit) into its own ends and stores the round's scores.
      const QSplit qsp{qsplit_rot, qsplit_lo, qsplit_hi};
      // a round holds at most 16 keys x 16 heads = 256 near-tie dots: [0, 256) the list, [256, 512) the patches
      static_assert(2 * 256 * sizeof(uint16_t) <= sizeof(L.dots[0]), "dot list and patches of one round");
      uint16_t *Dl = reinterpret_cast<uint16_t *>(L.dots[wave]);
      uint16_t *Pt = Dl + 256;
      const int dq = lane >> 2, sub = lane & 3;
      for (int base = 0; base < nlist; base += 16) {
        const int key_l = klist[min(base + l16, nlist - 1)];
        tile_mfma(key_l, acc, accs);
        uint32_t pl[2], ph[2];
        (void)interval_ends(acc, accs, pl, ph);
        // this lane's near-tie dots: bit b = head 4 g + b (half b & 1 of pl[b >> 1]); lanes past the list none
        uint32_t m = 0;
        if (base + l16 < nlist) {
          const uint32_t d0 = pl[0] ^ ph[0], d1 = pl[1] ^ ph[1];
          m = ((d0 & 0xFFFFu) ? 1u : 0u) | ((d0 >> 16) ? 2u : 0u) | ((d1 & 0xFFFFu) ? 4u : 0u) | ((d1 >> 16) ? 8u : 0u);
        }
        uint32_t nd_u;
        uint32_t pos = wave_excl_scan_bits<3>(static_cast<uint32_t>(__builtin_popcount(m)), nd_u);
        for (uint32_t mm = m; mm != 0u; mm &= mm - 1u) Dl[pos++] = static_cast<uint16_t>((lane << 2) | __builtin_ctz(mm));
        n_exact += nd_u;
        const int nd = static_cast<int>(nd_u);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int b0 = 0; b0 < nd; b0 += 16) {
          // the quad's dot (idle quads repeat the last one; the result is identical): lane sl's head bit
          const int dcur = Dl[min(b0 + dq, nd - 1)];
          const int sl = dcur >> 2;
          const int h = 4 * (sl >> 4) + (dcur & 3);
          const int kl = klist[base + (sl & 15)];
          int scur;
          const uint16_t r = quad_exact_dot<HT, KD>(L, wave, sub, h, kl, q, qsp, qa, qrow0, scur);
          if (sub == 0 && b0 + dq < nd) {
            Pt[dcur] = (r & 0x8000) ? 0u : r;  // ReLU (also maps -0 to +0)
            if (scur > 84) ++n_unres;  // counted: dots that needed the integer accumulator
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (m != 0u) {
#pragma unroll
          for (int bit = 0; bit < 4; ++bit)
            if ((m >> bit) & 1u) {
              const uint32_t v = Pt[(lane << 2) | bit];
              uint32_t &w2 = pl[bit >> 1];
              w2 = (bit & 1) ? ((w2 & 0xFFFFu) | (v << 16)) : ((w2 & 0xFFFF0000u) | v);
            }
        }
        // the round's scores from the patched values (every listed key is in range and before the causal limit)
        const float G = group_sum<HT, WBF>([&](int i) { return pl[i]; }, wv);
        const float tot = combine_groups(G);
        if (g == 0 && base + l16 < nlist) orow[static_cast<uint32_t>(kb0 + key_l)] = WBF ? round_score_bf16(tot) : tot;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    } else {
      // all four groups' ends of each key saved as a deferred entry, and the entries' near-tie dots computed
      // exactly and their scores rewritten whenever another 16 could overflow the entries
      for (int base = 0; base < nlist; base += 16) {
        const int key_l = klist[min(base + l16, nlist - 1)];
        tile_mfma(key_l, acc, accs);
        uint32_t pl[2 * HT], ph[2 * HT];
        // every listed key is in range and before the causal limit; lanes past the list repeat its last key
        const uint32_t km = key_mask(interval_ends(acc, accs, pl, ph) &
                                     __builtin_amdgcn_ballot_w64(base + l16 < nlist));
        if ((km >> l16) & 1u) {
          const int e = nent + __builtin_popcount(km & ((1u << l16) - 1u));
          KeyEntry<HT> &en = L.ent[wave][e];
#pragma unroll
          for (int p = 0; p < 2 * HT; ++p) {
            en.pl[g][p] = pl[p];
            en.ph[g][p] = ph[p];
          }
          if (g == 0) en.key = kb0 + key_l;
        }
        nent += __builtin_popcount(km);
        if (nent + 16 > kEntCap || base + 16 >= nlist) {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          if (nent > 0)
            flush_entries<HT, KD, WBF>(L, wave, lane, nent, q, qa, qrow0, orow, limit, T, kb0, wv, n_exact, n_unres,
                                       QSplit{qsplit_rot, qsplit_lo, qsplit_hi});
          nent = 0;
        }
      }
    }
  }
  // masked tiles (at or past the causal limit)
  for (int key_l = 16 * nlive + lane; key_l < nk; key_l += 64) orow[static_cast<uint32_t>(kb0 + key_l)] = -INFINITY;
  if (stats != nullptr) {
    if (lane == 0 && n_exact) atomicAdd(&stats[0], n_exact);
    if (n_unres) atomicAdd(&stats[1], n_unres);
  }
  }  // !BOUND
  }  // !FEW
}

template <int HT, int KD>
int launch_scores_ht(const uint16_t *q, const uint16_t *k, const void *w, int w_bf16, const float *qn,
                     const int32_t *qsp, const float *kn, const int32_t *ksp, float *scores, int64_t B, int64_t S,
                     int64_t T, int64_t kbs, int64_t kns, int causal, int64_t start_pos, int ratio, float bound_c, uint32_t *stats,
                     float *bounds, uint32_t *row_state, const float *ksc, hipStream_t stream,
                     const QSplit *qsplit) {
  const QSplit qs = qsplit != nullptr ? *qsplit : QSplit{nullptr, 0, 0};
  dim3 grid(static_cast<unsigned>(ceil_div(T, kKR)), static_cast<unsigned>(ceil_div(S, kQW)),
            static_cast<unsigned>(B));
  const float bound_r = bound_c / score_bound_c(KD);  // the per-dot half-widths' scale (16-head exact kernel)
  // XCD tiling (Pq x Pk = 8) that minimises the L2 fills: each query group's rows are read by Pk XCDs,
  // each key block by Pq; 0 keeps the launch order (slice not a multiple of 8 or no tiling divides it)
  int xcd_pk = 0;
  if ((static_cast<int64_t>(grid.x) * grid.y) % 8 == 0) {
    const double qbytes = static_cast<double>(S) * 16 * HT * KD, kbytes = static_cast<double>(T) * KD;  // either format
    double best = 0.0;
    for (int pk = 1; pk <= 8; pk *= 2) {
      const int pq = 8 / pk;
      if (grid.x % pk != 0 || grid.y % pq != 0) continue;
      const double cost = qbytes * pk + kbytes * pq;
      if (xcd_pk == 0 || cost < best) {
        best = cost;
        xcd_pk = pk;
      }
    }
  }
  if (bounds != nullptr || ksc != nullptr) {
    if constexpr (HT == 4 && KD == 128) {
      if (bounds == nullptr) return fail(KS_ERR_INVALID, "indexer scores: FP8 keys need the bound-emitting kernel");
      if (row_state == nullptr) return fail(KS_ERR_INVALID, "indexer scores: score bounds need the row states");
      // up to kFewQueries queries a batch: a workgroup per query, its waves over the keys (at most ~4 rounds of
      // workgroups, each wave then taking several groups)
      const bool few = S <= kFewQueries;
      if (few) {
        const int64_t per_row = ceil_div(T, 64 * kQW), rows = B * S;
        const int64_t most = ceil_div(kFewTargetWgs, rows);
        grid = dim3(static_cast<unsigned>(per_row < most ? per_row : most), static_cast<unsigned>(S),
                    static_cast<unsigned>(B));
      }
      auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, stream, q, k, w, qn, qsp, kn, ksp, scores, S,
                           static_cast<int>(T), kbs, kns, causal, start_pos, ratio, bound_c, stats, xcd_pk, bounds, row_state,
                           ksc, bound_r, qs.rot, qs.lo, qs.hi);
      };
      auto pick = [&](auto WBF) {
        constexpr bool wbf = decltype(WBF)::value;
        if (ksc != nullptr && few) run(indexer_scores_kernel<HT, KD, wbf, true, true, true>);
        else if (ksc != nullptr) run(indexer_scores_kernel<HT, KD, wbf, true, false, true>);
        else if (few) run(indexer_scores_kernel<HT, KD, wbf, true, true, false>);
        else run(indexer_scores_kernel<HT, KD, wbf, true, false, false>);
      };
      if (w_bf16) pick(std::true_type{});
      else pick(std::false_type{});
    } else {
      return fail(KS_ERR_INVALID, "indexer scores: score bounds need H = 64 and D = 128");
    }
  } else if (w_bf16) {
    hipLaunchKernelGGL((indexer_scores_kernel<HT, KD, true, false>), grid, dim3(kThreads), 0, stream, q, k, w, qn, qsp,
                       kn, ksp, scores, S, static_cast<int>(T), kbs, kns, causal, start_pos, ratio, bound_c, stats, xcd_pk,
                       nullptr, nullptr, nullptr, bound_r, qs.rot, qs.lo, qs.hi);
  } else {
    hipLaunchKernelGGL((indexer_scores_kernel<HT, KD, false, false>), grid, dim3(kThreads), 0, stream, q, k, w, qn,
                       qsp, kn, ksp, scores, S, static_cast<int>(T), kbs, kns, causal, start_pos, ratio, bound_c, stats,
                       xcd_pk, nullptr, nullptr, nullptr, bound_r, qs.rot, qs.lo, qs.hi);
  }
  KS_CHECK_LAUNCH("indexer_scores_kernel");
  return KS_OK;
}

template <int KD>
int launch_scores_d(const uint16_t *q, const uint16_t *k, const void *w, int w_bf16, const float *qn,
                    const int32_t *qsp, const float *kn, const int32_t *ksp, float *scores, int64_t B, int64_t S,
                    int64_t H, int64_t T, int64_t kbs, int64_t kns, int causal, int64_t start_pos, int ratio, float bound_c,
                    uint32_t *stats, float *bounds, uint32_t *row_state, const float *ksc,
                    hipStream_t stream, const QSplit *qsplit) {
  switch (H) {
    case 16:
      return launch_scores_ht<1, KD>(q, k, w, w_bf16, qn, qsp, kn, ksp, scores, B, S, T, kbs, kns, causal, start_pos,
                                     ratio, bound_c, stats, bounds, row_state, ksc, stream, qsplit);
    case 32:
      return launch_scores_ht<2, KD>(q, k, w, w_bf16, qn, qsp, kn, ksp, scores, B, S, T, kbs, kns, causal, start_pos,
                                     ratio, bound_c, stats, bounds, row_state, ksc, stream, qsplit);
    case 64:
      return launch_scores_ht<4, KD>(q, k, w, w_bf16, qn, qsp, kn, ksp, scores, B, S, T, kbs, kns, causal, start_pos,
                                     ratio, bound_c, stats, bounds, row_state, ksc, stream, qsplit);
    default:
      return fail(KS_ERR_INVALID, "indexer scores: H=%lld, supported: 16, 32, 64", (long long)H);
  }
}

}  // namespace

int launch_indexer_scores(const uint16_t *q, const uint16_t *k, const void *w, int w_bf16, const float *qn,
                          const int32_t *qsp, const float *kn, const int32_t *ksp, float *scores, int64_t B,
                          int64_t S, int64_t H, int64_t D, int64_t T, int64_t kbs, int causal, int64_t start_pos,
                          int ratio, float bound_c, uint32_t *stats, hipStream_t stream, float *bounds,
                          uint32_t *row_state, const float *ksc,
                          const QSplit *qsplit, int64_t kns) {
  if (kns == 0) kns = kbs;
  if (D == 128)
    return launch_scores_d<128>(q, k, w, w_bf16, qn, qsp, kn, ksp, scores, B, S, H, T, kbs, kns, causal, start_pos, ratio,
                                bound_c, stats, bounds, row_state, ksc, stream, qsplit);
  if (D == 64)
    return launch_scores_d<64>(q, k, w, w_bf16, qn, qsp, kn, ksp, scores, B, S, H, T, kbs, kns, causal, start_pos, ratio,
                               bound_c, stats, bounds, row_state, ksc, stream, qsplit);
  return fail(KS_ERR_INVALID, "indexer scores: D=%lld, supported: 64, 128", (long long)D);
}

}  // namespace ks

namespace {
int check_scores_args(const uint16_t *q, const uint16_t *k, const void *w, const float *qn, const int32_t *qsp,
                      const float *kn, const int32_t *ksp, float *scores, int64_t B, int64_t S, int64_t H, int64_t D,
                      int64_t T, int64_t kbs, int32_t ratio, int64_t start_pos) {
  KS_CHECK_ARG(D == 128 || D == 64, "ks_indexer_scores: D=%lld, the kernel is built for head_dim 64 and 128",
               (long long)D);
  KS_CHECK_ARG(H == 16 || H == 32 || H == 64, "ks_indexer_scores: H=%lld must be 16, 32 or 64", (long long)H);
  KS_CHECK_ARG(B >= 0 && S >= 0, "ks_indexer_scores: negative B or S");
  KS_CHECK_ARG(B < 65536 && S < (int64_t(1) << 24), "ks_indexer_scores: B or S too large");
  KS_CHECK_ARG(T >= 1 && T < (int64_t(1) << 31), "ks_indexer_scores: T=%lld out of range", (long long)T);
  KS_CHECK_ARG(kbs >= T, "ks_indexer_scores: k_batch_stride=%lld < T=%lld", (long long)kbs, (long long)T);
  KS_CHECK_ARG(ratio >= 1 && start_pos >= 0, "ks_indexer_scores: ratio must be >= 1 and start_pos >= 0");
  KS_CHECK_ARG(q && k && w && qn && qsp && kn && ksp && scores, "ks_indexer_scores: null pointer");
  KS_CHECK_ARG(ks::aligned(q, 16) && ks::aligned(k, 16) && ks::aligned(scores, 4),
               "ks_indexer_scores: q and k must be 16-byte aligned");
  return KS_OK;
}
}  // namespace

extern "C" int ks_indexer_scores(const uint16_t *q, const uint16_t *k, const void *w, int32_t w_bf16,
                                 const float *q_norm, const int32_t *q_span, const float *k_norm,
                                 const int32_t *k_span, float *scores, int64_t B, int64_t S, int64_t H, int64_t D,
                                 int64_t T, int64_t k_batch_stride, int32_t causal, int64_t start_pos, int32_t ratio,
                                 void *stream) {
  ks::last_error().clear();
  int rc = check_scores_args(q, k, w, q_norm, q_span, k_norm, k_span, scores, B, S, H, D, T, k_batch_stride, ratio,
                             start_pos);
  if (rc != KS_OK) return rc;
  if (B * S == 0) return KS_OK;
  return ks::launch_indexer_scores(q, k, w, w_bf16 ? 1 : 0, q_norm, q_span, k_norm, k_span, scores, B, S, H, D,
                                   T, k_batch_stride, causal ? 1 : 0, start_pos, ratio, ks::score_bound_c(D), nullptr,
                                   static_cast<hipStream_t>(stream));
}

// Diagnostic (not part of the public header): the interval constant the public entry points use for 128-dim
// dots, and for D-dimensional ones.
extern "C" float ks_dbg_score_bound_c(void) { return ks::kScoreBoundC; }
extern "C" float ks_dbg_score_bound_c_d(int64_t D) { return ks::score_bound_c(D); }

// Diagnostic variant (not part of the public header): explicit error-bound constant and a device counter
// pair stats[0] += exact recomputations, stats[1] += dots outside the provably exact range.
extern "C" int ks_dbg_indexer_scores(const uint16_t *q, const uint16_t *k, const void *w, int32_t w_bf16,
                                     const float *q_norm, const int32_t *q_span, const float *k_norm,
                                     const int32_t *k_span, float *scores, int64_t B, int64_t S, int64_t H, int64_t D,
                                     int64_t T, int64_t k_batch_stride, int32_t causal, int64_t start_pos,
                                     int32_t ratio, float bound_c, uint32_t *stats, void *stream) {
  ks::last_error().clear();
  int rc = check_scores_args(q, k, w, q_norm, q_span, k_norm, k_span, scores, B, S, H, D, T, k_batch_stride, ratio,
                             start_pos);
  if (rc != KS_OK) return rc;
  if (B * S == 0) return KS_OK;
  return ks::launch_indexer_scores(q, k, w, w_bf16 ? 1 : 0, q_norm, q_span, k_norm, k_span, scores, B, S, H, D,
                                   T, k_batch_stride, causal ? 1 : 0, start_pos, ratio, bound_c, stats,
                                   static_cast<hipStream_t>(stream));
}

// Diagnostic variant of the bounded score kernel (not part of the public header), for timing it alone:
// as ks_dbg_indexer_scores with fp32 weights, 64 heads and D = 128, plus the per-score bounds [B, S, T] and the bounded
// selection's workspace part (ks_dbg_topk_bounded_slots(B S, T) 64-bit slots), whose row states receive the rows'
// histogram scales.  kmax is not used.
extern "C" int ks_dbg_indexer_scores_bounded(const uint16_t *q, const uint16_t *k, const float *w,
                                             const float *q_norm, const int32_t *q_span, const float *k_norm,
                                             const int32_t *k_span, float *scores, float *bounds, float *kmax,
                                             uint64_t *part, int64_t B, int64_t S, int64_t T, int32_t causal,
                                             int64_t start_pos, void *stream) {
  ks::last_error().clear();
  int rc = check_scores_args(q, k, w, q_norm, q_span, k_norm, k_span, scores, B, S, 64, 128, T, T, 1, start_pos);
  if (rc != KS_OK) return rc;
  KS_CHECK_ARG(bounds && part, "ks_dbg_indexer_scores_bounded: null pointer");
  KS_CHECK_ARG(T <= 32768, "ks_dbg_indexer_scores_bounded: T <= 32768");
  if (B * S == 0) return KS_OK;
  return ks::launch_indexer_scores(q, k, w, 0, q_norm, q_span, k_norm, k_span, scores, B, S, 64, 128, T, T,
                                   causal ? 1 : 0, start_pos, 1, ks::kScoreBoundC, nullptr,
                                   static_cast<hipStream_t>(stream), bounds,
                                   ks::topk_bounded_state(part, B * S, T));
}
