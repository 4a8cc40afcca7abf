// Joint top-k / top-p token sampling for gfx950: one workgroup per logits row (the algorithm
// below), or a row spread over several (further down).
//
// Semantics (src/engine/sampling.rs:239-269, 330-372, 409-428):
//   * parameters are normalised as SamplingParams::normalized does: a top_p
//     that is not finite or lies outside [0, 1] becomes 1; top_k <= 0 or
//     top_k > vocab means the whole vocabulary;
//   * temperature <= 0 or top_p == 0 -> argmax of the raw logits (first index
//     of the maximum, NaN counting as the maximum, as torch's argmax);
//   * otherwise s = cast(logit * (1 / temperature)) in the logits dtype (a
//     tensor divided by a scalar is computed as a multiply by the fp32
//     reciprocal on the GPU) and p = softmax(s) in fp32; both cutoffs are taken on that ORIGINAL p:
//       top-k keeps p >= (k-th largest p)       (ties at the boundary kept)
//       top-p keeps p >= v*, v* = the largest value whose "mass at or above"
//             reaches top_p; when rounding keeps every prefix below top_p the
//             smallest p is the cutoff (the reference's clamp to vocab-1);
//     a token survives when it passes both, and one token is drawn from the
//     surviving p renormalised;
//   * a row whose distribution is invalid (NaN anywhere, every logit -inf, or a scaled
//     logit of +inf, which makes the reference's softmax NaN) yields -1, the
//     reference's invalid-distribution sentinel
//     (sampling_bridge.cpp: output.masked_fill_(!valid, -1)).
//
// Algorithm:
//   pass 1  row max and sum of exp (online), NaN detection;
//   pass 2-4 radix selection over the fp32 bit pattern of p (non-negative, so
//     the bits order like the values), 12 + 10 + 9 bits. Each pass builds a
//     count histogram (top-k) and a mass histogram (top-p) in LDS and a
//     workgroup suffix scan picks the bin holding the cutoff. Mass is summed in
//     64-bit fixed point (2^-40 units) so the histogram, and hence the cutoff,
//     does not depend on the order of the LDS atomics: equal seeds give equal
//     tokens;
//   pass 5  exponential race: the surviving token with the largest s + G,
//     G = -log(-log(u)) a Gumbel variate, is an exact draw from the surviving
//     distribution (Gumbel-max). u comes from Philox4x32-10 (Salmon et al.,
//     SC'11) keyed by the seed, with counter (element/4, row, offset), so the
//     draw needs no prefix scan and no renormalising sum.
// Without either cutoff only the race pass runs; greedy rows run one argmax pass.
#include <cfloat>

#include "common.h"

namespace mi355x {
namespace {

constexpr int kThreads = 1024;
constexpr int kWarps = kThreads / kWave;
constexpr int kBins0 = 4096;  // bits 30..19 of p (bit 31, the sign, is always 0)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kFixedScale = 1099511627776.0f;  // 2^40
constexpr uint32_t kCandidates = 2048;  // candidate path: (index, s, p) lists in LDS

// Logits element access for dtype codes 0 (bf16), 1 (fp16), 2 (fp32).
template <int DT>
struct Logit {
  using Word = uint16_t;
  static constexpr int kVec = 8;
  __device__ __forceinline__ static float to_float(Word w) { return Elem<DT>::to_float(w); }
  __device__ __forceinline__ static float round(float f) {
    return Elem<DT>::to_float(Elem<DT>::from_float(f));
  }
};
template <>
struct Logit<2> {
  using Word = float;
  static constexpr int kVec = 4;
  __device__ __forceinline__ static float to_float(Word w) { return w; }
  // The scaled logit must be the rounded product: without the barrier the compiler may fuse
  // x * (1 / T) into a later s - max as one fma, which differs from the rounded s by up to half
  // an ulp, and can differ between the passes (the top token's p then missing its own cutoff).
  __device__ __forceinline__ static float round(float f) {
    asm volatile("" : "+v"(f));
    return f;
  }
};

// Philox4x32-10 (Random123): 10 rounds, key schedule bumped between rounds.
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    const uint32_t lo0 = 0xD2511F53u * c.x, hi0 = __umulhi(0xD2511F53u, c.x);
    const uint32_t lo1 = 0xCD9E8D57u * c.z, hi1 = __umulhi(0xCD9E8D57u, c.z);
    c = make_uint4(hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0);
  }
  return c;
}

// Uniform in (0, 1) from 23 random bits, then a Gumbel variate.
__device__ __forceinline__ float gumbel(uint32_t bits) {
  const float u = (static_cast<float>(bits >> 9) + 0.5f) * 1.1920928955078125e-07f;  // 2^-23
  return -__logf(-__logf(u));
}

struct SampleArgs {
  const void* logits;
  int64_t rows, vocab, stride;
  const float* temperature;
  const int32_t* top_k;
  const float* top_p;
  uint32_t seed_lo, seed_hi, offset_lo, offset_hi;
  int64_t* out;
};

// Workgroup reductions through a small LDS scratch array.
struct Shared {
  uint32_t cnt[kBins0];
  unsigned long long mass[kBins0];
  float red_f[kWarps];
  float red_g[kWarps];
  int64_t red_i[kWarps];
  uint32_t scan_c[kWarps];
  unsigned long long scan_m[kWarps];
  // Selection state broadcast to the workgroup.
  uint32_t k_prefix, k_rem, p_prefix, p_lowest;
  unsigned long long p_rem;
  int p_found, k_found, k_active;
};

// Unsigned key that orders like the float value (non-NaN): larger s, larger key.
__device__ __forceinline__ uint32_t order_key(float s) {
  const uint32_t u = __float_as_uint(s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

__device__ __forceinline__ bool better(float v, int64_t i, float bv, int64_t bi) {
  // Larger value wins, NaN beats everything, lower index breaks ties.
  const bool vn = v != v, bn = bv != bv;
  if (vn || bn) return vn && (!bn || i < bi);
  return v > bv || (v == bv && i < bi);
}

__device__ void block_argmax(Shared& sh, float& v, int64_t& i) {
  const int lane = threadIdx.x % kWave, warp = threadIdx.x / kWave;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float ov = __shfl_xor(v, off);
    const int64_t oi = __shfl_xor(i, off);
    if (better(ov, oi, v, i)) {
      v = ov;
      i = oi;
    }
  }
  if (lane == 0) {
    sh.red_f[warp] = v;
    sh.red_i[warp] = i;
  }
  __syncthreads();
  v = sh.red_f[0];
  i = sh.red_i[0];
  for (int w = 1; w < kWarps; ++w)
    if (better(sh.red_f[w], sh.red_i[w], v, i)) {
      v = sh.red_f[w];
      i = sh.red_i[w];
    }
  __syncthreads();
}

// Visit every element of the row as (index, value). The vector body uses
// 128-bit loads when the row is aligned; a scalar loop covers the rest.
template <int DT, typename F>
__device__ __forceinline__ void for_each(const SampleArgs& a, int64_t row, bool vec, F&& f) {
  using L = Logit<DT>;
  using W = typename L::Word;
  const W* base = static_cast<const W*>(a.logits) + row * a.stride;
  int64_t start = 0;
  if (vec) {
    const int64_t groups = a.vocab / L::kVec;
    for (int64_t g = threadIdx.x; g < groups; g += kThreads) {
      const uint4 raw = ld128(base + g * L::kVec);
      const W* w = reinterpret_cast<const W*>(&raw);
#pragma unroll
      for (int j = 0; j < L::kVec; ++j) f(g * L::kVec + j, L::to_float(w[j]));
    }
    start = groups * L::kVec;
  }
  for (int64_t i = start + threadIdx.x; i < a.vocab; i += kThreads) f(i, L::to_float(base[i]));
}

// Inclusive workgroup prefix sum of (count, mass) in thread order.
__device__ void block_scan(Shared& sh, uint32_t& c, unsigned long long& m, uint32_t& total_c,
                           unsigned long long& total_m) {
  const int lane = threadIdx.x % kWave, warp = threadIdx.x / kWave;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t oc = __shfl_up(c, off);
    const unsigned long long om = __shfl_up(m, off);
    if (lane >= off) {
      c += oc;
      m += om;
    }
  }
  if (lane == kWave - 1) {
    sh.scan_c[warp] = c;
    sh.scan_m[warp] = m;
  }
  __syncthreads();
  uint32_t pc = 0;
  unsigned long long pm = 0;
  total_c = 0;
  total_m = 0;
  for (int w = 0; w < kWarps; ++w) {
    if (w < warp) {
      pc += sh.scan_c[w];
      pm += sh.scan_m[w];
    }
    total_c += sh.scan_c[w];
    total_m += sh.scan_m[w];
  }
  c += pc;
  m += pm;
  __syncthreads();
}

__device__ __forceinline__ float probability(float s, float m, float inv_z) {
  return exp2f((s - m) * kLog2e) * inv_z;
}
__device__ __forceinline__ unsigned long long fixed_mass(float p) {
  return static_cast<unsigned long long>(p * kFixedScale + 0.5f);
}
// Mass that the top-p cutoff has to reach: at least one unit, so the top bin is selectable.
__device__ __forceinline__ unsigned long long mass_target(float top_p) {
  const unsigned long long t = static_cast<unsigned long long>(top_p * kFixedScale);
  return t ? t : 1ull;
}
// Below the k-th largest scaled logit by far more than the rounding of p: every token under
// this edge has a p strictly below the k-th largest p.
__device__ __forceinline__ float candidate_edge(float s_k, float m) {
  return s_k - (fabsf(s_k - m) + 1.f) * 0x1p-12f;
}

// Both cutoffs and the draw among n gathered candidates (cand_p is scratch; the lists are in
// LDS and complete: every token of the row whose p can reach the k-th largest is listed).
// False, and nothing written, when fewer than k candidates exist or, without MASSLESS, the k-th p
// has no fixed-point mass under a top-p cutoff (the branch for it costs sample_row, whose search
// finds the cutoff as well, the unrolling of its scans: 60 -> 72 us for 256 rows of 20,000 cut by
// top-p). All kThreads threads call it.
template <bool MASSLESS>
__device__ __forceinline__ bool finish_candidates(Shared& sh, const SampleArgs& a, int64_t row,
                                                  const uint32_t* cand_i, const float* cand_s,
                                                  float* cand_p, uint32_t n, float m, float inv_z,
                                                  int64_t top_k, float top_p) {
  const bool use_p = top_p < 1.f;
  const unsigned long long p_target = mass_target(top_p);
  for (uint32_t t = threadIdx.x; t < n; t += kThreads)
    cand_p[t] = probability(cand_s[t], m, inv_z);
  if (threadIdx.x == 0) sh.k_found = 0;
  __syncthreads();
  // The k-th largest p: the candidate value v with #(p > v) < k <= #(p >= v).
  for (uint32_t t = threadIdx.x; t < n; t += kThreads) {
    const float v = cand_p[t];
    uint32_t gt = 0, ge = 0;
    for (uint32_t u = 0; u < n; ++u) {
      gt += cand_p[u] > v;
      ge += cand_p[u] >= v;
    }
    if (gt < static_cast<uint32_t>(top_k) && ge >= static_cast<uint32_t>(top_k)) {
      sh.red_f[0] = v;  // every thread that gets here writes the same value
      sh.k_found = 1;
    }
  }
  __syncthreads();
  const float p_k = sh.red_f[0];
  if (!sh.k_found || (!MASSLESS && use_p && fixed_mass(p_k) == 0)) return false;
  float cut = p_k;
  if (use_p) {
    // Mass at or above p_k; when it reaches top_p, the top-p cutoff is the largest
    // candidate value whose mass at or above reaches it.
    unsigned long long mk = 0;
    for (uint32_t t = threadIdx.x; t < n; t += kThreads)
      if (cand_p[t] >= p_k) mk += fixed_mass(cand_p[t]);
    uint32_t zc = 0;
    uint32_t tc;
    unsigned long long tm;
    block_scan(sh, zc, mk, tc, tm);
    if (tm >= p_target) {
      float best_v = p_k;
      for (uint32_t t = threadIdx.x; t < n; t += kThreads) {
        const float v = cand_p[t];
        if (v < p_k) continue;
        unsigned long long mv = 0;
        for (uint32_t u = 0; u < n; ++u)
          if (cand_p[u] >= v) mv += fixed_mass(cand_p[u]);
        if (mv >= p_target) best_v = fmaxf(best_v, v);
      }
      float bv = best_v;
      int64_t bi = 0;
      block_argmax(sh, bv, bi);
      cut = bv;
    } else if (MASSLESS && fixed_mass(p_k) == 0) {
      // Rounding kept the whole mass below the target, and all of it lies above p_k: the cutoff
      // is the lowest p that has any.
      float low = -INFINITY;
      for (uint32_t t = threadIdx.x; t < n; t += kThreads)
        if (fixed_mass(cand_p[t])) low = fmaxf(low, -cand_p[t]);
      int64_t bi = 0;
      block_argmax(sh, low, bi);
      cut = -low;
    }
  }
  // The race over the surviving candidates (order-independent: larger key, then lower index).
  float best = -INFINITY;
  int64_t best_i = a.vocab;
  for (uint32_t t = threadIdx.x; t < n; t += kThreads) {
    const float pt = cand_p[t];
    if (!(pt > 0.f && pt >= cut)) continue;
    const int64_t i = cand_i[t];
    const uint4 rnd =
        philox4x32_10(make_uint4(static_cast<uint32_t>(i >> 2), static_cast<uint32_t>(row),
                                 a.offset_lo, a.offset_hi),
                      a.seed_lo, a.seed_hi);
    const uint32_t words[4] = {rnd.x, rnd.y, rnd.z, rnd.w};
    const float key = cand_s[t] + gumbel(words[i & 3]);
    if (key > best || (key == best && i < best_i)) {
      best = key;
      best_i = i;
    }
  }
  block_argmax(sh, best, best_i);
  if (threadIdx.x == 0) a.out[row] = best_i < a.vocab ? best_i : -1;
  return true;
}

// One whole row by one workgroup.
template <int DT>
__device__ __forceinline__ void sample_row(Shared& sh, const SampleArgs& a, int64_t row, bool vec) {
  const int64_t vocab = a.vocab;

  float temperature = a.temperature[row];
  float top_p = a.top_p[row];
  if (!(top_p >= 0.f && top_p <= 1.f)) top_p = 1.f;  // NaN/inf/out of range -> 1
  int64_t top_k = a.top_k[row];
  if (top_k <= 0 || top_k > vocab) top_k = vocab;

  if (temperature <= 0.f || top_p == 0.f) {
    float bv = -INFINITY;
    int64_t bi = vocab;  // any real index beats the sentinel
    bool first = true;
    for_each<DT>(a, row, vec, [&](int64_t i, float x) {
      if (first || better(x, i, bv, bi)) {
        bv = x;
        bi = i;
        first = false;
      }
    });
    block_argmax(sh, bv, bi);
    if (threadIdx.x == 0) a.out[row] = bi < vocab ? bi : 0;
    return;
  }

  using L = Logit<DT>;
  const float inv_t = 1.f / temperature;
  auto scaled = [&](float x) { return L::round(x * inv_t); };
  const bool filter = top_k < vocab || top_p < 1.f;
  const uint32_t k0 = a.seed_lo, k1 = a.seed_hi;

  // Race over the survivors of `keep`; also reports whether a NaN was seen.
  auto race = [&](auto keep, bool& nan_seen, float& best, int64_t& best_i) {
    best = -INFINITY;
    best_i = vocab;
    int64_t cached_group = -1;
    uint4 rnd = make_uint4(0, 0, 0, 0);
    for_each<DT>(a, row, vec, [&](int64_t i, float x) {
      const float s = scaled(x);
      if (s != s || s == INFINITY) nan_seen = true;
      if (!keep(s) || s == -INFINITY) return;
      const int64_t group = i >> 2;
      if (group != cached_group) {
        rnd = philox4x32_10(make_uint4(static_cast<uint32_t>(group), static_cast<uint32_t>(row),
                                       a.offset_lo, a.offset_hi),
                            k0, k1);
        cached_group = group;
      }
      const uint32_t words[4] = {rnd.x, rnd.y, rnd.z, rnd.w};
      const float key = s + gumbel(words[i & 3]);
      if (key > best || (key == best && i < best_i)) {
        best = key;
        best_i = i;
      }
    });
  };

  if (!filter) {
    bool nan_seen = false;
    float best;
    int64_t best_i;
    race([](float) { return true; }, nan_seen, best, best_i);
    const int any_nan = __syncthreads_or(nan_seen);
    block_argmax(sh, best, best_i);
    if (threadIdx.x == 0) a.out[row] = (any_nan || best_i >= vocab) ? -1 : best_i;
    return;
  }

  // Top-k rows first try a shorter route (the candidate path below); pass 1 then also
  // counts the scaled logits in 4,096 bins of their top order-key bits.
  const bool fast_k = top_k < vocab;
  if (fast_k) {
    for (int b = threadIdx.x; b < kBins0; b += kThreads) sh.cnt[b] = 0;
    __syncthreads();
  }
  // Pass 1: max and sum of exp(s - max).
  float m = -INFINITY, z = 0.f;
  bool nan_seen = false;
  for_each<DT>(a, row, vec, [&](int64_t, float x) {
    const float s = scaled(x);
    if (fast_k && s == s && s != -INFINITY) atomicAdd(&sh.cnt[order_key(s) >> 20], 1u);
    if (s != s || s == INFINITY) {  // softmax of a row holding +inf is NaN throughout
      nan_seen = true;
      return;
    }
    if (s == -INFINITY) return;
    if (s > m) {
      z = z * exp2f((m - s) * kLog2e) + 1.f;
      m = s;
    } else {
      z += exp2f((s - m) * kLog2e);
    }
  });
  {
    const int lane = threadIdx.x % kWave, warp = threadIdx.x / kWave;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float om = __shfl_xor(m, off), oz = __shfl_xor(z, off);
      const float nm = fmaxf(m, om);
      z = (m == -INFINITY ? 0.f : z * exp2f((m - nm) * kLog2e)) +
          (om == -INFINITY ? 0.f : oz * exp2f((om - nm) * kLog2e));
      m = nm;
    }
    if (lane == 0) {
      sh.red_f[warp] = m;
      sh.red_g[warp] = z;
    }
    const int any_nan = __syncthreads_or(nan_seen);
    m = -INFINITY;
    for (int w = 0; w < kWarps; ++w) m = fmaxf(m, sh.red_f[w]);
    z = 0.f;
    for (int w = 0; w < kWarps; ++w)
      if (sh.red_f[w] != -INFINITY) z += sh.red_g[w] * exp2f((sh.red_f[w] - m) * kLog2e);
    __syncthreads();
    if (any_nan || m == -INFINITY || !(z > 0.f)) {
      if (threadIdx.x == 0) a.out[row] = -1;
      return;
    }
  }
  const float inv_z = 1.f / z;
  auto prob = [&](float s) { return probability(s, m, inv_z); };
  const bool use_p = top_p < 1.f;
  const unsigned long long p_target = mass_target(top_p);

  // Candidate path (top-k rows): the order-key histogram of pass 1 gives the bin b1 that
  // holds the k-th largest scaled logit. Every token with s >= s_lo (the bin's lower edge
  // less a margin far above the rounding of p) is a candidate, and every other token's p is
  // below every candidate's that lies in or above b1, so the k-th largest p of the row, the
  // top-p cutoff at or above it (its mass in the same 2^-40 fixed point) and the survivors
  // are all found among the candidates, which are gathered once into LDS. Exactly the
  // cutoffs and draw of the radix path below; that path runs when the candidates do not
  // fit (heavy ties), a row has fewer than k finite logits, or the k-th p has no fixed-point
  // mass. Two row passes instead of four, one of them without exponentials.
  if (fast_k) {
    // Bin b1 from the top, through the same thread-owns-4-bins suffix scan as below.
    const int b0 = threadIdx.x * 4;
    uint32_t c4[4];
    for (int j = 0; j < 4; ++j) c4[j] = sh.cnt[b0 + j];
    uint32_t csum = c4[0] + c4[1] + c4[2] + c4[3];
    unsigned long long zero = 0;
    uint32_t total_c;
    unsigned long long total_m;
    block_scan(sh, csum, zero, total_c, total_m);
    uint32_t c_above = total_c - csum;
    if (threadIdx.x == 0) sh.k_found = 0;
    __syncthreads();
    for (int j = 3; j >= 0; --j) {
      if (c4[j] && c_above < static_cast<uint32_t>(top_k) &&
          c_above + c4[j] >= static_cast<uint32_t>(top_k)) {
        sh.k_prefix = static_cast<uint32_t>(b0 + j);
        sh.k_rem = c_above + c4[j];  // tokens in bins b1 and above
        sh.k_found = 1;
      }
      c_above += c4[j];
    }
    __syncthreads();
    bool ok = sh.k_found && sh.k_rem <= kCandidates;
    if (ok) {
      const float s_lo = candidate_edge(key_value(sh.k_prefix << 20), m);
      uint32_t* cand_i = reinterpret_cast<uint32_t*>(sh.mass);
      float* cand_s = reinterpret_cast<float*>(cand_i + kCandidates);
      float* cand_p = cand_s + kCandidates;
      if (threadIdx.x == 0) sh.p_lowest = 0;  // candidate count
      __syncthreads();
      for_each<DT>(a, row, vec, [&](int64_t i, float x) {
        const float s = scaled(x);
        if (!(s >= s_lo) || s == -INFINITY) return;
        const uint32_t slot = atomicAdd(&sh.p_lowest, 1u);
        if (slot < kCandidates) {
          cand_i[slot] = static_cast<uint32_t>(i);
          cand_s[slot] = s;
        }
      });
      __syncthreads();
      const uint32_t n = sh.p_lowest;
      ok = n <= kCandidates;
      if (ok) {
        if (finish_candidates<false>(sh, a, row, cand_i, cand_s, cand_p, n, m, inv_z, top_k,
                                     top_p))
          return;
      }
    }
    __syncthreads();  // the candidate lists alias the mass histogram of the radix path
  }

  // Passes 2-4: radix selection of the two cutoffs over the bits of p.
  if (threadIdx.x == 0) {
    sh.k_prefix = 0;
    sh.k_rem = static_cast<uint32_t>(top_k);
    sh.k_active = top_k < vocab;
    sh.p_prefix = 0;
    sh.p_rem = p_target;
  }
  constexpr int kShift[3] = {19, 9, 0};
  constexpr int kBits[3] = {12, 10, 9};
  for (int pass = 0; pass < 3; ++pass) {
    const int shift = kShift[pass], bits = kBits[pass];
    const int nbins = 1 << bits;
    for (int b = threadIdx.x; b < nbins; b += kThreads) {
      sh.cnt[b] = 0;
      sh.mass[b] = 0;
    }
    if (threadIdx.x == 0) {
      sh.p_found = 0;
      sh.k_found = 0;
      sh.p_lowest = 0xffffffffu;
    }
    __syncthreads();
    const uint32_t kp = sh.k_prefix, pp = sh.p_prefix;
    const bool use_k = sh.k_active;
    const int above = shift + bits;
    for_each<DT>(a, row, vec, [&](int64_t, float x) {
      const float s = scaled(x);
      if (s == -INFINITY) return;
      const float p = prob(s);
      const uint32_t key = __float_as_uint(p);
      const uint32_t bin = (key >> shift) & (nbins - 1);
      const uint32_t hi = above >= 32 ? 0u : key >> above;
      if (use_k && hi == kp) atomicAdd(&sh.cnt[bin], 1u);
      if (use_p && hi == pp) {
        const unsigned long long fx = fixed_mass(p);
        if (fx) atomicAdd(&sh.mass[bin], fx);
      }
    });
    __syncthreads();

    // Each thread owns 4 consecutive bins; the suffix above them is the total
    // minus the inclusive prefix of the thread sums.
    const int b0 = threadIdx.x * 4;
    uint32_t c4[4] = {0, 0, 0, 0};
    unsigned long long m4[4] = {0, 0, 0, 0};
    for (int j = 0; j < 4; ++j)
      if (b0 + j < nbins) {
        c4[j] = sh.cnt[b0 + j];
        m4[j] = sh.mass[b0 + j];
      }
    uint32_t csum = c4[0] + c4[1] + c4[2] + c4[3];
    unsigned long long msum = m4[0] + m4[1] + m4[2] + m4[3];
    uint32_t total_c;
    unsigned long long total_m;
    block_scan(sh, csum, msum, total_c, total_m);
    uint32_t c_above = total_c - csum;
    unsigned long long m_above = total_m - msum;
    const uint32_t k_rem = sh.k_rem;
    const unsigned long long p_rem = sh.p_rem;
    for (int j = 3; j >= 0; --j) {
      const uint32_t b = static_cast<uint32_t>(b0 + j);
      if (use_k && c4[j] && c_above < k_rem && c_above + c4[j] >= k_rem) {
        sh.k_prefix = (kp << bits) | b;
        sh.k_rem = k_rem - c_above;
        sh.k_found = 1;
      }
      if (use_p && m4[j] && m_above < p_rem && m_above + m4[j] >= p_rem) {
        sh.p_prefix = (pp << bits) | b;
        sh.p_rem = p_rem - m_above;
        sh.p_found = 1;
      }
      if (use_p && m4[j]) atomicMin(&sh.p_lowest, b);
      c_above += c4[j];
      m_above += m4[j];
    }
    __syncthreads();
    // Fewer than k finite logits: the top-k cutoff keeps everything.
    if (use_k && threadIdx.x == 0 && !sh.k_found) sh.k_active = 0;
    if (use_p && threadIdx.x == 0 && !sh.p_found) {
      // Rounding kept every prefix below the target: keep the whole lowest bin.
      const uint32_t b = sh.p_lowest == 0xffffffffu ? 0u : sh.p_lowest;
      sh.p_prefix = (pp << bits) | b;
      sh.p_rem = sh.mass[b];
    }
    __syncthreads();
  }
  const float cut_k = sh.k_active ? __uint_as_float(sh.k_prefix) : 0.f;
  const float cut_p = use_p ? __uint_as_float(sh.p_prefix) : 0.f;
  const float cut = fmaxf(cut_k, cut_p);

  // Pass 5: exponential race over the survivors.
  bool unused = false;
  float best;
  int64_t best_i;
  race([&](float s) { const float p = prob(s); return p > 0.f && p >= cut; }, unused, best,
       best_i);
  block_argmax(sh, best, best_i);
  if (threadIdx.x == 0) a.out[row] = best_i < vocab ? best_i : -1;
}

template <int DT>
__global__ __launch_bounds__(kThreads) void sample_kernel(SampleArgs a, bool vec) {
  __shared__ Shared sh;
  sample_row<DT>(sh, a, blockIdx.x, vec);
}

// ---------------------------------------------------------------------------
// A row over several workgroups. One workgroup per row leaves the chip idle for a handful of
// rows and walks a row two to five times; here every workgroup holds one segment of a row in
// registers, so the logits are read once for greedy, unfiltered and top-k rows. Bound by
// VALU work where the rows are many (an exponential per logit; 256 rows of 151,936 bf16 logits,
// top-k 50 and top-p 0.9: 37 us a call, 26 + 11 traced, against 65 with one workgroup per row), by
// latency and launches where they are few (5 mixed rows 209 -> 42 us, 5 top-k rows 56 -> 21):
//   sample_segments  per segment: the argmax, or the race's best token, or the segment's max
//                    and sum of exp(s - max); top-k rows also list the tokens at or above a
//                    bound on the segment's k-th largest (the k-th largest of the 256 threads'
//                    maxima);
//   mass_level       rows cut by top-p alone: mass histograms over the order key of s, a few
//                    bits per launch, each launch picking the bin that holds the cutoff in the
//                    previous launch's histogram (p grows with s, so the cutoff on s is the
//                    cutoff on p);
//   race_segments    those rows' race over the survivors, per segment;
//   sample_finish    one workgroup per row joins the segments. Rows whose lists overflow (heavy
//                    ties) or whose parameters fit none of the above take sample_row. Rows with
//                    fewer than k finite logits (a grammar's mask) and rows whose k-th p has no
//                    fixed-point mass (sharp logits) are joined too: 5 rows of 151,936 with 30
//                    tokens allowed 95 us when walked whole after the segments, 16 joined, with
//                    logits of deviation 25 283 and 21.
// Cutoffs and draws are sample_row's: masses are the same fixed-point sums, the race is the
// same, and the sum of exp differs by its fp32 rounding only.
// ---------------------------------------------------------------------------
constexpr int kSegThreads = 256;
constexpr int kSegWarps = kSegThreads / kWave;
constexpr int kChunk = kSegThreads * 8;   // elements a workgroup takes per step
constexpr int kMaxChunks = 4;             // steps held in registers (8: half the waves fit)
constexpr int kMaxSegments = 256;         // per row
constexpr uint32_t kSegList = 512;        // listed tokens per segment
constexpr int64_t kSplitTopK = 128;       // largest k of the segment lists
constexpr uint32_t kRowOwn = 8192;        // listed tokens of a row loaded before the bound is known
constexpr int kSegPeaks = kSegThreads / 16;
constexpr int kLevelBins = 1024;          // bins of the levels after the first

enum class Rule { kGreedy, kRace, kTopK, kTopP, kWhole };

struct RowRule {
  Rule rule;
  float temperature, top_p;
  int64_t top_k;
};

__device__ __forceinline__ RowRule row_rule(const SampleArgs& a, int64_t row, bool top_p_rows) {
  RowRule r;
  r.temperature = a.temperature[row];
  r.top_p = a.top_p[row];
  if (!(r.top_p >= 0.f && r.top_p <= 1.f)) r.top_p = 1.f;
  r.top_k = a.top_k[row];
  if (r.top_k <= 0 || r.top_k > a.vocab) r.top_k = a.vocab;
  if (r.temperature <= 0.f || r.top_p == 0.f)
    r.rule = Rule::kGreedy;
  else if (r.top_k == a.vocab)
    r.rule = r.top_p < 1.f ? (top_p_rows ? Rule::kTopP : Rule::kWhole) : Rule::kRace;
  else
    r.rule = r.top_k <= kSplitTopK ? Rule::kTopK : Rule::kWhole;
  return r;
}

struct Segment {
  float m, z;         // max of s and sum of exp(s - m)
  float bound;        // top-k rows: every token with s >= bound is listed
  uint32_t count;     // listed tokens (more than kSegList: the list is incomplete)
  float best;         // argmax value or race key
  uint32_t best_i;    // its index; vocab when the segment has none
  uint32_t bad;       // a NaN or +inf among s
  uint32_t pad;
};

struct LevelState {
  uint32_t prefix, pad;
  unsigned long long rem;
};

struct SplitArgs {
  Segment* seg;              // [rows][segments]
  float* peak;               // [rows][segments][kSegPeaks]: maxima of 16 threads each
  uint2* list;               // [rows][segments][kSegList]: (index, bits of s)
  LevelState* state;         // [rows][4]
  unsigned long long* hist;  // [rows][kBins0 + 2 kLevelBins], top_p_rows only
  int32_t segments;
  bool vec, top_p_rows;
};
constexpr int64_t kHistWords = kBins0 + 2 * kLevelBins;

// Bits of the order key told apart by each level: all the bits a logit of the type can differ
// in (fp16 values have 10 mantissa bits of fp32's 23 and more exponents in their denormals).
template <int DT>
__device__ __forceinline__ constexpr int level_bits(int level) {
  if (level == 0) return 12;
  return DT == 0 ? 4 : DT == 1 ? 7 : 10;
}
template <int DT>
constexpr int kLevels = DT == 2 ? 3 : 2;

// max(a, b, c) in one instruction; a NaN among them is passed over. (fmaxf spends a second
// instruction on each operand, for signalling NaNs.)
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// The chunk's 8 logits of this thread. Elements past the row are -inf, before and after scaling.
// VEC: 16-byte aligned rows of a multiple of 8 logits, so 8 are all inside or all past the row.
template <int DT, bool VEC>
struct Chunk {
  using W = typename Logit<DT>::Word;
  static constexpr int kWords = DT == 2 ? 2 : 1;
  static constexpr uint32_t kNone = DT == 0 ? 0xff80ff80u : DT == 1 ? 0xfc00fc00u : 0xff800000u;
  uint4 raw[kWords];
  __device__ __forceinline__ void load(const SampleArgs& a, int64_t row, uint32_t e) {
    const W* base = static_cast<const W*>(a.logits) + row * a.stride;
    const uint32_t vocab = static_cast<uint32_t>(a.vocab);
#pragma unroll
    for (int j = 0; j < kWords; ++j) raw[j] = make_uint4(kNone, kNone, kNone, kNone);
    if constexpr (VEC) {
      if (e < vocab) {
#pragma unroll
        for (int j = 0; j < kWords; ++j) raw[j] = ld128(base + e + j * (8 / kWords));
      }
    } else {
      W v[8];
      __builtin_memcpy(v, raw, sizeof(v));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (e + j < vocab) v[j] = base[e + j];
      __builtin_memcpy(raw, v, sizeof(raw));
    }
  }
  __device__ __forceinline__ void values(float (&f)[8]) const {
    if constexpr (DT == 2) {
      __builtin_memcpy(f, raw, sizeof(f));
    } else {
      unpack8<DT>(raw[0], f);
    }
  }
  // Replaces the logits by the scaled logits s; returns their maximum (NaN aside). Rounding
  // keeps order, so the largest product rounds to the largest s.
  __device__ __forceinline__ float scale(float inv_t, uint32_t e, uint32_t vocab) {
    float f[8];
    values(f);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f[j] = f[j] * inv_t;
      if constexpr (DT == 2) f[j] = Logit<2>::round(f[j]);
      if constexpr (!VEC)
        if (e + j >= vocab) f[j] = -INFINITY;  // -inf times 0 (an infinite temperature) is NaN
    }
    float top = max3(max3(max3(f[0], f[1], f[2]), f[3], f[4]), max3(f[5], f[6], f[7]), -INFINITY);
    top = Logit<DT>::round(top);
    if constexpr (DT == 2)
      __builtin_memcpy(raw, f, sizeof(f));
    else
      raw[0] = pack8<DT>(f);
    if constexpr (VEC)
      if (e >= vocab) {
#pragma unroll
        for (int j = 0; j < kWords; ++j) raw[j] = make_uint4(kNone, kNone, kNone, kNone);
        top = -INFINITY;
      }
    return top;
  }
  // Forgets what the compiler knows of the values, so that a later pass unpacks them again
  // rather than keeping 8 floats a chunk alive.
  __device__ __forceinline__ void repack() {
#pragma unroll
    for (int j = 0; j < kWords; ++j)
      asm volatile("" : "+v"(raw[j].x), "+v"(raw[j].y), "+v"(raw[j].z), "+v"(raw[j].w));
  }
};

struct alignas(16) SegShared {
  float peak[kSegThreads];
  float red_f[kSegWarps];
  uint32_t red_i[kSegWarps];
  float bound;
  uint32_t count;
};

// The k-th largest of a wave's values, 4 per lane, by the 16 top bits of their order keys (so at
// least k of them reach the result); -inf when fewer than k are finite. One ballot per value
// and bit: no LDS and no barriers.
__device__ __forceinline__ float kth_largest(const float (&v)[4], uint32_t k) {
  uint32_t key[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) key[t] = v[t] == -INFINITY ? 0u : order_key(v[t]);
  uint32_t found = 0;
#pragma unroll
  for (int b = 31; b >= 16; --b) {
    const uint32_t next = found | (1u << b);
    uint32_t c = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) c += __popcll(__ballot(key[t] >= next));
    found = c >= k ? next : found;
  }
  return found ? key_value(found) : -INFINITY;
}

__device__ __forceinline__ float wave_max(float x) {
  x = row16_max(x);
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}

// Workgroup best (value, index) of a segment: larger value, then lower index; NaN above all.
__device__ __forceinline__ void segment_best(SegShared& sh, float& v, uint32_t& i) {
  const int lane = threadIdx.x % kWave, warp = threadIdx.x / kWave;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float ov = __shfl_xor(v, off);
    const uint32_t oi = __shfl_xor(i, off);
    if (better(ov, oi, v, i)) {
      v = ov;
      i = oi;
    }
  }
  if (lane == 0) {
    sh.red_f[warp] = v;
    sh.red_i[warp] = i;
  }
  __syncthreads();
  v = sh.red_f[0];
  i = sh.red_i[0];
  for (int w = 1; w < kSegWarps; ++w)
    if (better(sh.red_f[w], sh.red_i[w], v, i)) {
      v = sh.red_f[w];
      i = sh.red_i[w];
    }
}

// Race keys of 8 neighbouring tokens starting at e; `keep` tells which take part.
template <typename Keep>
__device__ __forceinline__ void race8(const SampleArgs& a, int64_t row, uint32_t e,
                                      const float (&s)[8], Keep&& keep, float& best,
                                      uint32_t& best_i) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    bool any = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) any = any || keep(s[4 * h + j]);
    if (!any) continue;
    const uint4 rnd =
        philox4x32_10(make_uint4((e >> 2) + h, static_cast<uint32_t>(row),
                                 a.offset_lo, a.offset_hi),
                      a.seed_lo, a.seed_hi);
    const uint32_t words[4] = {rnd.x, rnd.y, rnd.z, rnd.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!keep(s[4 * h + j])) continue;
      const float key = s[4 * h + j] + gumbel(words[j]);
      const uint32_t i = e + 4 * h + j;
      if (key > best || (key == best && i < best_i)) {
        best = key;
        best_i = i;
      }
    }
  }
}

// Max and sum of exp over a row's segments. Every wave that calls it gets the same bits.
// False for an invalid distribution (NaN, +inf, or nothing finite).
__device__ __forceinline__ bool join_segments(const Segment* seg, int n, float& m, float& z) {
  const int lane = threadIdx.x % kWave;
  m = -INFINITY;
  bool bad = false;
  for (int j = lane; j < n; j += kWave) {
    m = fmaxf(m, seg[j].m);
    bad = bad || seg[j].bad;
  }
  m = wave_max(m);
  z = 0.f;
  for (int j = lane; j < n; j += kWave)
    if (seg[j].m != -INFINITY) z += seg[j].z * exp2f((seg[j].m - m) * kLog2e);
  z = wave_sum(z);
  return !__any(bad) && m != -INFINITY && z > 0.f;
}

template <int DT, int NCH, bool VEC>
__global__ __launch_bounds__(kSegThreads) void sample_segments(SampleArgs a, SplitArgs p) {
  __shared__ SegShared sh;
  const int64_t row = blockIdx.y;
  const int tid = threadIdx.x, lane = tid % kWave, warp = tid / kWave;
  const RowRule r = row_rule(a, row, p.top_p_rows);
  if (r.rule == Rule::kWhole) return;  // sample_finish takes the row whole
  // Indexes fit 32 bits: a split row has at most kMaxSegments * kMaxChunks * kChunk elements.
  const uint32_t vocab = static_cast<uint32_t>(a.vocab);
  const uint32_t e0 = blockIdx.x * uint32_t(NCH * kChunk) + tid * 8;
  Segment* out = p.seg + row * p.segments + blockIdx.x;

  // Unfiltered rows stream their chunks (the race's random words would crowd out chunks held in
  // registers).
  if (r.rule == Rule::kRace) {
    const float inv_t = 1.f / r.temperature;
    float best = -INFINITY;
    uint32_t best_i = vocab;
    bool bad = false;
    Chunk<DT, VEC> next;
    next.load(a, row, e0);
#pragma unroll 1
    for (int c = 0; c < NCH; ++c) {
      Chunk<DT, VEC> x = next;
      const uint32_t e = e0 + c * kChunk;
      if (c + 1 < NCH) next.load(a, row, e + kChunk);
      float s[8];
      x.scale(inv_t, e, vocab);
      x.values(s);
#pragma unroll
      for (int j = 0; j < 8; ++j) bad = bad || !(s[j] < INFINITY);
      race8(a, row, e, s, [](float v) { return v > -INFINITY; }, best, best_i);
    }
    const int any_bad = __syncthreads_or(bad);
    segment_best(sh, best, best_i);
    if (tid == 0) {
      out->best = best;
      out->best_i = best_i;
      out->bad = any_bad;
    }
    return;
  }

  if (r.rule == Rule::kTopP) {
    // The row's histograms for the next launches, cleared by its segments together.
    unsigned long long* h = p.hist + row * kHistWords;
    for (int64_t i = int64_t(blockIdx.x) * kSegThreads + tid; i < kHistWords;
         i += int64_t(p.segments) * kSegThreads)
      h[i] = 0;
  }
  Chunk<DT, VEC> x[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) x[c].load(a, row, e0 + c * kChunk);

  if (r.rule == Rule::kGreedy) {
    // A thread looks for its first maximum chunk by chunk, and element by element only in
    // chunks that raise it or hold a NaN (their sum is one).
    float best = -INFINITY;
    uint32_t best_i = vocab;  // any real index beats the sentinel
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      float f[8];
      x[c].values(f);
      const uint32_t e = e0 + c * kChunk;
      const float top = max3(max3(max3(f[0], f[1], f[2]), f[3], f[4]), max3(f[5], f[6], f[7]), best);
      const float sum = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
      if (best_i != vocab && !(top > best) && sum == sum) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (e + j < vocab && better(f[j], e + j, best, best_i)) {
          best = f[j];
          best_i = e + j;
        }
    }
    segment_best(sh, best, best_i);
    if (tid == 0) {
      out->best = best;
      out->best_i = best_i;
    }
    return;
  }

  const float inv_t = 1.f / r.temperature;
  float cm[NCH], tm = -INFINITY;  // maxima per chunk and thread, then of the workgroup
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    cm[c] = x[c].scale(inv_t, e0 + c * kChunk, vocab);
    tm = max3(tm, cm[c], -INFINITY);
    x[c].repack();
    __builtin_amdgcn_sched_barrier(0);
  }
  const bool listed = r.rule == Rule::kTopK;
  const float rm = row16_max(tm);
  float wm = fmaxf(rm, __shfl_xor(rm, 16));
  wm = fmaxf(wm, __shfl_xor(wm, 32));
  if (lane == 0) sh.red_f[warp] = wm;
  if (listed) {
    sh.peak[tid] = tm;
    if (lane % 16 == 0)
      p.peak[(row * p.segments + blockIdx.x) * kSegPeaks + tid / 16] = rm;
    if (tid == 0) sh.count = 0;
  }
  __syncthreads();
  float m = sh.red_f[0];
  for (int w = 1; w < kSegWarps; ++w) m = fmaxf(m, sh.red_f[w]);
  if (m == -INFINITY || m == INFINITY) {  // nothing finite, or a +inf: only a NaN is to be found
    bool bad = m == INFINITY;
    for (int c = 0; c < NCH; ++c) {
      float s[8];
      x[c].values(s);
      for (int j = 0; j < 8; ++j) bad = bad || s[j] != s[j];
    }
    const int any_bad = __syncthreads_or(bad);
    if (tid == 0) *out = Segment{m, 0.f, 0.f, 0u, 0.f, vocab, static_cast<uint32_t>(any_bad), 0u};
    return;
  }
  if (listed && warp == 0) {
    // At least k tokens of the segment reach the k-th largest of its threads' maxima.
    const float4 v4 = *reinterpret_cast<const float4*>(sh.peak + 4 * lane);
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    const float t = kth_largest(v, static_cast<uint32_t>(r.top_k));
    if (lane == 0) sh.bound = t == -INFINITY ? -FLT_MAX : t - (fabsf(t - m) + 1.f) * 0x1p-11f;
  }

  // fp32 sums with the hardware exponential: a term it flushes to zero lies below 2^-126
  // beside the maximum's own 1.
  float z = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    float s[8];
    x[c].values(s);
#pragma unroll
    for (int j = 0; j < 8; ++j) z += __builtin_amdgcn_exp2f((s[j] - m) * kLog2e);
    x[c].repack();
    __builtin_amdgcn_sched_barrier(0);
  }
  float bound = 0.f;
  if (listed) {
    __syncthreads();
    bound = sh.bound;
    uint2* list = p.list + (row * p.segments + blockIdx.x) * int64_t(kSegList);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      if (cm[c] >= bound) {
        float s[8];
        x[c].values(s);
        uint32_t hits = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) hits |= s[j] >= bound ? 1u << j : 0u;
        while (hits) {
          const uint32_t j = __builtin_ctz(hits);
          hits &= hits - 1;
          float v = s[0];
#pragma unroll
          for (uint32_t t = 1; t < 8; ++t) v = j == t ? s[t] : v;
          const uint32_t slot = atomicAdd(&sh.count, 1u);
          if (slot < kSegList) list[slot] = make_uint2(e0 + c * kChunk + j, __float_as_uint(v));
        }
      }
    }
  }
  z = wave_sum(z);
  __syncthreads();  // red_f's readers are done; the list is complete
  if (lane == 0) sh.red_f[warp] = z;
  __syncthreads();
  if (tid == 0) {
    z = (sh.red_f[0] + sh.red_f[1]) + (sh.red_f[2] + sh.red_f[3]);
    *out = Segment{m, z, bound, sh.count, 0.f, vocab, z != z ? 1u : 0u, 0u};  // a NaN among s
  }
}

// Scan of the previous level's histogram by one workgroup of kSegThreads: the bin where the
// mass from the top reaches st.rem joins the prefix; when rounding keeps every prefix below it,
// the lowest bin that holds mass.
template <int NBINS>
__device__ __forceinline__ LevelState next_state(const unsigned long long* hist, LevelState st,
                                                 int bits, unsigned long long* sh_m,
                                                 uint32_t* sh_bin, unsigned long long* sh_rem) {
  constexpr int kOwn = NBINS / kSegThreads;
  const int tid = threadIdx.x, lane = tid % kWave, warp = tid / kWave;
  unsigned long long own[kOwn], sum = 0;
  int lowest = NBINS;
#pragma unroll
  for (int j = kOwn - 1; j >= 0; --j) {
    own[j] = hist[tid * kOwn + j];
    sum += own[j];
    if (own[j]) lowest = tid * kOwn + j;
  }
  unsigned long long incl = sum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned long long o = __shfl_down(incl, off);
    if (lane + off < kWave) incl += o;
  }
  if (tid == 0) *sh_bin = NBINS;
  if (lane == 0) sh_m[warp] = incl;
  __syncthreads();
  unsigned long long above = incl - sum, total = 0;
  for (int w = 0; w < kSegWarps; ++w) {
    if (w > warp) above += sh_m[w];
    total += sh_m[w];
  }
  if (total < st.rem) {
    if (lowest < NBINS) atomicMin(sh_bin, static_cast<uint32_t>(lowest));
    __syncthreads();
    const uint32_t b = *sh_bin < NBINS ? *sh_bin : 0u;
    return LevelState{(st.prefix << bits) | b, 0u, hist[b]};
  }
#pragma unroll
  for (int j = kOwn - 1; j >= 0; --j) {
    if (own[j] && above < st.rem && above + own[j] >= st.rem) {
      *sh_bin = static_cast<uint32_t>(tid * kOwn + j);
      *sh_rem = st.rem - above;
    }
    above += own[j];
  }
  __syncthreads();
  return LevelState{(st.prefix << bits) | *sh_bin, 0u, *sh_rem};
}

struct LevelShared {
  unsigned long long mass[kBins0];
  unsigned long long sum[kSegWarps];
  unsigned long long rem;
  uint32_t bin;
};

// The state after `level` histograms (level >= 1), kept by the row's first segment.
template <int DT>
__device__ __forceinline__ LevelState level_state(const SplitArgs& p, int64_t row, int level,
                                                  LevelShared& sh) {
  const unsigned long long* h = p.hist + row * kHistWords;
  LevelState* st = p.state + row * 4;
  const LevelState prev = st[level - 1];
  const LevelState now =
      level == 1 ? next_state<kBins0>(h, prev, level_bits<DT>(0), sh.sum, &sh.bin, &sh.rem)
                 : next_state<kLevelBins>(h + kBins0 + (level - 2) * kLevelBins, prev,
                                          level_bits<DT>(level - 1), sh.sum, &sh.bin, &sh.rem);
  if (blockIdx.x == 0 && threadIdx.x == 0) st[level] = now;
  return now;
}

template <int DT, int LEVEL, bool VEC>
__global__ __launch_bounds__(kSegThreads) void mass_level(SampleArgs a, SplitArgs p, int chunks) {
  __shared__ LevelShared sh;
  const int64_t row = blockIdx.y;
  const RowRule r = row_rule(a, row, p.top_p_rows);
  if (r.rule != Rule::kTopP) return;
  float m, z;
  if (!join_segments(p.seg + row * p.segments, p.segments, m, z)) return;
  constexpr int kNBins = LEVEL == 0 ? kBins0 : kLevelBins;
  uint32_t prefix = 0;
  if constexpr (LEVEL > 0)
    prefix = level_state<DT>(p, row, LEVEL, sh).prefix;
  else if (blockIdx.x == 0 && threadIdx.x == 0)
    p.state[row * 4] = LevelState{0u, 0u, mass_target(r.top_p)};
  for (int b = threadIdx.x; b < kNBins; b += kSegThreads) sh.mass[b] = 0;
  __syncthreads();
  constexpr int kAbove = LEVEL == 0 ? 32 : LEVEL == 1 ? 20 : 20 - level_bits<DT>(1);
  constexpr int kBits = level_bits<DT>(LEVEL);
  const float inv_z = 1.f / z, inv_t = 1.f / r.temperature;
  const uint32_t vocab = static_cast<uint32_t>(a.vocab);
  const uint32_t e0 = blockIdx.x * uint32_t(chunks * kChunk) + threadIdx.x * 8;
  for (int c = 0; c < chunks; ++c) {
    const uint32_t e = e0 + c * kChunk;
    if (e >= vocab) break;
    Chunk<DT, VEC> x;
    x.load(a, row, e);
    x.scale(inv_t, e, vocab);
    float s[8];
    x.values(s);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t key = order_key(s[j]);
      if (LEVEL > 0 && key >> (kAbove & 31) != prefix) continue;
      const unsigned long long fx = fixed_mass(probability(s[j], m, inv_z));  // 0 for -inf
      if (fx) atomicAdd(&sh.mass[key >> (kAbove - kBits) & ((1u << kBits) - 1u)], fx);
    }
  }
  __syncthreads();
  unsigned long long* h =
      p.hist + row * kHistWords + (LEVEL == 0 ? 0 : kBins0 + (LEVEL - 1) * kLevelBins);
  for (int b = threadIdx.x; b < (1 << kBits); b += kSegThreads)
    if (sh.mass[b]) atomicAdd(&h[b], sh.mass[b]);
}

template <int DT, bool VEC>
__global__ __launch_bounds__(kSegThreads) void race_segments(SampleArgs a, SplitArgs p,
                                                             int chunks) {
  __shared__ LevelShared sh;
  __shared__ SegShared sg;
  const int64_t row = blockIdx.y;
  const RowRule r = row_rule(a, row, p.top_p_rows);
  if (r.rule != Rule::kTopP) return;
  float m, z;
  if (!join_segments(p.seg + row * p.segments, p.segments, m, z)) return;
  constexpr int kShift = 20 - (kLevels<DT> - 1) * level_bits<DT>(1);
  const uint32_t prefix = level_state<DT>(p, row, kLevels<DT>, sh).prefix;
  // The cutoff's s: the prefix's bits, the others as they are in every value of the type.
  uint32_t key = prefix << kShift;
  if (!(key & 0x80000000u)) key |= (1u << kShift) - 1u;
  const float s_cut = key_value(key);
  const float inv_z = 1.f / z, inv_t = 1.f / r.temperature;
  const float cut = probability(s_cut, m, inv_z);
  const float edge = candidate_edge(s_cut, m);  // no token below it has a p that reaches cut
  const uint32_t vocab = static_cast<uint32_t>(a.vocab);
  const uint32_t e0 = blockIdx.x * uint32_t(chunks * kChunk) + threadIdx.x * 8;
  float best = -INFINITY;
  uint32_t best_i = vocab;
  for (int c = 0; c < chunks; ++c) {
    const uint32_t e = e0 + c * kChunk;
    if (e >= vocab) break;
    Chunk<DT, VEC> x;
    x.load(a, row, e);
    x.scale(inv_t, e, vocab);
    float s[8];
    x.values(s);
    race8(a, row, e, s,
          [&](float v) {
            if (!(v >= edge)) return false;
            const float q = probability(v, m, inv_z);
            return q > 0.f && q >= cut;
          },
          best, best_i);
  }
  segment_best(sg, best, best_i);
  if (threadIdx.x == 0) {
    Segment* out = p.seg + row * p.segments + blockIdx.x;
    out->best = best;
    out->best_i = best_i;
  }
}

// finish_candidates for at most 64 R candidates by one wave, each pair compared through lane
// broadcasts: with 60 candidates 4 us against the workgroup-wide version's 16 (its LDS round
// trips). False as well when tokens that could share the k-th p may not have been listed, the
// lists being complete down to listed_to only.
template <int R>
__device__ __forceinline__ bool finish_wave(const SampleArgs& a, int64_t row, const uint32_t* cand_i,
                            const float* cand_s, uint32_t n, float m, float inv_z, int64_t top_k,
                            float top_p, float listed_to) {
  const int lane = threadIdx.x % kWave;
  const bool use_p = top_p < 1.f;
  const uint32_t k = static_cast<uint32_t>(top_k);
  float s[R], p[R];
  uint32_t gt[R], ge[R];
  unsigned long long fx[R], mass[R];  // mass at or above the own p
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const uint32_t c = lane + kWave * t;
    s[t] = c < n ? cand_s[c] : -INFINITY;
    p[t] = c < n ? probability(s[t], m, inv_z) : -1.f;
    fx[t] = c < n ? fixed_mass(p[t]) : 0ull;
    gt[t] = ge[t] = 0;
    mass[t] = 0;
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int some = min(kWave, static_cast<int>(n) - kWave * t);
    for (int u = 0; u < some; ++u) {
      const float v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p[t]), u));
      const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(fx[t]), u);
      const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(fx[t] >> 32), u);
      const unsigned long long f = (static_cast<unsigned long long>(hi) << 32) | lo;
#pragma unroll
      for (int w = 0; w < R; ++w) {
        gt[w] += v > p[w];
        const bool above = v >= p[w];
        ge[w] += above;
        mass[w] += above ? f : 0ull;
      }
    }
  }
  // The k-th largest p and the mass at or above it.
  float p_k = -1.f;
  bool reached = false;
#pragma unroll
  for (int t = 0; t < R; ++t)
    if (p[t] >= 0.f && gt[t] < k && ge[t] >= k) {
      p_k = p[t];
      reached = mass[t] >= mass_target(top_p);
    }
  reached = __any(reached);
  p_k = wave_max(p_k);
  if (p_k < 0.f) return false;
  float s_k = INFINITY;  // the lowest s that has it
#pragma unroll
  for (int t = 0; t < R; ++t)
    if (p[t] == p_k) s_k = fminf(s_k, s[t]);
  s_k = -wave_max(-s_k);
  if (listed_to > candidate_edge(s_k, m)) return false;
  float cut = p_k;
  if (use_p && reached) {
#pragma unroll
    for (int t = 0; t < R; ++t)
      if (p[t] > cut && mass[t] >= mass_target(top_p)) cut = p[t];
    cut = wave_max(cut);
  } else if (use_p && fixed_mass(p_k) == 0) {
    // Rounding kept the whole mass below the target, and all of it lies above p_k: the cutoff is
    // the lowest p that has any.
    float low = INFINITY;
#pragma unroll
    for (int t = 0; t < R; ++t)
      if (fx[t]) low = fminf(low, p[t]);
    cut = -wave_max(-low);
  }
  float best = -INFINITY;
  uint32_t best_i = static_cast<uint32_t>(a.vocab);
#pragma unroll
  for (int t = 0; t < R; ++t) {
    if (!(p[t] > 0.f && p[t] >= cut)) continue;
    const uint32_t i = cand_i[lane + kWave * t];
    const uint4 rnd = philox4x32_10(
        make_uint4(i >> 2, static_cast<uint32_t>(row), a.offset_lo, a.offset_hi), a.seed_lo,
        a.seed_hi);
    const uint32_t w01 = i & 1 ? rnd.y : rnd.x, w23 = i & 1 ? rnd.w : rnd.z;
    const float key = s[t] + gumbel(i & 2 ? w23 : w01);
    if (key > best || (key == best && i < best_i)) {
      best = key;
      best_i = i;
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float ov = __shfl_xor(best, off);
    const uint32_t oi = __shfl_xor(best_i, off);
    if (ov > best || (ov == best && oi < best_i)) {
      best = ov;
      best_i = oi;
    }
  }
  if (lane == 0) a.out[row] = best_i < a.vocab ? static_cast<int64_t>(best_i) : -1;
  return true;
}

struct alignas(16) FinishShared {
  Segment seg[kMaxSegments];
  uint32_t offset[kMaxSegments];
  uint32_t count;
  float edge;
  int ok;
  Shared row;
};

template <int DT>
__global__ __launch_bounds__(kThreads) void sample_finish(SampleArgs a, SplitArgs p) {
  __shared__ FinishShared sh;
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid % kWave, warp = tid / kWave;
  const int n = p.segments;
  if (tid < 2 * n)  // two 16-byte halves per segment
    reinterpret_cast<uint4*>(sh.seg)[tid] =
        reinterpret_cast<const uint4*>(p.seg + row * p.segments)[tid];
  const RowRule r = row_rule(a, row, p.top_p_rows);
  if (r.rule == Rule::kWhole) {
    sample_row<DT>(sh.row, a, row, p.vec);
    return;
  }
  __syncthreads();
  const Segment* seg = sh.seg;
  if (r.rule != Rule::kTopK) {
    bool bad = false;
    if (r.rule == Rule::kTopP) {
      float m, z;
      bad = !join_segments(seg, n, m, z);
    }
    float best = -INFINITY;
    int64_t best_i = a.vocab;
    if (!bad && tid < n) {
      best = seg[tid].best;
      best_i = seg[tid].best_i;
      if (r.rule == Rule::kRace) bad = seg[tid].bad != 0;
    }
    const int any_bad = __syncthreads_or(bad);
    block_argmax(sh.row, best, best_i);
    if (tid == 0) {
      if (r.rule == Rule::kGreedy)
        a.out[row] = best_i < a.vocab ? best_i : 0;
      else
        a.out[row] = any_bad || best_i >= a.vocab ? -1 : best_i;
    }
    return;
  }

  float m, z;
  if (!join_segments(seg, n, m, z)) {
    if (tid == 0) a.out[row] = -1;
    return;
  }
  // Top-k: every wave finds the offsets of the segments' lists in the row's (the same values
  // into the same words, and a wave's LDS operations are in order, so it can read what its own
  // lanes wrote) and loads its tokens; meanwhile one wave takes a lower bound of the
  // k-th largest s from the segments' peaks, folded into 256 groups. The tokens that reach the
  // bound, little more than k, are kept for finish_candidates' work.
  uint32_t k = static_cast<uint32_t>(r.top_k);
  uint32_t total = 0;
  bool full = false;
  for (int j0 = 0; j0 < n; j0 += kWave) {
    const int j = j0 + lane;
    const uint32_t c = j < n ? seg[j].count : 0;
    full = full || c > kSegList;
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t o = __shfl_up(incl, off);
      if (lane >= off) incl += o;
    }
    if (j < n) sh.offset[j] = total + incl - c;
    total += __shfl(incl, kWave - 1);
  }
  bool ok = !__any(full);  // the same in every wave
  if (ok) {
    // Fewer listed tokens than k: no segment had k finite logits, so every finite one is listed,
    // and the cutoff at their number keeps them all, as the row's own does.
    k = min(k, total);
    constexpr int kOwn = kRowOwn / kThreads;
    const uint2* lists = p.list + row * n * int64_t(kSegList);
    auto listed = [&](uint32_t i) {
      int lo = 0, hi = n;  // the last segment whose list starts at or before i
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (sh.offset[mid] <= i)
          lo = mid;
        else
          hi = mid;
      }
      return lists[lo * int64_t(kSegList) + (i - sh.offset[lo])];
    };
    uint2 own[kOwn];
#pragma unroll
    for (int t = 0; t < kOwn; ++t) {
      const uint32_t i = tid + t * kThreads;
      if (i >= total) break;
      own[t] = listed(i);
    }
    if (warp == 0) {
      const float* peak = p.peak + row * n * kSegPeaks;
      float v[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      for (int i = 4 * lane; i < kSegPeaks * n; i += 4 * kWave) {
        const float4 q = *reinterpret_cast<const float4*>(peak + i);
        v[0] = fmaxf(v[0], q.x);
        v[1] = fmaxf(v[1], q.y);
        v[2] = fmaxf(v[2], q.z);
        v[3] = fmaxf(v[3], q.w);
      }
      const float t = kth_largest(v, k);
      if (lane == 0) {
        sh.edge = t == -INFINITY ? -FLT_MAX : candidate_edge(t, m);
        sh.count = 0;
      }
    }
    __syncthreads();
    const float edge = sh.edge;
    uint32_t* cand_i = reinterpret_cast<uint32_t*>(sh.row.mass);
    float* cand_s = reinterpret_cast<float*>(cand_i + kCandidates);
    float* cand_p = cand_s + kCandidates;
    auto keep = [&](uint2 token) {
      const float s = __uint_as_float(token.y);
      if (!(s >= edge)) return;
      const uint32_t slot = atomicAdd(&sh.count, 1u);
      if (slot < kCandidates) {
        cand_i[slot] = token.x;
        cand_s[slot] = s;
      }
    };
#pragma unroll
    for (int t = 0; t < kOwn; ++t) {
      if (tid + t * kThreads >= total) break;
      keep(own[t]);
    }
    // A k near the lists' largest, or many segments, list more.
    for (uint32_t i = tid + kRowOwn; i < total; i += kThreads) keep(listed(i));
    float listed_to = -FLT_MAX;
    for (int j = lane; j < n; j += kWave)
      if (seg[j].m != -INFINITY) listed_to = fmaxf(listed_to, seg[j].bound);
    listed_to = wave_max(listed_to);
    __syncthreads();
    const uint32_t kept = sh.count;
    // One wave up to 64 candidates, and up to 128 under a top-p cutoff, whose masses the whole
    // workgroup sums anew for every candidate (top-k 50 and top-p 0.9, 96 rows of 57,000, about 70
    // candidates: 24.3 us a call with one wave, 27.8 workgroup-wide; top-k 100 of one row of
    // 151,936 29.6 with the workgroup, 37.7 with one wave of four candidates a lane).
    if (kept <= kWave || (kept <= 2 * kWave && r.top_p < 1.f)) {
      if (warp == 0) {
        const float inv_z = 1.f / z;
        const bool done =
            kept <= kWave
                ? finish_wave<1>(a, row, cand_i, cand_s, kept, m, inv_z, k, r.top_p, listed_to)
                : finish_wave<2>(a, row, cand_i, cand_s, kept, m, inv_z, k, r.top_p, listed_to);
        if (lane == 0) sh.ok = done;
      }
      __syncthreads();
      ok = sh.ok != 0;
    } else {
      // The whole workgroup, where the bound itself shows the lists complete.
      ok = kept <= kCandidates && listed_to <= edge &&
           finish_candidates<true>(sh.row, a, row, cand_i, cand_s, cand_p, kept, m, 1.f / z, k,
                                   r.top_p);
    }
  }
  if (ok) return;
  __syncthreads();
  sample_row<DT>(sh.row, a, row, p.vec);
}

// How a call is split: chunks of kChunk logits per workgroup, workgroups per row. More chunks
// (fewer lists to join) while they still give 1,024 workgroups, four per CU, and kMinSegments
// segments, whose peaks bound the k-th largest for every k of the lists. Rows of up to 8 chunks
// are quicker in one launch (2,300 logits, top-k 50: 18 us against 27), and above 1,024 rows one
// workgroup per row fills the chip by itself.
constexpr int kMinSegments = 9;
static_assert(kMinSegments * kSegPeaks >= kSplitTopK, "a bound for every k");
struct SplitPlan {
  int chunks, segments;  // segments 0: one workgroup per row (sample_kernel)
};

SplitPlan split_plan(int64_t rows, int64_t vocab) {
  const int64_t total = (vocab + kChunk - 1) / kChunk;
  int chunks = 1;
  if (rows > 1024 || total < kMinSegments) return {0, 0};
  auto count = [&](int c) { return (total + c - 1) / c; };
  while (chunks < kMaxChunks &&
         ((rows * count(2 * chunks) >= 1024 && count(2 * chunks) >= kMinSegments) ||
          count(chunks) > kMaxSegments))
    chunks *= 2;
  const int64_t segments = count(chunks);
  if (segments > kMaxSegments) return {0, 0};
  return {chunks, static_cast<int>(segments)};
}

template <int DT, bool VEC>
void launch_segments(const SampleArgs& a, const SplitArgs& p, int chunks, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>(p.segments), static_cast<uint32_t>(a.rows));
  const dim3 block(kSegThreads);
  switch (chunks) {
    case 1: sample_segments<DT, 1, VEC><<<grid, block, 0, s>>>(a, p); break;
    case 2: sample_segments<DT, 2, VEC><<<grid, block, 0, s>>>(a, p); break;
    default: sample_segments<DT, kMaxChunks, VEC><<<grid, block, 0, s>>>(a, p); break;
  }
  if (p.top_p_rows) {
    mass_level<DT, 0, VEC><<<grid, block, 0, s>>>(a, p, chunks);
    mass_level<DT, 1, VEC><<<grid, block, 0, s>>>(a, p, chunks);
    if constexpr (kLevels<DT> > 2) mass_level<DT, 2, VEC><<<grid, block, 0, s>>>(a, p, chunks);
    race_segments<DT, VEC><<<grid, block, 0, s>>>(a, p, chunks);
  }
}

template <int DT>
void launch_split(const SampleArgs& a, const SplitArgs& p, int chunks, hipStream_t s) {
  if (p.vec && a.vocab % 8 == 0)
    launch_segments<DT, true>(a, p, chunks, s);
  else
    launch_segments<DT, false>(a, p, chunks, s);
  sample_finish<DT><<<dim3(static_cast<uint32_t>(a.rows)), dim3(kThreads), 0, s>>>(a, p);
}

int64_t round256(int64_t n) { return (n + 255) / 256 * 256; }

// Checks shared by the two entries; fills the arguments. `done`: nothing to launch.
const char* sample_args(const void* logits, int64_t rows, int64_t vocab, int64_t row_stride,
                        int dtype, const float* temperature, const int32_t* top_k,
                        const float* top_p, uint64_t seed, uint64_t offset, int64_t* out,
                        SampleArgs* a, bool* vec, bool* done) {
  *done = false;
  if (rows < 0 || vocab <= 0 || row_stride < vocab) return set_error("mi355x_sample: bad shape");
  if (vocab >= (int64_t(1) << 32) || rows >= (int64_t(1) << 31))
    return set_error("mi355x_sample: shape too large");
  if (dtype < 0 || dtype > 2)
    return set_error("mi355x_sample: dtype must be 0 (bf16), 1 (fp16) or 2 (fp32)");
  if (rows == 0) {
    *done = true;
    return nullptr;
  }
  if (!logits || !temperature || !top_k || !top_p || !out)
    return set_error("mi355x_sample: null pointer");
  a->logits = logits;
  a->rows = rows;
  a->vocab = vocab;
  a->stride = row_stride;
  a->temperature = temperature;
  a->top_k = top_k;
  a->top_p = top_p;
  a->seed_lo = static_cast<uint32_t>(seed);
  a->seed_hi = static_cast<uint32_t>(seed >> 32);
  a->offset_lo = static_cast<uint32_t>(offset);
  a->offset_hi = static_cast<uint32_t>(offset >> 32);
  a->out = out;
  const int per_vec = dtype == 2 ? 4 : 8;
  *vec = aligned(logits, 16) && row_stride % per_vec == 0;
  return nullptr;
}

}  // namespace
}  // namespace mi355x

using namespace mi355x;

extern "C" const char* mi355x_sample(const void* logits, int64_t rows, int64_t vocab,
                                     int64_t row_stride, int dtype, const float* temperature,
                                     const int32_t* top_k, const float* top_p, uint64_t seed,
                                     uint64_t offset, int64_t* out, void* stream) {
  SampleArgs a{};
  bool vec = false, done = false;
  if (const char* e = sample_args(logits, rows, vocab, row_stride, dtype, temperature, top_k,
                                  top_p, seed, offset, out, &a, &vec, &done))
    return e;
  if (done) return nullptr;
  auto s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<uint32_t>(rows));
  if (dtype == 0)
    sample_kernel<0><<<grid, dim3(kThreads), 0, s>>>(a, vec);
  else if (dtype == 1)
    sample_kernel<1><<<grid, dim3(kThreads), 0, s>>>(a, vec);
  else
    sample_kernel<2><<<grid, dim3(kThreads), 0, s>>>(a, vec);
  return launch_status("mi355x_sample");
}

extern "C" int64_t mi355x_sample_workspace_bytes(int64_t rows, int64_t vocab, bool top_p_rows) {
  if (rows <= 0 || vocab <= 0 || vocab >= (int64_t(1) << 32)) return 0;
  const int64_t n = rows * split_plan(rows, vocab).segments;
  if (n == 0) return 0;
  return round256(n * int64_t(sizeof(Segment))) + n * kSegPeaks * 4 +
         n * kSegList * int64_t(sizeof(uint2)) + round256(rows * 4 * int64_t(sizeof(LevelState))) +
         (top_p_rows ? rows * kHistWords * 8 : 0);
}

extern "C" const char* mi355x_sample_split(const void* logits, int64_t rows, int64_t vocab,
                                           int64_t row_stride, int dtype,
                                           const float* temperature, const int32_t* top_k,
                                           const float* top_p, uint64_t seed, uint64_t offset,
                                           int64_t* out, bool top_p_rows, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
  SampleArgs a{};
  bool vec = false, done = false;
  if (const char* e = sample_args(logits, rows, vocab, row_stride, dtype, temperature, top_k,
                                  top_p, seed, offset, out, &a, &vec, &done))
    return e;
  if (done) return nullptr;
  const SplitPlan plan = split_plan(rows, vocab);
  if (plan.segments == 0) return set_error("mi355x_sample_split: shape not split");
  if (!workspace || !aligned(workspace, 16) ||
      workspace_bytes < mi355x_sample_workspace_bytes(rows, vocab, top_p_rows))
    return set_error("mi355x_sample_split: workspace too small");
  SplitArgs p{};
  const int64_t n = rows * plan.segments;
  auto* base = static_cast<uint8_t*>(workspace);
  p.seg = reinterpret_cast<Segment*>(base);
  base += round256(n * int64_t(sizeof(Segment)));
  p.peak = reinterpret_cast<float*>(base);
  base += n * kSegPeaks * 4;
  p.list = reinterpret_cast<uint2*>(base);
  base += n * kSegList * int64_t(sizeof(uint2));
  p.state = reinterpret_cast<LevelState*>(base);
  base += round256(rows * 4 * int64_t(sizeof(LevelState)));
  p.hist = reinterpret_cast<unsigned long long*>(base);
  p.segments = plan.segments;
  p.vec = vec;
  p.top_p_rows = top_p_rows;
  auto s = static_cast<hipStream_t>(stream);
  if (dtype == 0)
    launch_split<0>(a, p, plan.chunks, s);
  else if (dtype == 1)
    launch_split<1>(a, p, plan.chunks, s);
  else
    launch_split<2>(a, p, plan.chunks, s);
  return launch_status("mi355x_sample_split");
}
