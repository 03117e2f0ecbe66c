// The reference sampler on the device: Sampler.next (engine/sampler.py:76-108) over rows of logits.
//
// The steps and their float32 operations are the reference's, in its order: presence penalty on the raw logits
// (:80-82), argmax at temperature <= 0 (:83-84), division by the temperature (:85), the top-k threshold (:86-88),
// softmax (:89, :67-69), top-p (:90-97), min-p (:98-100) and the inverse-CDF draw with the caller's uniform
// (:101-108). The parameters arrive sanitized (SampleParams.sanitized, :45-64) and the uniforms from the sampler's
// splitmix64 stream, both on the host. The order of every sum is defined here (the reference's comes from numpy):
//   * z, the top-p mass and the final total are hierarchical sums: a sub-chunk of 16 entries summed sequentially
//     from 0, the 64 sub-chunk totals of a 1024-entry chunk by the xor butterfly, the chunk totals sequentially;
//   * top-p ranks entry j by rho_j = key(p_j) << 20 | (2^20 - 1 - j) (probability descending, index ascending:
//     the stable argsort of :91); cum(rho) = hierarchical sum of p_i over rho_i > rho; j is kept iff
//     cum(rho_j) < top_p. cum falls as rho grows, so the kept set is rho_j >= r* for the smallest r* with
//     cum(r*) < top_p, found 4 bits at a time from the top (13 rounds, 16 candidates each);
//   * the draw takes the first entry whose hierarchical running sum reaches u * total (u == 0: exceeds 0),
//     chunk, then sub-chunk, then entry, each level falling back to the last nonzero one.
// exp is ss_expf. A total that is not finite and > 0 falls back to the argmax of the raw logits (:105-106).
// Entries below the top-k threshold get weight exactly 0 (exp(-inf - m) = 0 for finite m; when m is not finite the
// total is NaN whatever the masked weights are, and the draw takes the fallback).
//
// Every launch covers R rows at once (blockIdx.y). Accept mode is the sampled verify round of _mtp_decode
// (engine/generate.py:208-229) over D+1 rows: row i is reached only if rows 0..i-1 drew their drafts, so its
// penalty set is seen + drafts[0..i) and all rows are drawn together; their last row, or a last kernel, walks them in
// order (a non-finite row ends the round without a draw, :210-212; the round goes on while the token equals the
// draft). The launch sequence depends only on the parameters, so it can be captured in a graph: three launches for
// rows with a top-k of at most 512 (below), one launch per step otherwise.
#include <type_traits>

#include "ss_common.hpp"
#include "ss_launch.hpp"

namespace ss {

namespace {

constexpr int kSub = 16;
constexpr int kChunk = 64 * kSub;
constexpr int kPerLane = 16;  // chunk arrays of up to 1024 chunks (V <= 2^20)
constexpr int kRhoBits = 52;  // 32 key bits above 20 index bits
constexpr int kRounds = kRhoBits / 4;
constexpr int kFlagNonfinite = 1, kFlagBadDraft = 2, kFlagFallback = 8;
constexpr int kKeys = 2048;  // group keys of a top-k row, at most
// Candidates a chunk of a top-k row lists: all of it in rows of up to 64 chunks, 512 beyond.
__host__ __device__ constexpr int slots_of(int nch) { return nch <= 64 ? 1024 : 512; }
constexpr int kHistShards = 8;  // copies of each top-k histogram; chunk c adds to copy c % 8 (fewer atomics per bin)

SS_DEV bool is_nan(float v) { return v != v; }
SS_DEV bool is_finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

// NaN-largest order-preserving key with -0 == +0 (the order np.sort gives :87).
SS_DEV uint32_t nkey(float v) { return is_nan(v) ? 0xFFFFFFFFu : ss_key(v == 0.f ? 0.f : v); }

SS_DEV uint64_t rho_of(float p, int j) {
  return ((uint64_t)ss_key(p) << 20) | (uint64_t)((1u << 20) - 1u - (uint32_t)j);
}

// argmax key: the first maximum, NaN counting as the largest (np.argmax).
SS_DEV uint64_t amax_key(float v, int j) { return ((uint64_t)nkey(v) << 32) | (0xFFFFFFFFu - (uint32_t)j); }

// Byte offsets of one row's workspace; rows follow each other `bytes` apart.
struct Layout {
  size_t L, P, cmax, cnan, ckey, craw, cbad, etot, ftot, tsum, stot, hist, rr, res, cnz, cand, gkey, done, bytes;
};

__host__ __device__ inline Layout layout_of(int V, int nch) {
  Layout l{};
  size_t o = 0;
  auto take = [&o](size_t b) {
    const size_t p = o;
    o += (b + 255) & ~(size_t)255;
    return p;
  };
  l.L = take((size_t)V * 4);                // logits after penalty and temperature
  l.P = take((size_t)V * 4);                // exp, then probabilities, then the final weights
  l.cmax = take((size_t)nch * 4);           // chunk maxima of the logits, later of the kept probabilities
  l.cnan = take((size_t)nch * 4);
  l.ckey = take((size_t)nch * 8);           // argmax keys of the penalized logits
  l.craw = take((size_t)nch * 8);           // argmax keys of the raw logits
  l.cbad = take((size_t)nch * 4);           // chunk holds a non-finite raw logit
  l.etot = take((size_t)nch * 4);           // chunk totals of exp
  l.ftot = take((size_t)nch * 4);           // chunk totals of the final weights
  l.tsum = take((size_t)2 * 16 * nch * 4);  // top-p candidate masses, two rounds alternating
  l.stot = take((size_t)64 * nch * 4);      // sub-chunk totals of the final weights
  l.hist = take(4 * kHistShards * 256 * 4);  // top-k radix histograms, one per 8-bit pass, kHistShards copies
  l.rr = take((size_t)(kRounds + 1) * 8);   // top-p prefix at the start of each round
  l.res = take(16);                         // token, fallback flag, non-finite row
  l.cnz = take((size_t)nch * 4);            // candidates per chunk (top-k rows)
  l.cand = take((size_t)nch * slots_of(nch) * 8);  // a chunk's candidates (index << 32 | logit bits)
  l.gkey = take((size_t)kKeys * 4);         // largest key of each group of the row (top-k rows)
  l.done = take(4);                         // accept mode: rows drawn (row 0's word)
  l.bytes = o;
  return l;
}

struct SW {
  float *L, *P, *cmax;
  int* cnan;
  uint64_t *ckey, *craw;
  int* cbad;
  float *etot, *ftot, *tsum, *stot;
  int* hist;
  uint64_t* rr;
  int* res;
  int* cnz;
  uint64_t* cand;
  uint32_t* gkey;
  int* done;
};

SS_DEV SW sw_of(void* work, int V, int nch, int row) {
  const Layout l = layout_of(V, nch);
  uint8_t* b = static_cast<uint8_t*>(work) + (size_t)row * l.bytes;
  SW s;
  s.L = reinterpret_cast<float*>(b + l.L);
  s.P = reinterpret_cast<float*>(b + l.P);
  s.cmax = reinterpret_cast<float*>(b + l.cmax);
  s.cnan = reinterpret_cast<int*>(b + l.cnan);
  s.ckey = reinterpret_cast<uint64_t*>(b + l.ckey);
  s.craw = reinterpret_cast<uint64_t*>(b + l.craw);
  s.cbad = reinterpret_cast<int*>(b + l.cbad);
  s.etot = reinterpret_cast<float*>(b + l.etot);
  s.ftot = reinterpret_cast<float*>(b + l.ftot);
  s.tsum = reinterpret_cast<float*>(b + l.tsum);
  s.stot = reinterpret_cast<float*>(b + l.stot);
  s.hist = reinterpret_cast<int*>(b + l.hist);
  s.rr = reinterpret_cast<uint64_t*>(b + l.rr);
  s.res = reinterpret_cast<int*>(b + l.res);
  s.cnz = reinterpret_cast<int*>(b + l.cnz);
  s.cand = reinterpret_cast<uint64_t*>(b + l.cand);
  s.gkey = reinterpret_cast<uint32_t*>(b + l.gkey);
  s.done = reinterpret_cast<int*>(b + l.done);
  return s;
}

struct SampArgs {
  const float* x;  // [R, V]
  int V, nch, R;
  const int32_t* gen;  // sorted penalty set
  int n_gen;
  const int32_t* drafts;  // accept mode: [R - 1]; row i also penalizes drafts[0..i)
  float temperature, top_p, min_p, pp;
  int top_k;
  const float* u;  // [R]
  int32_t* out;    // single row: [2] (token, flags); accept mode: [R + 4]
  int accept;
  void* work;
};

SS_DEV bool in_sorted(const int32_t* g, int n, int j) {
  int lo = 0, hi = n - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const int v = g[mid];
    if (v == j) return true;
    if (v < j) lo = mid + 1;
    else hi = mid - 1;
  }
  return false;
}

SS_DEV bool penalized(const SampArgs& a, int row, int j) {
  if (a.pp == 0.f) return false;
  if (a.n_gen > 0 && in_sorted(a.gen, a.n_gen, j)) return true;
  for (int k = 0; k < row; ++k)
    if (a.drafts[k] == j) return true;
  return false;
}

// Chunk c's hierarchical total of the lane values v[i] (entries c*1024 + 16*lane + i): sequential per lane, then
// the butterfly; `sub` receives the lane's sub-chunk total.
SS_DEV float chunk_sum(const float (&v)[kSub], float& sub) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kSub; ++i) s = s + v[i];
  sub = s;
  return ss_wave_sum(s);
}

// Stages a chunk array [n <= 1024] in LDS for the sequential scans below (one wave, every lane), zero-padded to a
// multiple of 16 entries (16-byte aligned).
SS_DEV const float* stage(const float* a, int n) {
  __shared__ __attribute__((aligned(16))) float buf[kPerLane * 64];
  const int lane = threadIdx.x & 63;
  float v[kPerLane];
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) v[k] = lane + 64 * k < n ? a[lane + 64 * k] : 0.f;
#pragma unroll
  for (int k = 0; k < kPerLane; ++k)
    if (lane + 64 * k < ((n + 15) & ~15)) buf[lane + 64 * k] = v[k];
  __syncthreads();
  return buf;
}

// ((s + b[0]) + b[1]) + ... + b[n-1] over a zero-padded, 16-byte aligned LDS array: 16 entries read as four
// unconditional 16-byte loads before their in-order adds, the bound applied by selects in the last, partial group.
SS_DEV float lds_seq_sum(const float* b, int n, float s) {
  // whole groups of 16 add without a bound check; only the last, partial group selects
  const float4* b4 = reinterpret_cast<const float4*>(b);
  for (int q = 0; q < n; q += 16) {
    const float4 a0 = b4[q / 4], a1 = b4[q / 4 + 1], a2 = b4[q / 4 + 2], a3 = b4[q / 4 + 3];
    const float t[16] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w,
                         a2.x, a2.y, a2.z, a2.w, a3.x, a3.y, a3.z, a3.w};
    if (q + 16 <= n) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s = s + t[i];
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float nx = s + t[i];
        s = q + i < n ? nx : s;
      }
    }
  }
  return s;
}

// Every lane: ((a[0] + a[1]) + ...) + a[n-1] of a chunk array.
SS_DEV float seq_sum(const float* a, int n) { return lds_seq_sum(stage(a, n), n, 0.f); }

SS_DEV uint64_t max_u64_of(const uint64_t* a, int n) {
  const int lane = threadIdx.x & 63;
  uint64_t m = 0;
#pragma unroll
  for (int k = 0; k < kPerLane; ++k)
    if (lane + 64 * k < n) m = a[lane + 64 * k] > m ? a[lane + 64 * k] : m;
  return ss_wave_max_u64(m);
}

// Every lane: the logits' maximum over the chunk maxima (NaN when any chunk holds a NaN, as numpy's max).
SS_DEV float row_max(const SW& w, int nch) {
  const int lane = threadIdx.x & 63;
  float m = -__builtin_inff();
  uint32_t nan = 0;
#pragma unroll
  for (int k = 0; k < kPerLane; ++k) {
    const int q = lane + 64 * k;
    if (q < nch) {
      m = fmaxf(m, w.cmax[q]);
      nan |= (uint32_t)w.cnan[q];
    }
  }
  m = ss_wave_max(m);
  return ss_wave_or(nan) ? __uint_as_float(0x7FC00000u) : m;
}

// One 8-bit radix step of the top-k select, whole wave: the bin of the need-th largest key among those counted in
// `hist` (bins descending, counting multiplicity); need becomes its rank inside the bin. Every lane gets the same.
template <int SH = kHistShards>
SS_DEV void select_pass(const int* hist, int& need, uint32_t& prefix, int shift) {
  const int lane = threadIdx.x & 63;
  int hs[SH][4];
#pragma unroll
  for (int c = 0; c < SH; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) hs[c][q] = hist[256 * c + 255 - 4 * lane - q];
  int h[4], s = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    h[q] = 0;
#pragma unroll
    for (int c = 0; c < SH; ++c) h[q] += hs[c][q];
    s += h[q];
  }
  int incl = s;  // inclusive prefix over lanes = count of keys in bins >= 252 - 4 * lane
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  const int above = incl - s;
  const bool mine = above < need && need <= incl;
  const uint64_t bal = __ballot(mine);
  const int src = bal ? (int)__builtin_ctzll(bal) : 0;
  int b = 0, nn = need - above;
  if (mine) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (h[q] >= nn) {
        b = 255 - 4 * lane - q;
        break;
      }
      nn -= h[q];
    }
  }
  b = __shfl(b, src);
  nn = __shfl(nn, src);
  need = nn;
  prefix |= (uint32_t)b << shift;
}

// One wave: the 4-bit top-p digit of a round from its candidate masses (lane d sums candidate d's chunk totals in
// chunk order): the smallest d whose mass is below top_p (candidate 15 always is: it is the previous round's bound).
// All lanes stage the masses in LDS first, so the loads are in flight together.
// The 16 candidate rows go to dynamic LDS (topp_lds_bytes(nch) at launch) at a zero-padded stride, so a launch
// holds only what its vocabulary needs.
SS_DEV int topp_digit(const float* tsum, int nch, float top_p) {
  constexpr int B = 32;
  extern __shared__ float4 topp_dyn[];
  float* tb = reinterpret_cast<float*>(topp_dyn);
  const int lane = threadIdx.x & 63;
  const int nchp = (nch + 15) & ~15;
  const int n = 16 * nch;
  for (int i = lane; i < 16 * nchp; i += 64) tb[i] = 0.f;
  for (int i0 = 0; i0 < n; i0 += 64 * B) {
    float v[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int idx = i0 + 64 * q + lane;
      v[q] = idx < n ? tsum[idx] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int idx = i0 + 64 * q + lane;
      if (idx < n) {
        const int d = idx / nch;
        tb[d * nchp + (idx - d * nch)] = v[q];
      }
    }
  }
  __syncthreads();
  const float cum = lds_seq_sum(tb + (lane & 15) * nchp, nch, 0.f);
  const uint64_t ok = __ballot(lane < 16 && cum < top_p);
  return ok ? (int)__builtin_ctzll(ok) : 15;
}

}  // namespace

// Clears the top-k histograms of every row.
__global__ __launch_bounds__(256) void samp_begin_kernel(SampArgs a) {
  SW w = sw_of(a.work, a.V, a.nch, blockIdx.x);
  for (int i = threadIdx.x; i < 4 * kHistShards * 256; i += 256) w.hist[i] = 0;
}

// 1. penalty and temperature into L; argmax keys of the penalized and of the raw logits; non-finite flags; chunk
// maxima; (has_k) the first top-k histogram (top 8 key bits).
__global__ __launch_bounds__(64) void samp_prep_kernel(SampArgs a, int has_k) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  const float* x = a.x + (size_t)row * a.V;
  __shared__ int hist[256];
  if (has_k) {
    for (int i = lane; i < 256; i += 64) hist[i] = 0;
    __syncthreads();
  }
  float xv[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    xv[i] = j < a.V ? x[j] : 0.f;
  }
  const bool sampled = a.temperature > 0.f;
  uint64_t kp = 0, kr = 0;
  uint32_t bad = 0, nan = 0;
  float m = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    if (j < a.V) {
      const float xx = xv[i];
      bad |= !is_finite(xx);
      float l = penalized(a, row, j) ? xx - a.pp : xx;
      const uint64_t k1 = amax_key(l, j), k2 = amax_key(xx, j);
      kp = k1 > kp ? k1 : kp;
      kr = k2 > kr ? k2 : kr;
      if (sampled) {
        l = l / a.temperature;
        w.L[j] = l;
        m = fmaxf(m, l);
        nan |= is_nan(l);
        if (has_k) atomicAdd(&hist[nkey(l) >> 24], 1);  // integer counts: order-free
      }
    }
  }
  kp = ss_wave_max_u64(kp);
  kr = ss_wave_max_u64(kr);
  bad = ss_wave_or(bad);
  nan = ss_wave_or(nan);
  m = ss_wave_max(m);
  if (lane == 0) {
    w.ckey[c] = kp;
    w.craw[c] = kr;
    w.cbad[c] = (int)bad;
    w.cmax[c] = m;
    w.cnan[c] = (int)nan;
  }
  if (has_k) {
    __syncthreads();
    for (int b = lane; b < 256; b += 64)
      if (hist[b]) atomicAdd(&w.hist[256 * (c % kHistShards) + b], hist[b]);
  }
}

// 2. top-k histogram pass 1..3: keys matching the prefix the earlier passes selected, next 8 bits.
__global__ __launch_bounds__(64) void samp_hist_kernel(SampArgs a, int pass) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  __shared__ int hist[256];
  for (int i = lane; i < 256; i += 64) hist[i] = 0;
  int need = a.top_k;
  uint32_t prefix = 0;
  for (int p = 0; p < pass; ++p) select_pass(w.hist + kHistShards * 256 * p, need, prefix, 24 - 8 * p);
  const int shift = 24 - 8 * pass;
  const uint32_t hmask = 0xFFFFFFFFu << (shift + 8);
  float lv[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    lv[i] = j < a.V ? w.L[j] : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    const uint32_t k = nkey(lv[i]);
    if (j < a.V && (k & hmask) == prefix) atomicAdd(&hist[(k >> shift) & 255], 1);
  }
  __syncthreads();
  for (int b = lane; b < 256; b += 64)
    if (hist[b]) atomicAdd(&w.hist[kHistShards * 256 * pass + 256 * (c % kHistShards) + b], hist[b]);
}

// 3. e = exp(l - m) into P (0 below the top-k threshold) and the chunk totals.
__global__ __launch_bounds__(64) void samp_exp_kernel(SampArgs a, int has_k) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  float kth = -__builtin_inff();
  if (has_k) {
    int need = a.top_k;
    uint32_t prefix = 0;
    for (int p = 0; p < 4; ++p) select_pass(w.hist + kHistShards * 256 * p, need, prefix, 24 - 8 * p);
    kth = prefix == 0xFFFFFFFFu ? __uint_as_float(0x7FC00000u) : ss_unkey(prefix);
  }
  const float m = row_max(w, a.nch);
  float v[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    const float l = j < a.V ? w.L[j] : 0.f;
    v[i] = j < a.V ? (l < kth ? 0.f : ss_expf(l - m)) : 0.f;
    if (j < a.V) w.P[j] = v[i];
  }
  float sub;
  const float t = chunk_sum(v, sub);
  if (lane == 0) w.etot[c] = t;
}

// 4. top-p round k: fold the previous round's digit into the prefix r, then chunk c's hierarchical masses of p over
// rho > r | d << s | (2^s - 1), d = 0..15. Round 0 also normalizes p = e / z.
__global__ __launch_bounds__(64) void samp_topp_kernel(SampArgs a, int round) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  const int nch = a.nch;
  const int s = kRhoBits - 4 - 4 * round;
  float pv[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    pv[i] = j < a.V ? w.P[j] : 0.f;
  }
  uint64_t r = 0;
  if (round > 0)
    r = w.rr[round - 1] | ((uint64_t)topp_digit(w.tsum + ((round - 1) & 1) * 16 * nch, nch, a.top_p) << (s + 4));
  if (c == 0 && lane == 0) w.rr[round] = r;
  if (round == 0) {
    const float z = seq_sum(w.etot, nch);
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      const int j = c * kChunk + lane * kSub + i;
      pv[i] = pv[i] / z;
      if (j < a.V) w.P[j] = pv[i];
    }
  }
  // rho > r | d << s | (2^s - 1) holds for every d when rho is above r in the bits over the round's digit, and for
  // d < t when those bits equal r's and t is rho's digit; p = 0 adds nothing, so zero entries are skipped.
  const uint64_t r_hi = r >> (s + 4);
  float acc[16];
#pragma unroll
  for (int d = 0; d < 16; ++d) acc[d] = 0.f;
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    const float p = pv[i];
    if (j < a.V && p != 0.f) {
      const uint64_t rho = rho_of(p, j);
      const uint64_t hi = rho >> (s + 4);
      const int lim = hi > r_hi ? 16 : (hi == r_hi ? (int)((rho >> s) & 15) : 0);
#pragma unroll
      for (int d = 0; d < 16; ++d) acc[d] = acc[d] + (d < lim ? p : 0.f);
    }
  }
  float* out = w.tsum + (round & 1) * 16 * nch;
#pragma unroll
  for (int d = 0; d < 16; ++d) {
    const float t = ss_wave_sum(acc[d]);
    if (lane == 0) out[d * nch + c] = t;
  }
}

// 5. (has_p) keep rho >= r*; (min_p > 0) chunk maxima of the kept probabilities. `norm`: p = e / z here.
__global__ __launch_bounds__(64) void samp_keep_kernel(SampArgs a, int has_p, int norm) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  const int nch = a.nch;
  float pv[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    pv[i] = j < a.V ? w.P[j] : 0.f;
  }
  uint64_t r = 0;
  if (has_p) {
    r = w.rr[kRounds - 1] | (uint64_t)topp_digit(w.tsum + ((kRounds - 1) & 1) * 16 * nch, nch, a.top_p);
  }
  const float z = norm ? seq_sum(w.etot, nch) : 1.f;
  float m = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    if (j < a.V) {
      float p = norm ? pv[i] / z : pv[i];
      const bool drop = has_p && !(rho_of(p, j) >= r);
      if (drop) p = 0.f;
      if (drop || norm) w.P[j] = p;
      m = fmaxf(m, p);
    }
  }
  m = ss_wave_max(m);
  if (lane == 0) w.cmax[c] = m;
}

// 6. min-p cutoff (has_minp) and the hierarchical totals of the final weights. `norm`: p = e / z here.
__global__ __launch_bounds__(64) void samp_total_kernel(SampArgs a, int has_minp, int norm) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  float cutoff = 0.f;
  if (has_minp) {
    float pm = -__builtin_inff();
#pragma unroll
    for (int k = 0; k < kPerLane; ++k)
      if (lane + 64 * k < a.nch) pm = fmaxf(pm, w.cmax[lane + 64 * k]);
    cutoff = ss_wave_max(pm) * a.min_p;
  }
  const float z = norm ? seq_sum(w.etot, a.nch) : 1.f;
  float v[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    v[i] = j < a.V ? w.P[j] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = c * kChunk + lane * kSub + i;
    float p = norm ? v[i] / z : v[i];
    const bool drop = has_minp && p < cutoff;
    if (drop) p = 0.f;
    if (j < a.V && (drop || norm)) w.P[j] = p;
    v[i] = j < a.V ? p : 0.f;
  }
  float sub;
  const float t = chunk_sum(v, sub);
  w.stot[c * 64 + lane] = sub;
  if (lane == 0) w.ftot[c] = t;
}

// The inverse-CDF descent over the final weights, whole wave (every lane follows the same scan): chunk totals ct in LDS
// (zero-padded to a multiple of 16), their sum `total`, sub-chunk totals stot[64 nch], weights P[V] -> the token.
static SS_DEV int draw_descent(float u, float total, const float* ct, int nch, const float* stot, const float* P, int V) {
  const int lane = threadIdx.x & 63;
  const bool ge = u != 0.f;
  const float target = ge ? u * total : 0.f;
  auto hit = [&](float x) { return ge ? x >= target : x > target; };
  // The first chunk whose running total hits the target is the count of leading misses: the zero padding adds +0
  // and, following a miss with the same total, cannot be the first hit, so no bound check runs per entry.
  int lead = 0, clast = -1;
  bool alive = true;
  float base = 0.f, run = 0.f;
  const float4* c4 = reinterpret_cast<const float4*>(ct);
  for (int q0 = 0; q0 < nch; q0 += 16) {  // 16 unconditional reads (the padding is zero), then the in-order scan
    const float4 a0 = c4[q0 / 4], a1 = c4[q0 / 4 + 1], a2 = c4[q0 / 4 + 2], a3 = c4[q0 / 4 + 3];
    const float t[16] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w,
                         a2.x, a2.y, a2.z, a2.w, a3.x, a3.y, a3.z, a3.w};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float nx = run + t[i];
      alive = alive && !hit(nx);
      base = alive ? nx : base;
      lead += alive ? 1 : 0;
      clast = t[i] > 0.f ? q0 + i : clast;
      run = nx;
    }
  }
  int cs = lead < nch ? lead : -1;
  if (cs < 0) {
    cs = clast < 0 ? 0 : clast;
    base = lds_seq_sum(ct, cs, 0.f);
  }
  const float st = stot[cs * 64 + lane];
  int slead = 0, blast = -1;
  float sbase = base;
  run = base;
  alive = true;
#pragma unroll 16
  for (int b = 0; b < 64; ++b) {
    const float t = ss_readlane_f(st, b);
    const float nx = run + t;
    blast = t > 0.f ? b : blast;
    alive = alive && !hit(nx);
    sbase = alive ? nx : sbase;
    slead += alive ? 1 : 0;
    run = nx;
  }
  int bs = slead < 64 ? slead : -1;
  if (bs < 0) {
    bs = blast < 0 ? 0 : blast;
    sbase = base;
    for (int b = 0; b < bs; ++b) sbase = sbase + ss_readlane_f(st, b);
  }
  const int j0 = cs * kChunk + bs * kSub;
  const int jl = j0 + (lane & (kSub - 1));
  const float val = jl < V ? P[jl] : 0.f;
  int pick = -1, last = -1;
  run = sbase;
  for (int i = 0; i < kSub; ++i) {
    const int j = j0 + i;
    if (j >= V) break;
    const float e = ss_readlane_f(val, i);
    if (e > 0.f) last = j;
    run = run + e;
    if (hit(run)) {
      pick = j;
      break;
    }
  }
  if (pick < 0) pick = last >= 0 ? last : (j0 < V ? j0 : V - 1);
  return pick;
}

// 7. the draw, one wave per row (every lane follows the same scan); greedy rows take the argmax.
__global__ __launch_bounds__(64) void samp_draw_kernel(SampArgs a) {
  const int row = blockIdx.x, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  const int nch = a.nch;
  auto finish = [&](int tok, int fb, int nonfinite) {
    if (lane != 0) return;
    if (a.accept) {
      w.res[0] = tok;
      w.res[1] = fb;
      w.res[2] = nonfinite;
    } else {
      a.out[0] = tok;
      a.out[1] = fb;
    }
  };
  if (a.accept) {
    uint32_t b = 0;
#pragma unroll
    for (int k = 0; k < kPerLane; ++k)
      if (lane + 64 * k < nch) b |= (uint32_t)w.cbad[lane + 64 * k];
    if (ss_wave_or(b)) {
      finish(-1, 0, 1);
      return;
    }
  }
  if (!(a.temperature > 0.f)) {
    const uint64_t k = max_u64_of(w.ckey, nch);
    finish((int)(0xFFFFFFFFu - (uint32_t)k), 0, 0);
    return;
  }
  const float* ct = stage(w.ftot, nch);  // zero-padded to a multiple of 16
  const float total = lds_seq_sum(ct, nch, 0.f);
  if (!is_finite(total) || !(total > 0.f)) {
    const uint64_t k = max_u64_of(w.craw, nch);
    finish((int)(0xFFFFFFFFu - (uint32_t)k), 1, 0);
    return;
  }
  finish(draw_descent(a.u[row], total, ct, nch, w.stot, w.P, a.V), 0, 0);
}

// ---------------------------------------------------------------- top-k rows in three launches
// A row with 0 < top_k <= kTopkMax (and top_k < V) carries weight on its top-k survivors only, so after the k-th largest
// logit is known everything else is work on a few dozen values, done by one workgroup per row in LDS:
//   1. samp_scan_kernel, one wave per 1024-entry chunk: raw argmax, non-finite flag, chunk maximum, and the largest key
//      of each of G groups of the chunk (a power of two, up to one entry a group: the smallest that gives 2 k groups);
//   2. samp_cand_kernel, one wave per chunk: tau, the largest threshold with zero low 16 bits that at least k group
//      maxima reach, bounds the k-th largest entry from below; the chunk's entries >= tau whose exp is not 0 are listed
//      in index order (an entry with exp 0 carries no weight, and when fewer than k entries carry weight all of them
//      survive, whatever the k-th is);
//   3. samp_topk_draw_kernel, one workgroup per row: the exact k-th by ranks, exp, z, top-p, min-p and the draw.
// The operations and sums are those of the launches below (or_sample's): sums over zeros change no bit of a
// non-negative sum, so a chunk total is the butterfly over its nonzero leaves and chunks without survivors drop out.
// More than kCand candidates, a chunk's slots or kSurv survivors (ties at the threshold) take the whole sequence inside the
// workgroup. Latency bound. Three rows over 248,320 tokens at the default parameters (top-k 40, top-p 0.95): 32 us per
// round (5 + 7 + 21 in the kernels); eleven launches (four radix passes over the row, exp, a top-p search in one
// workgroup, keep, totals, draw, accept walk) took 106.
// k from 40 to 512 (one row of normal logits, us, the eleven launches / these three): V 1000 64-132 / 38-85, 5000 67-120 /
// 29-51, 32,000 73-126 / 29-50, 60,000 73-139 / 29-55, 248,320 91-3094 / 28-81. Of that, against groups of 16 entries or
// more and sums by one wave: at most 16 groups a chunk left small rows without a bound (every entry listed, the lists
// overflowed, the whole sequence in one workgroup: k 512 at V 32,000 339), and one wave walked the chunks with several
// survivors one by one (k 400 at V 60,000 241, now 53). A flat row of 248,320: 3.2 ms (4.5).
constexpr int kTopkMax = 512;
constexpr int kCand = 2048, kSurv = 1024;
constexpr int kRankMax = 256;  // longest list whose k-th key is found by ranks

SS_DEV float logit_of(const SampArgs& a, const float* x, int row, int j) {
  const float xx = x[j];
  return (penalized(a, row, j) ? xx - a.pp : xx) / a.temperature;
}

// The chunk's 16 entries of this lane; 16-byte loads where every row is 16-byte aligned (`vec`).
SS_DEV void load_chunk(const float* x, int j0, int V, bool vec, float (&v)[kSub]) {
  if (vec && j0 + kSub <= V) {
#pragma unroll
    for (int q = 0; q < kSub / 4; ++q) {
      const uint4 t = ldg16(x + j0 + 4 * q);
      v[4 * q] = __uint_as_float(t.x);
      v[4 * q + 1] = __uint_as_float(t.y);
      v[4 * q + 2] = __uint_as_float(t.z);
      v[4 * q + 3] = __uint_as_float(t.w);
    }
  } else {
#pragma unroll
    for (int i = 0; i < kSub; ++i) v[i] = j0 + i < V ? x[j0 + i] : 0.f;
  }
}

SS_DEV float unkey_nan(uint32_t k) { return k == 0xFFFFFFFFu ? __uint_as_float(0x7FC00000u) : ss_unkey(k); }

__global__ __launch_bounds__(64) void samp_scan_kernel(SampArgs a, int groups, int vec) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  SW w = sw_of(a.work, a.V, a.nch, row);
  const int j0 = c * kChunk + lane * kSub;
  float xv[kSub];
  load_chunk(a.x + (size_t)row * a.V, j0, a.V, vec != 0, xv);
  // the first maximum of the raw logits, and the largest key after the penalty (the temperature is applied to the
  // maxima: division by it is monotone, so the maximum of the quotients is the quotient of the maximum)
  uint32_t br = 0, bp = 0, bad = 0, ek[kSub];  // ek: each entry's key after the penalty (0: none)
  int ir = 0;
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = j0 + i;
    ek[i] = 0u;
    if (j < a.V) {
      const uint32_t k = nkey(xv[i]);
      bad |= !is_finite(xv[i]);
      ir = k > br ? j : ir;
      br = k > br ? k : br;
      ek[i] = a.pp != 0.f && penalized(a, row, j) ? nkey(xv[i] - a.pp) : k;
      bp = ek[i] > bp ? ek[i] : bp;
    }
  }
  const uint64_t kr = ss_wave_max_u64(br ? ((uint64_t)br << 32) | (0xFFFFFFFFu - (uint32_t)ir) : 0ull);
  bad = ss_wave_or(bad);
  auto mx = [](uint32_t p, uint32_t q) { return p > q ? p : q; };
  auto scaled = [&](uint32_t k) { return k ? nkey(unkey_nan(k) / a.temperature) : 0u; };
  auto put = [&](int g) {  // the group of 64 / g lanes
    if (groups == g && (lane & (64 / g - 1)) == 0) w.gkey[c * g + lane / (64 / g)] = scaled(bp);
  };
  auto put_parts = [&](auto h_c) {  // H groups a lane
    constexpr int H = decltype(h_c)::value;
    if (groups != 64 * H) return;
#pragma unroll
    for (int g = 0; g < H; ++g) {
      uint32_t k = 0;
#pragma unroll
      for (int i = 0; i < kSub / H; ++i) k = mx(k, ek[g * (kSub / H) + i]);
      w.gkey[c * groups + lane * H + g] = scaled(k);
    }
  };
  put_parts(std::integral_constant<int, 16>{});
  put_parts(std::integral_constant<int, 8>{});
  put_parts(std::integral_constant<int, 4>{});
  put_parts(std::integral_constant<int, 2>{});
  put(64);
  bp = mx(bp, ss_xor_lane<1>(bp));
  put(32);
  bp = mx(bp, ss_xor_lane<2>(bp));
  put(16);
  bp = mx(bp, ss_xor_lane<4>(bp));
  put(8);
  bp = mx(bp, ss_xor_lane<8>(bp));
  put(4);
  uint32_t lo, hi;
  ss_pair<16>(bp, lo, hi);
  bp = mx(lo, hi);
  put(2);
  ss_pair<32>(bp, lo, hi);
  bp = mx(lo, hi);
  if (lane == 0) {
    const uint32_t k = scaled(bp);
    if (groups == 1) w.gkey[c] = k;
    w.craw[c] = kr;
    w.cbad[c] = (int)bad;
    w.cmax[c] = unkey_nan(k);
    w.cnan[c] = k == 0xFFFFFFFFu;
    if (c == 0 && row == 0) *w.done = 0;
  }
}

// NV: group keys per lane.
template <int NV>
__global__ __launch_bounds__(64) void samp_cand_kernel(SampArgs a, int groups, int vec) {
  const int c = blockIdx.x, row = blockIdx.y, lane = threadIdx.x, slots = slots_of(a.nch);
  SW w = sw_of(a.work, a.V, a.nch, row);
  const float* x = a.x + (size_t)row * a.V;
  const int ng = groups * a.nch, j0 = c * kChunk + lane * kSub;
  uint32_t gk[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) gk[i] = lane + 64 * i < ng ? w.gkey[lane + 64 * i] : 0u;
  float xv[kSub];
  load_chunk(x, j0, a.V, vec != 0, xv);
  uint32_t kmax = gk[0];  // the row's largest key: its maximum (NaN: the row takes the fallback, whatever is listed)
#pragma unroll
  for (int i = 1; i < NV; ++i) kmax = gk[i] > kmax ? gk[i] : kmax;
  const float m = unkey_nan(ss_wave_max_u32(kmax));
  uint32_t tau = 0;
  if (a.top_k <= ng) {
#pragma unroll 1
    for (int b = 31; b >= 16; --b) {
      const uint32_t t = tau | (1u << b);
      uint32_t n = 0;
#pragma unroll
      for (int i = 0; i < NV; ++i) n += gk[i] >= t;
      n = ss_butterfly(n, [](uint32_t p, uint32_t q) { return p + q; });
      tau = (int)n >= a.top_k ? t : tau;
    }
  }
  uint32_t take = 0;
  float lv[kSub];
#pragma unroll
  for (int i = 0; i < kSub; ++i) {
    const int j = j0 + i;
    const float l = (j < a.V && penalized(a, row, j) ? xv[i] - a.pp : xv[i]) / a.temperature;
    lv[i] = l;
    if (j < a.V && nkey(l) >= tau) take |= 1u << i;
  }
  if (__ballot(take != 0)) {
    // l < m - 103.98 is exactly exp 0 (ss_expf's bound); NaN compares false and is dropped with its row
#pragma unroll
    for (int i = 0; i < kSub; ++i)
      if (!(lv[i] - m >= -103.97208404541015625f)) take &= ~(1u << i);
  }
  const int nz = __popc(take);
  int incl = nz;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d);
    incl += lane >= d ? o : 0;
  }
  int pos = incl - nz;
#pragma unroll
  for (int i = 0; i < kSub; ++i)
    if ((take >> i) & 1u) {
      if (pos < slots) w.cand[(size_t)c * slots + pos] = ((uint64_t)(uint32_t)(j0 + i) << 32) | __float_as_uint(lv[i]);
      ++pos;
    }
  if (lane == 63) w.cnz[c] = incl;
}

// The accept walk of the sampled round from the rows' results, one thread (see samp_decide_kernel).
SS_DEV void accept_walk(const SampArgs& a) {
  const int D = a.R - 1;
  int na = 0, ne = 0, nu = 0, fl = 0;
  for (int i = 0; i <= D; ++i) {
    const SW w = sw_of(a.work, a.V, a.nch, i);
    const int tok = __hip_atomic_load(w.res, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int fb = __hip_atomic_load(w.res + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__hip_atomic_load(w.res + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      fl |= kFlagNonfinite;
      break;
    }
    a.out[4 + i] = tok;
    ne = i + 1;
    if (a.temperature > 0.f) nu = i + 1;
    if (fb) fl |= kFlagFallback;
    if (i == D) break;
    const int d = a.drafts[i];
    if (d < 0 || d >= a.V) fl |= kFlagBadDraft;
    if (tok != d) break;
    na = i + 1;
  }
  for (int i = ne; i <= D; ++i) a.out[4 + i] = -1;
  a.out[0] = na;
  a.out[1] = ne;
  a.out[2] = nu;
  a.out[3] = fl;
}

constexpr int kDrawThreads = 1024, kDrawWaves = kDrawThreads / 64;

struct DrawSmem {
  int off[kDrawThreads];       // inclusive candidate counts over the chunks
  int j[kCand];                // candidates, then (j2, p) the survivors, in index order
  float l[kCand];
  __attribute__((aligned(16))) uint32_t key[kCand];  // zero-padded to a multiple of 8
  int j2[kSurv], rank[kSurv];
  float p[kSurv];              // exp, probabilities, final weights
  __attribute__((aligned(16))) uint64_t rho[kSurv];  // zero-padded to a multiple of 4
  float by_rank[kSurv];        // probabilities by rank
  int start[kSurv + 1];        // first survivor of each active chunk
  int multi[kSurv];            // the active chunk has survivors in more than one sub-chunk
  int mlist[kSurv];            // the chunks that have
  __attribute__((aligned(16))) float ct[kDrawThreads];  // chunk totals (the draw; the in-workgroup sequence)
  int wsum[kDrawWaves];
  uint32_t wmax[kDrawWaves];
  int hist[256];
  uint32_t kth;
  int pick, digit, prefix, need;
  float z;
};

// Inclusive sum over the workgroup of v (threads in order); `total` the sum over all.
SS_DEV int block_scan(int v, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d);
    incl += lane >= d ? o : 0;
  }
  __syncthreads();
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int q = 0; q < kDrawWaves; ++q) {
    incl += q < w ? wsum[q] : 0;
    t += wsum[q];
  }
  total = t;
  return incl;
}

// Hierarchical sum of the survivors of rank < m (whole workgroup): the active chunks' totals into s.ct (zero-padded to a
// multiple of 16), then their sum in order, by every wave. A chunk whose survivors share one sub-chunk is their sum in
// index order (the butterfly adds zeros), by one thread; another (nm of them) takes the butterfly over its leaves, by one
// wave, its survivors handed round by lane reads.
SS_DEV float masked_sum(DrawSmem& s, int na, int nm, int m) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  __syncthreads();  // the sums of the call before have been read
  if (tid < ((na + 15) & ~15)) {
    float v = 0.f;
    if (tid < na && !s.multi[tid]) {
      const int q0 = s.start[tid], q1 = s.start[tid + 1];
      const float p0 = s.p[q0];
      v = s.rank[q0] < m ? p0 : 0.f;
      for (int q = q0 + 1; q < q1; ++q) {
        const float nx = v + s.p[q];
        v = s.rank[q] < m ? nx : v;
      }
    }
    if (tid >= na || !s.multi[tid]) s.ct[tid] = v;
  }
  for (int i = wv; i < nm; i += kDrawWaves) {
    const int t = s.mlist[i], q0 = s.start[t], q1 = s.start[t + 1];
    float leaf = 0.f;
    if (q1 - q0 > 64) {  // lane b finds its run of survivors (sub-chunk b) by bisection
      int lo = q0, hi = q1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (((s.j2[mid] & (kChunk - 1)) >> 4) < lane) lo = mid + 1;
        else hi = mid;
      }
      for (int q = lo; q < q1 && ((s.j2[q] & (kChunk - 1)) >> 4) == lane; ++q) {
        const float nx = leaf + s.p[q];
        leaf = s.rank[q] < m ? nx : leaf;
      }
    } else {
      const int n = q1 - q0, q = lane < n ? q0 + lane : q0;
      const float p = s.p[q];
      const int at = s.rank[q] < m ? (s.j2[q] & (kChunk - 1)) >> 4 : -1;
      for (int k = 0; k < n; ++k) {
        const float nx = leaf + ss_readlane_f(p, k);
        leaf = __builtin_amdgcn_readlane(at, k) == lane ? nx : leaf;
      }
    }
    leaf = ss_wave_sum(leaf);
    if (lane == 0) s.ct[t] = leaf;
  }
  __syncthreads();
  return lds_seq_sum(s.ct, na, 0.f);
}

// The key of rank `need` (largest first, counting multiplicity) among key(0) .. key(n - 1), whole workgroup.
template <class F>
SS_DEV void radix_select(DrawSmem& s, int n, F key, int need, uint32_t& prefix) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  prefix = 0;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    __syncthreads();
    if (tid < 256) s.hist[tid] = 0;
    __syncthreads();
    for (int j = tid; j < n; j += kDrawThreads) {
      const uint32_t k = key(j);
      if (pass == 0 || (k >> (shift + 8)) == (prefix >> (shift + 8))) atomicAdd(&s.hist[(k >> shift) & 255], 1);
    }
    __syncthreads();
    if (wv == 0) {
      select_pass<1>(s.hist, need, prefix, shift);
      if (lane == 0) {
        s.prefix = (int)prefix;
        s.need = need;
      }
    }
    __syncthreads();
    prefix = (uint32_t)s.prefix;
    need = s.need;
  }
}

// The whole sequence of a top-k row inside the workgroup (the launches below, chunk by chunk): more candidates or
// survivors than the lists hold. Returns the token, or -1 when the total is not finite and > 0.
SS_DEV int draw_in_workgroup(const SampArgs& a, const SW& w, DrawSmem& s, int row, float m, float* masses) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nch = a.nch;
  const float* x = a.x + (size_t)row * a.V;
  for (int j = tid; j < a.V; j += kDrawThreads) w.L[j] = logit_of(a, x, row, j);
  uint32_t prefix = 0;
  radix_select(s, a.V, [&](int j) { return nkey(w.L[j]); }, a.top_k, prefix);
  const float kth = unkey_nan(prefix);
  for (int c = wv; c < nch; c += kDrawWaves) {
    float v[kSub], sub;
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      const int j = c * kChunk + lane * kSub + i;
      const float l = j < a.V ? w.L[j] : 0.f;
      v[i] = j < a.V ? (l < kth ? 0.f : ss_expf(l - m)) : 0.f;
      if (j < a.V) w.P[j] = v[i];
    }
    const float t = chunk_sum(v, sub);
    if (lane == 0) s.ct[c] = t;
  }
  __syncthreads();
  if (tid == 0) {
    float z = 0.f;
    for (int c = 0; c < nch; ++c) z = z + s.ct[c];
    s.z = z;
  }
  __syncthreads();
  const float z = s.z;
  uint64_t r = 0;
  if (a.top_p < 1.f) {
    for (int round = 0; round < kRounds; ++round) {
      const int sft = kRhoBits - 4 - 4 * round;
      const uint64_t r_hi = r >> (sft + 4);
      for (int c = wv; c < nch; c += kDrawWaves) {
        float acc[16];
#pragma unroll
        for (int d = 0; d < 16; ++d) acc[d] = 0.f;
#pragma unroll
        for (int i = 0; i < kSub; ++i) {
          const int j = c * kChunk + lane * kSub + i;
          const float p = j < a.V ? w.P[j] / z : 0.f;
          if (j < a.V && p != 0.f) {
            const uint64_t rho = rho_of(p, j);
            const uint64_t hi = rho >> (sft + 4);
            const int lim = hi > r_hi ? 16 : (hi == r_hi ? (int)((rho >> sft) & 15) : 0);
#pragma unroll
            for (int d = 0; d < 16; ++d) acc[d] = acc[d] + (d < lim ? p : 0.f);
          }
        }
#pragma unroll
        for (int d = 0; d < 16; ++d) {
          const float t = ss_wave_sum(acc[d]);
          if (lane == 0) masses[d * nch + c] = t;
        }
      }
      __syncthreads();
      if (wv == 0) {
        float cum = 0.f;
        for (int c = 0; c < nch; ++c) cum = cum + masses[(lane & 15) * nch + c];
        const uint64_t ok = __ballot(lane < 16 && cum < a.top_p);
        if (lane == 0) s.digit = ok ? (int)__builtin_ctzll(ok) : 15;
      }
      __syncthreads();
      r |= (uint64_t)s.digit << sft;
    }
  }
  // keep rho >= r; the largest kept probability for min-p
  float pm = -__builtin_inff();
  for (int j = tid; j < a.V; j += kDrawThreads) {
    float p = w.P[j] / z;
    if (a.top_p < 1.f && !(rho_of(p, j) >= r)) p = 0.f;
    w.P[j] = p;
    pm = fmaxf(pm, p);
  }
  pm = ss_wave_max(pm);
  __syncthreads();
  if (lane == 0) masses[wv] = pm;
  __syncthreads();
  for (int q = 0; q < kDrawWaves; ++q) pm = fmaxf(pm, masses[q]);
  const float cutoff = pm * a.min_p;
  if (tid < kDrawThreads) s.ct[tid] = 0.f;
  __syncthreads();
  for (int c = wv; c < nch; c += kDrawWaves) {
    float v[kSub], sub;
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      const int j = c * kChunk + lane * kSub + i;
      float p = j < a.V ? w.P[j] : 0.f;
      if (a.min_p > 0.f && p < cutoff) {
        p = 0.f;
        if (j < a.V) w.P[j] = 0.f;
      }
      v[i] = p;
    }
    const float t = chunk_sum(v, sub);
    w.stot[c * 64 + lane] = sub;
    if (lane == 0) s.ct[c] = t;
  }
  __syncthreads();
  int pick = -1;
  if (wv == 0) {
    const float total = lds_seq_sum(s.ct, nch, 0.f);
    if (is_finite(total) && total > 0.f) pick = draw_descent(a.u[row], total, s.ct, nch, w.stot, w.P, a.V);
    if (lane == 0) s.pick = pick;
  }
  __syncthreads();
  return s.pick;
}

__global__ __launch_bounds__(kDrawThreads) void samp_topk_draw_kernel(SampArgs a) {
  extern __shared__ __attribute__((aligned(16))) float masses[];  // [16][nch]: the in-workgroup sequence
  __shared__ __attribute__((aligned(16))) DrawSmem s;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nch = a.nch;
  SW w = sw_of(a.work, a.V, nch, row);
  auto finish = [&](int tok, int fb, int nonfinite) {  // whole workgroup
    if (tid != 0) return;
    if (!a.accept) {
      a.out[0] = tok;
      a.out[1] = fb;
      return;
    }
    __hip_atomic_store(w.res, tok, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w.res + 1, fb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w.res + 2, nonfinite, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // the results are performed before the arrival below is counted
    int* done = sw_of(a.work, a.V, nch, 0).done;
    if (__hip_atomic_fetch_add(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.R - 1) accept_walk(a);
  };
  const int cnt = tid < nch ? w.cnz[tid] : 0;
  const bool bad = tid < nch && w.cbad[tid] != 0, over = cnt > slots_of(nch);
  const uint32_t cm = tid < nch ? nkey(w.cmax[tid]) : 0u;
  const uint32_t wm = ss_wave_max_u32(cm);
  if (lane == 0) s.wmax[wv] = wm;
  if (__syncthreads_or(a.accept && bad)) return finish(-1, 0, 1);
  uint32_t km = s.wmax[0];
#pragma unroll
  for (int q = 1; q < kDrawWaves; ++q) km = s.wmax[q] > km ? s.wmax[q] : km;
  const float m = unkey_nan(km);
  if (!is_finite(m)) {
    // exp(l - m) is NaN somewhere (or everywhere): the total is NaN, and the draw takes the raw argmax
    const uint64_t k = max_u64_of(w.craw, nch);
    return finish((int)(0xFFFFFFFFu - (uint32_t)k), 1, 0);
  }
  int n;
  s.off[tid] = block_scan(cnt, s.wsum, n);
  int ns = 0, na = 0, nm = 0;
  float z = 0.f;
  bool slow = __syncthreads_or(over) || n > kCand;
  if (!slow) {
    // gather the candidates in index order
    for (int q = tid; q < n; q += kDrawThreads) {
      int lo = 0, hi = nch - 1;  // the first chunk whose inclusive count exceeds q
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s.off[mid] > q) hi = mid;
        else lo = mid + 1;
      }
      const uint64_t e = w.cand[(size_t)lo * slots_of(nch) + (q - (lo ? s.off[lo - 1] : 0))];
      s.j[q] = (int)(e >> 32);
      s.l[q] = __uint_as_float((uint32_t)e);
      s.key[q] = nkey(s.l[q]);
    }
    if (tid < 8 && n + tid < kCand) s.key[n + tid] = 0u;
    if (tid == 0) s.kth = 0u;
    __syncthreads();
    // the k-th largest key, counting multiplicity: by ranks of a short list, by four 8-bit radix passes of a long one
    if (n > a.top_k && n <= kRankMax) {
      for (int q = tid; q < n; q += kDrawThreads) {
        const uint32_t k = s.key[q];  // above 0, the padding's key
        int gt = 0, ge = 0;
        for (int t = 0; t < n; t += 8) {
          const uint4 o0 = *reinterpret_cast<const uint4*>(s.key + t), o1 = *reinterpret_cast<const uint4*>(s.key + t + 4);
          gt += (o0.x > k) + (o0.y > k) + (o0.z > k) + (o0.w > k) + (o1.x > k) + (o1.y > k) + (o1.z > k) + (o1.w > k);
          ge += (o0.x >= k) + (o0.y >= k) + (o0.z >= k) + (o0.w >= k) + (o1.x >= k) + (o1.y >= k) + (o1.z >= k) +
                (o1.w >= k);
        }
        if (gt < a.top_k && a.top_k <= ge) s.kth = k;  // the same value from every thread that holds it
      }
      __syncthreads();
    } else if (n > a.top_k) {
      uint32_t prefix = 0;
      radix_select(s, n, [&](int q) { return s.key[q]; }, a.top_k, prefix);
      if (tid == 0) s.kth = prefix;
      __syncthreads();
    }
    const uint32_t kth = s.kth;
    // survivors, in index order
    const int q0 = 2 * tid, q1 = q0 + 1;
    const bool k0 = q0 < n && s.key[q0] >= kth, k1 = q1 < n && s.key[q1] >= kth;
    int pos = block_scan((int)k0 + (int)k1, s.wsum, ns) - (int)k0 - (int)k1;
    slow = ns > kSurv;
    if (!slow) {
      if (k0) {
        s.j2[pos] = s.j[q0];
        s.p[pos] = ss_expf(s.l[q0] - m);
        ++pos;
      }
      if (k1) {
        s.j2[pos] = s.j[q1];
        s.p[pos] = ss_expf(s.l[q1] - m);
      }
      __syncthreads();
      // active chunks: first survivor of each, and whether its survivors span several sub-chunks
      const bool head = tid < ns && (tid == 0 || (s.j2[tid] >> 10) != (s.j2[tid - 1] >> 10));
      const int t = block_scan(head ? 1 : 0, s.wsum, na) - 1;
      if (tid < kSurv) s.multi[tid] = 0;
      if (head) s.start[t] = tid;
      if (tid == 0) s.start[na] = ns;
      __syncthreads();
      if (tid < ns && !head && (s.j2[tid] >> 4) != (s.j2[tid - 1] >> 4)) s.multi[t] = 1;
      if (tid < ns) s.rank[tid] = 0;
      __syncthreads();
      const int mine = tid < na ? s.multi[tid] : 0;
      const int at = block_scan(mine, s.wsum, nm) - mine;
      if (mine) s.mlist[at] = tid;
      z = masked_sum(s, na, nm, 1);
    }
  }
  if (slow) {
    const int pick = draw_in_workgroup(a, w, s, row, m, masses);
    if (pick >= 0) return finish(pick, 0, 0);
    const uint64_t k = max_u64_of(w.craw, nch);
    return finish((int)(0xFFFFFFFFu - (uint32_t)k), 1, 0);
  }
  // probabilities and their ranks by rho (descending; distinct, they end in the index)
  if (tid < ns) {
    s.p[tid] = s.p[tid] / z;
    s.rho[tid] = rho_of(s.p[tid], s.j2[tid]);
  } else if (tid < ns + 4 && tid < kSurv) {
    s.rho[tid] = 0ull;
  }
  __syncthreads();
  if (tid < ns) {
    const uint64_t r = s.rho[tid];
    int rk = 0;
    for (int t = 0; t < ns; t += 4) {
      const ulonglong2 a0 = *reinterpret_cast<const ulonglong2*>(s.rho + t);
      const ulonglong2 a1 = *reinterpret_cast<const ulonglong2*>(s.rho + t + 2);
      rk += (a0.x > r) + (a0.y > r) + (a1.x > r) + (a1.y > r);
    }
    s.rank[tid] = rk;
    s.by_rank[rk] = s.p[tid];
  }
  __syncthreads();
  // top-p: cum(r) is a step function of the survivors, so the smallest r with cum(r) < top_p is the rho of the m'-th
  // survivor, m' the smallest m with S(m) >= top_p (S grows with m: every partial sum is a monotone function of
  // non-negative terms): the survivors of rank < m' stay. None: all stay.
  int keep = ns;
  if (a.top_p < 1.f) {
    // The first probe is the count at which the plain prefix sum by rank reaches top_p, then its neighbours: the
    // masses differ from it by rounding only, so two probes usually close the bracket.
    int g = 0;
    for (float run = 0.f; g < ns;) {
      const float v = g + lane < ns ? s.by_rank[g + lane] : 0.f;
      float incl = v;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float o = __shfl_up(incl, d);
        incl += lane >= d ? o : 0.f;
      }
      const uint64_t at = __ballot(run + incl >= a.top_p);
      if (at) {
        g += (int)__builtin_ctzll(at) + 1;
        break;
      }
      run += __shfl(incl, 63);
      g += 64;
    }
    int lo = 0, hi = ns + 1, step = 1;
    g = g < 1 ? 1 : (g > ns ? ns : g);
    while (hi - lo > 1) {
      int mid = g;
      if (mid <= lo || mid >= hi) mid = (lo + hi) >> 1;
      const bool up = masked_sum(s, na, nm, mid) >= a.top_p;  // the same in every wave
      if (up) hi = mid;
      else lo = mid;
      g = up ? mid - step : mid + step;
      step *= 2;
    }
    keep = hi < ns ? hi : ns;
  }
  // min-p on what stays: its largest probability is rank 0's
  const float cutoff = s.by_rank[0] * a.min_p;
  if (tid < ns && (s.rank[tid] >= keep || (a.min_p > 0.f && s.p[tid] < cutoff))) s.p[tid] = 0.f;
  const float total = masked_sum(s, na, nm, ns);
  if (wv != 0) return;  // one wave from here
  if (!is_finite(total) || !(total > 0.f)) {
    const uint64_t k = max_u64_of(w.craw, nch);
    return finish((int)(0xFFFFFFFFu - (uint32_t)k), 1, 0);
  }
  // the descent of draw_descent over the survivors: chunks, leaves and entries without weight leave its running sums
  // and its choices unchanged
  const float u = a.u[row];
  const bool ge = u != 0.f;
  const float target = ge ? u * total : 0.f;
  auto hit = [&](float v) { return ge ? v >= target : v > target; };
  int cs = -1, clast = -1;
  float base = 0.f, run = 0.f;
  for (int t0 = 0; t0 < na && cs < 0; t0 += 64) {
    const float v = t0 + lane < na ? s.ct[t0 + lane] : 0.f;
    const uint64_t pos = __ballot(v > 0.f);
    if (pos) clast = t0 + 63 - (int)__builtin_clzll(pos);
    const int nt = na - t0 < 64 ? na - t0 : 64;
    for (int q = 0; q < nt; ++q) {
      const float nx = run + ss_readlane_f(v, q);
      if (hit(nx)) {
        cs = t0 + q;
        base = run;
        break;
      }
      run = nx;
    }
  }
  if (cs < 0) {
    cs = clast;
    base = 0.f;
    for (int t = 0; t < cs; ++t) base = base + s.ct[t];
  }
  const int a0 = s.start[cs], a1 = s.start[cs + 1];
  float sub = 0.f;  // lane b: the total of sub-chunk b
  for (int q = a0; q < a1; ++q) {
    const float nx = sub + s.p[q];
    sub = ((s.j2[q] & (kChunk - 1)) >> 4) == lane ? nx : sub;
  }
  int bs = -1, blast = 0;
  float sbase = base;
  run = base;
  for (uint64_t todo = __ballot(sub > 0.f); todo; todo &= todo - 1) {
    const int b = (int)__builtin_ctzll(todo);
    const float nx = run + ss_readlane_f(sub, b);
    blast = b;
    if (hit(nx)) {
      bs = b;
      sbase = run;
      break;
    }
    run = nx;
  }
  if (bs < 0) {
    bs = blast;
    sbase = base;
    for (int b = 0; b < bs; ++b) sbase = sbase + ss_readlane_f(sub, b);
  }
  int pick = -1, last = -1;
  run = sbase;
  for (int q = a0; q < a1; ++q) {
    const int j = s.j2[q];
    if (((j & (kChunk - 1)) >> 4) != bs) continue;
    const float v = s.p[q];
    last = v > 0.f ? j : last;
    run = run + v;
    if (hit(run)) {
      pick = j;
      break;
    }
  }
  finish(pick >= 0 ? pick : last, 0, 0);
}

// 8. accept mode: the round, walking the rows in order (n_accept, n_emit, n_uniform, flags, tokens).
__global__ __launch_bounds__(64) void samp_decide_kernel(SampArgs a) {
  if (threadIdx.x == 0) accept_walk(a);
}

namespace {

SampArgs args_of(int V, int R, const int32_t* gen, int n_gen, float temperature, float top_p, int top_k,
                 float min_p, float pp, void* work) {
  SampArgs a{};
  a.V = V;
  a.nch = (V + kChunk - 1) / kChunk;
  a.R = R;
  a.gen = gen;
  a.n_gen = n_gen;
  a.temperature = temperature;
  a.top_p = top_p;
  a.top_k = top_k;
  a.min_p = min_p;
  a.pp = pp;
  a.work = work;
  return a;
}

size_t topp_lds_bytes(int nch) { return (size_t)16 * ((nch + 15) & ~15) * sizeof(float); }

// Groups per chunk of a top-k row: the smallest power of two that gives 2 k groups in the row, kKeys keys at most. Every
// k <= 512 gets its 2 k: a row of n chunks may have up to kKeys / n groups a chunk (rounded down to a power of two, one
// entry each at most), which is more than 1024 groups with entries in every row of more than one chunk; one chunk has a
// group per entry, and then the bound is the k-th largest entry itself but for its low bits.
int groups_of(const SampArgs& a) {
  int groups = 1;
  while (groups < kChunk && (int64_t)groups * a.V < (int64_t)2 * a.top_k * kChunk && 2 * groups * a.nch <= kKeys) groups *= 2;
  return groups;
}

// A top-k row's three launches (they draw, and in accept mode walk the round).
bool topk_rows(const SampArgs& a) {
  return a.temperature > 0.f && a.top_k > 0 && a.top_k < a.V && a.top_k <= kTopkMax && a.nch <= kDrawThreads;
}

hipError_t launch_topk_rows(const SampArgs& a, hipStream_t st) {
  const dim3 g(a.nch, a.R), b(64);
  const int groups = groups_of(a), ng = groups * a.nch, vec = a.V % 4 == 0 && reinterpret_cast<uintptr_t>(a.x) % 16 == 0;
  KernelCfg cfg;
  const hipError_t e = kernel_cfg(reinterpret_cast<const void*>(samp_topk_draw_kernel), kDrawThreads, 64 * 1024, &cfg);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(samp_scan_kernel, g, b, 0, st, a, groups, vec);
  if (ng <= 256) hipLaunchKernelGGL(samp_cand_kernel<4>, g, b, 0, st, a, groups, vec);
  else if (ng <= 1024) hipLaunchKernelGGL(samp_cand_kernel<16>, g, b, 0, st, a, groups, vec);
  else hipLaunchKernelGGL(samp_cand_kernel<32>, g, b, 0, st, a, groups, vec);
  hipLaunchKernelGGL(samp_topk_draw_kernel, dim3(a.R), dim3(kDrawThreads), (size_t)16 * a.nch * sizeof(float), st, a);
  return hipGetLastError();
}

// The rows' launch sequence of every other row; which kernels run depends only on the parameters.
void launch_rows(const SampArgs& a, hipStream_t st) {
  const dim3 g(a.nch, a.R), b(64);
  if (!(a.temperature > 0.f)) {
    hipLaunchKernelGGL(samp_prep_kernel, g, b, 0, st, a, 0);
    hipLaunchKernelGGL(samp_draw_kernel, dim3(a.R), b, 0, st, a);
    return;
  }
  const int has_k = a.top_k > 0 && a.top_k < a.V;
  const int has_p = a.top_p < 1.f;
  const int has_minp = a.min_p > 0.f;
  if (has_k) hipLaunchKernelGGL(samp_begin_kernel, dim3(a.R), dim3(256), 0, st, a);
  hipLaunchKernelGGL(samp_prep_kernel, g, b, 0, st, a, has_k);
  if (has_k)
    for (int pass = 1; pass < 4; ++pass) hipLaunchKernelGGL(samp_hist_kernel, g, b, 0, st, a, pass);
  hipLaunchKernelGGL(samp_exp_kernel, g, b, 0, st, a, has_k);
  if (has_p)
    for (int round = 0; round < kRounds; ++round)
      hipLaunchKernelGGL(samp_topp_kernel, g, b, topp_lds_bytes(a.nch), st, a, round);
  if (has_p || has_minp)
    hipLaunchKernelGGL(samp_keep_kernel, g, b, has_p ? topp_lds_bytes(a.nch) : 0, st, a, has_p, has_p ? 0 : 1);
  hipLaunchKernelGGL(samp_total_kernel, g, b, 0, st, a, has_minp, (has_p || has_minp) ? 0 : 1);
  hipLaunchKernelGGL(samp_draw_kernel, dim3(a.R), b, 0, st, a);
}

}  // namespace

int64_t sample_workspace_bytes(int V) {
  const int nch = (V + kChunk - 1) / kChunk;
  return (int64_t)layout_of(V, nch).bytes;
}

hipError_t launch_sample(const float* x, int V, const int32_t* gen, int n_gen, float temperature, float top_p,
                         int top_k, float min_p, float pp, const float* u, void* work, int32_t* out, hipStream_t st) {
  SampArgs a = args_of(V, 1, gen, n_gen, temperature, top_p, top_k, min_p, pp, work);
  a.x = x;
  a.u = u;
  a.out = out;
  if (topk_rows(a)) return launch_topk_rows(a, st);
  launch_rows(a, st);
  return hipGetLastError();
}

hipError_t launch_accept_sampled(const float* target, const int32_t* drafts, int D, int V, const int32_t* seen,
                                 int n_seen, float temperature, float top_p, int top_k, float min_p, float pp,
                                 const float* uniforms, void* work, int32_t* out, hipStream_t st) {
  SampArgs a = args_of(V, D + 1, seen, n_seen, temperature, top_p, top_k, min_p, pp, work);
  a.x = target;
  a.u = uniforms;
  a.drafts = drafts;
  a.out = out;
  a.accept = 1;
  if (topk_rows(a)) return launch_topk_rows(a, st);
  launch_rows(a, st);
  hipLaunchKernelGGL(samp_decide_kernel, dim3(1), dim3(64), 0, st, a);
  return hipGetLastError();
}

}  // namespace ss
