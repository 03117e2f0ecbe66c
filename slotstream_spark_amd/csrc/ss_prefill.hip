// Prefill MoE: rows sorted into expert-contiguous blocks, a grouped bf16 MFMA GEMM over affine-4bit records
// dequantized into MFMA registers, and the rank-order combine.
//
// Semantics follow kernels/moe_align.py:11-48, kernels/fused_moe_affine.py:39-172 (the reference's prefill path):
//  * moe_align: a stable counting sort of the rows by local expert (rows outside [0, num_local) are skipped); each
//    expert's rows padded to block_m with the sentinel R; every block of block_m positions belongs to one expert.
//    Computed without atomics in any order-dependent place: ranks inside a 1024-row chunk by ballots and per-wave
//    counts, chunk offsets by a sequential scan per expert.
//  * gate/up: h[r, n] = bf16(silu(g) * u), g = sum_k x[tok(r), k] * bf16(q*s + b)[n, k] with bf16 products and
//    fp32 accumulation (the dequantized weight is rounded to bf16 as the reference's _wtile does; q*s is exact
//    in fp32, so one rounding of q*s + b, fused or not, gives the same value).
//  * down: out_rows[r, n] = (sum_k h[r, k] * bf16(q*s + b)[n, k]) * row_weight[r], fp32.
//  * combine: out[t] = ((o[t,0] + o[t,1]) + ...) + o[t,K-1], sequential fp32.
// Every output row is accumulated in one fixed K order, whatever the tile shape and the number of rows.
#include <type_traits>

#include "ss_common.hpp"
#include "ss_launch.hpp"

namespace ss {

// ---------------------------------------------------------------- moe_align
// Three launches (count, scan, place; four with many keys or chunks), or one workgroup for up to kAlignChunk rows and
// keys: the plan is a chain of small dependent steps, so what it costs is launches and the latency inside each (190 rows,
// 512 keys, block_m 128: seven launches 17.4 us, one 9.0; 1024 rows 17.8 and 13.4).
constexpr int kAlignChunk = 1024;         // rows per workgroup of the counting kernel
constexpr int kAlignWaves = kAlignChunk / 64;

int64_t padded_rows(int64_t R, int num_local, int block_m) {
  const int64_t n = R + (int64_t)num_local * (block_m - 1);
  return (n + block_m - 1) / block_m * block_m;
}

// scratch ints: rank [R], chunk offsets [nchunk][num_local], pad_start [num_local + 1], totals [num_local]
int64_t align_scratch_ints(int64_t R, int num_local) {
  const int64_t nch = (R + kAlignChunk - 1) / kAlignChunk;
  return R + nch * num_local + 2 * (int64_t)num_local + 1;
}

namespace {

struct PlanArgs {
  const int32_t* le;  // [R] local expert of each row, or null: the rows' expert ids through the resident tables
  const int32_t* ids;
  const int32_t* map;
  int64_t map_base, map_len;
  const int64_t* slot_ptr;
  int64_t n_slots;
  int32_t* local;     // [R] local expert written with `ids` (-1: not resident)
  int* err;
  int64_t R, P, nb;   // rows; positions of sorted_rows to fill; entries of block_expert
  int nl, bm, nch;
  int32_t* rank;
  int32_t* chunk;
  int32_t* pad;
  int32_t* tot;
  int32_t* sorted_rows;
  int32_t* block_expert;
  int32_t* num_padded;
  MBlock* order;      // null, or the M blocks in launch order
};

// Key of row i: its local expert, nl for a row that is skipped, nl + 1 past R.
template <bool IDS>
SS_DEV int align_key(const PlanArgs& a, int64_t i) {
  if (i >= a.R) return a.nl + 1;
  if constexpr (!IDS) {
    const int v = a.le[i];
    return (v >= 0 && v < a.nl) ? v : a.nl;
  } else {
    const int e = a.ids[i];
    if (e < 0 || e >= a.nl) {
      ss_raise(a.err, SS_ERR_EXPERT_ID);
      return a.nl;
    }
    const int64_t mi = a.map_base + e;
    const int slot = mi < a.map_len ? a.map[mi] : -1;
    if (slot >= 0 && slot < a.n_slots) return e;
    ss_raise(a.err, SS_ERR_SLOT);
    return a.nl;
  }
}

// Rank of each thread's row among the earlier rows of the workgroup with the same key, and the workgroup's count of
// every key (cnt[w * nk + key], summed by the caller). Inside a wave the lanes holding the same key are the AND of the
// ballots of the key's bits; the earlier waves add their counts of that key from LDS.
SS_DEV int align_rank(int key, int nk, uint8_t* cnt) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int e = tid; e < kAlignWaves * nk; e += kAlignChunk) cnt[e] = 0;
  __syncthreads();
  uint64_t same = ~0ull;
  for (int b = 0; (nk - 1) >> b; ++b) {
    const uint64_t set = __ballot((key >> b) & 1);
    same &= (key >> b) & 1 ? set : ~set;
  }
  int r = __popcll(same & ((1ull << lane) - 1ull));
  if (r == 0) cnt[w * nk + key] = (uint8_t)__popcll(same);
  __syncthreads();
  for (int v = 0; v < w; ++v) r += cnt[v * nk + key];
  return r;
}

SS_DEV int align_count_of(const uint8_t* cnt, int nk, int e) {
  int c = 0;
#pragma unroll
  for (int v = 0; v < kAlignWaves; ++v) c += cnt[v * nk + e];
  return c;
}

// Record of expert e (0 when it is not resident; its rows are skipped, so no block names it).
SS_DEV int64_t record_of(const PlanArgs& a, int e) {
  const int64_t mi = a.map_base + e;
  const int slot = mi < a.map_len ? a.map[mi] : -1;
  return slot >= 0 && slot < a.n_slots ? a.slot_ptr[slot] : 0;
}

// One workgroup of 1024: the padded start of every key (ps, nl + 1 entries; hv: the heavy blocks before it), the
// expert of every M block and, with `order`, the blocks in launch order. Thread t holds the totals of keys
// kpt t .. kpt t + kpt - 1 in loc.
// Launch order: blocks with more than half their rows first, the others behind them, so the light blocks fill the
// chip's tail instead of leaving it to a few heavy ones. Layer, us, heavy first / plan order: top-10 of 512, Zipf routing,
// 200 tokens 101 / 107, 333 118 / 128, 1400 254 / 272, 2048 308 / 313, at H 2560 333 175 / 193, 3000 614 / 638; top-8 of 64
// 1000 tokens 141 / 160, 2048 245 / 268, 4096 402 / 416. It costs some long prompts, where plan order mixes full and
// partial blocks on a CU: 512 experts 4096 tokens 543 / 531, 8192 937 / 936 and 973 / 931 by the routing's seed, 256 experts
// 8192 791 / 753; no size tells these from 8192 at H 2560 (1353 / 1358) or 128 experts uniform 6000 (554 / 573).
SS_DEV void align_scan(const PlanArgs& a, const int (&loc)[4], int kpt, int* ps, int* hv) {
  __shared__ int wsum[2][16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int bm = a.bm, nl = a.nl;
  auto blocks_of = [&](int c) { return (c + bm - 1) / bm; };
  auto heavy_of = [&](int c) { return c / bm + (c % bm > bm / 2 ? 1 : 0); };
  int nbk = 0, nh = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (q < kpt) {
      nbk += blocks_of(loc[q]);
      nh += heavy_of(loc[q]);
    }
  int ib = nbk, ih = nh;  // inclusive scans over the wave, then over the waves
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int vb = __shfl_up(ib, off), vh = __shfl_up(ih, off);
    if (lane >= off) {
      ib += vb;
      ih += vh;
    }
  }
  if (lane == 63) {
    wsum[0][w] = ib;
    wsum[1][w] = ih;
  }
  __syncthreads();
  int run = ib - nbk, runh = ih - nh;
  for (int v = 0; v < w; ++v) {
    run += wsum[0][v];
    runh += wsum[1][v];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = kpt * tid + q;
    if (q < kpt && e < nl) {
      ps[e] = run * bm;
      hv[e] = runh;
      run += blocks_of(loc[q]);
      runh += heavy_of(loc[q]);
      if (e == nl - 1) {
        ps[nl] = run * bm;
        hv[nl] = runh;
      }
    }
  }
  __syncthreads();
  const int total = ps[nl], nheavy = hv[nl];
  if (tid == 0) *a.num_padded = total;
  for (int64_t q = tid; q < a.nb; q += 1024) {
    const int64_t pos = q * bm;
    if (pos >= total) {
      a.block_expert[q] = -1;
      continue;
    }
    int lo = 0, hi = nl;  // the last key e with ps[e] <= pos
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (ps[mid] <= pos) lo = mid;
      else hi = mid - 1;
    }
    a.block_expert[q] = lo;
    if (a.order) {
      const int b0 = ps[lo] / bm, j = (int)q - b0, h = hv[lo + 1] - hv[lo];
      const int at = j < h ? hv[lo] + j : nheavy + (b0 - hv[lo]) + (j - h);
      a.order[at] = MBlock{record_of(a, lo), lo, (int32_t)q};
    }
  }
}

}  // namespace

// Per chunk of rows: ranks and counts of every key.
template <bool IDS>
__global__ __launch_bounds__(kAlignChunk) void align_count_kernel(PlanArgs a) {
  extern __shared__ uint8_t sm_cnt[];  // [kAlignWaves][nl + 2]: per-wave counts (<= 64) of keys 0 .. nl + 1
  const int64_t i = (int64_t)blockIdx.x * kAlignChunk + threadIdx.x;
  const int key = align_key<IDS>(a, i), nk = a.nl + 2;
  const int r = align_rank(key, nk, sm_cnt);
  if (i < a.R) {
    a.rank[i] = r;
    if (IDS) a.local[i] = key < a.nl ? key : -1;
  }
  for (int e = threadIdx.x; e < a.nl; e += kAlignChunk)
    a.chunk[(int64_t)blockIdx.x * a.nl + e] = align_count_of(sm_cnt, nk, e);
}

// Exclusive offsets of key e over the chunks (in place); returns its total. The loads are independent, 32 in flight.
SS_DEV int align_keyscan(const PlanArgs& a, int e) {
  int run = 0;
  for (int c0 = 0; c0 < a.nch; c0 += 32) {
    int v[32];
#pragma unroll
    for (int c = 0; c < 32; ++c) v[c] = c0 + c < a.nch ? a.chunk[(int64_t)(c0 + c) * a.nl + e] : 0;
#pragma unroll
    for (int c = 0; c < 32; ++c) {
      if (c0 + c < a.nch) a.chunk[(int64_t)(c0 + c) * a.nl + e] = run;
      run += v[c];
    }
  }
  return run;
}

// The key offsets as a launch of their own, for more counts than one workgroup should pass over.
__global__ __launch_bounds__(64) void align_keyscan_kernel(PlanArgs a) {
  const int e = blockIdx.x * 64 + threadIdx.x;
  if (e < a.nl) a.tot[e] = align_keyscan(a, e);
}

// One workgroup: the keys' offsets over the chunks and totals (with `scan`; they are there otherwise), then the padded
// starts, the blocks' experts and the launch order.
__global__ __launch_bounds__(1024) void align_scan_kernel(PlanArgs a, int scan) {
  extern __shared__ int sm_scan[];  // [2][nl + 1]
  int* ps = sm_scan;
  int* hv = sm_scan + a.nl + 1;
  const int tid = threadIdx.x, nl = a.nl, kpt = (nl + 1023) / 1024;
  int loc[4] = {0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = kpt * tid + q;
    if (q >= kpt || e >= nl) continue;
    loc[q] = scan ? align_keyscan(a, e) : a.tot[e];
    if (scan) a.tot[e] = loc[q];
  }
  align_scan(a, loc, kpt, ps, hv);
  for (int e = tid; e <= nl; e += 1024) a.pad[e] = ps[e];
}

// sorted_rows: the row at every position that holds one, the sentinel R elsewhere (past a key's rows inside its padded
// range and past num_padded; with `order` positions past num_padded are left alone, no block reads them).
__global__ __launch_bounds__(256) void align_place_kernel(PlanArgs a) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p < a.P) {
    const int e = a.block_expert[p / a.bm];
    if (e < 0 ? a.order == nullptr : p - a.pad[e] >= a.tot[e]) a.sorted_rows[p] = (int32_t)a.R;
  }
  if (p < a.R) {
    const int v = a.le[p], key = v >= 0 && v < a.nl ? v : a.nl;
    if (key < a.nl) a.sorted_rows[a.pad[key] + a.chunk[p / kAlignChunk * a.nl + key] + a.rank[p]] = (int32_t)p;
  }
}

// The whole plan in one workgroup (R and num_local up to kAlignChunk).
template <bool IDS>
__global__ __launch_bounds__(kAlignChunk) void align_small_kernel(PlanArgs a) {
  extern __shared__ int sm_small[];  // [2][nl + 1] ints, [nl] totals, then the per-wave counts
  const int tid = threadIdx.x, nl = a.nl, nk = nl + 2;
  int* ps = sm_small;
  int* hv = ps + nl + 1;
  int* tot = hv + nl + 1;
  uint8_t* cnt = reinterpret_cast<uint8_t*>(tot + nl);
  const int key = align_key<IDS>(a, tid);
  const int r = align_rank(key, nk, cnt);
  if (IDS && tid < a.R) a.local[tid] = key < nl ? key : -1;
  int loc[4] = {0, 0, 0, 0};
  if (tid < nl) tot[tid] = loc[0] = align_count_of(cnt, nk, tid);
  align_scan(a, loc, 1, ps, hv);
  // the sentinel behind every key's rows (a wave for its 64 keys, one key after the other), and past the last one
  const int p0 = tid < nl ? ps[tid] + tot[tid] : 0, p1 = tid < nl ? ps[tid + 1] : 0, lane = tid & 63;
  for (uint64_t todo = __ballot(p0 < p1); todo; todo &= todo - 1) {
    const int src = (int)__builtin_ctzll(todo);
    const int q1 = __builtin_amdgcn_readlane(p1, src);
    for (int p = __builtin_amdgcn_readlane(p0, src) + lane; p < q1; p += 64) a.sorted_rows[p] = (int32_t)a.R;
  }
  if (!a.order)
    for (int64_t p = ps[nl] + tid; p < a.P; p += kAlignChunk) a.sorted_rows[p] = (int32_t)a.R;
  if (key < nl) a.sorted_rows[ps[key] + r] = tid;
}

// The keys' offsets are taken inside the scanning workgroup up to 1024 keys (one a thread) and this many counts, by a launch
// of their own past that. Measured (us, whole plan, inside / own launch): 512 keys x 49 chunks 13.3 / 17.0, 1024 x 49 17.0 /
// 18.4, 1024 x 81 20.7 / 19.4, 1024 x 196 32.9 / 25.2; 2000 x 2 16.5 / 16.5, 2000 x 20 23.2 / 17.4, 4096 x 1 21.6 / 18.7,
// 4096 x 81 158 / 27 (seven launches before: 43).
constexpr int64_t kScanCounts = 1 << 16;

static hipError_t launch_plan(PlanArgs a, int32_t* scratch, hipStream_t st) {
  a.nch = (int)((a.R + kAlignChunk - 1) / kAlignChunk);
  a.rank = scratch;
  a.chunk = a.rank + a.R;
  a.pad = a.chunk + (int64_t)a.nch * a.nl;
  a.tot = a.pad + a.nl + 1;
  const bool ids = a.le == nullptr;
  const size_t cnt = (size_t)kAlignWaves * (a.nl + 2);
  if (a.R <= kAlignChunk && a.nl <= kAlignChunk) {
    const size_t lds = (size_t)(3 * a.nl + 2) * 4 + cnt;
    if (ids) hipLaunchKernelGGL(align_small_kernel<true>, dim3(1), dim3(kAlignChunk), lds, st, a);
    else hipLaunchKernelGGL(align_small_kernel<false>, dim3(1), dim3(kAlignChunk), lds, st, a);
    return hipGetLastError();
  }
  if (a.nch > 0) {
    // up to 64 KB and a little more with 4096 experts
    KernelCfg cfg;
    hipError_t e = kernel_cfg(reinterpret_cast<const void*>(align_count_kernel<true>), kAlignChunk, 72 * 1024, &cfg);
    if (e == hipSuccess)
      e = kernel_cfg(reinterpret_cast<const void*>(align_count_kernel<false>), kAlignChunk, 72 * 1024, &cfg);
    if (e != hipSuccess) return e;
    if (ids) hipLaunchKernelGGL(align_count_kernel<true>, dim3(a.nch), dim3(kAlignChunk), cnt, st, a);
    else hipLaunchKernelGGL(align_count_kernel<false>, dim3(a.nch), dim3(kAlignChunk), cnt, st, a);
  }
  const bool scan = a.nl <= 1024 && (int64_t)a.nch * a.nl <= kScanCounts;
  if (!scan) hipLaunchKernelGGL(align_keyscan_kernel, dim3((a.nl + 63) / 64), dim3(64), 0, st, a);
  hipLaunchKernelGGL(align_scan_kernel, dim3(1), dim3(1024), (size_t)(2 * a.nl + 2) * 4, st, a, scan ? 1 : 0);
  if (ids) a.le = a.local;
  const int64_t n = a.P > a.R ? a.P : a.R;
  if (n > 0) hipLaunchKernelGGL(align_place_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_moe_align(const AlignArgs& q, hipStream_t st) {
  PlanArgs a{};
  a.le = q.local_expert;
  a.R = q.R;
  a.nl = q.num_local;
  a.bm = q.block_m;
  a.P = padded_rows(q.R, q.num_local, q.block_m);
  a.nb = a.P / q.block_m;
  a.sorted_rows = q.sorted_rows;
  a.block_expert = q.block_expert;
  a.num_padded = q.num_padded;
  // no rows: nothing is read through le, which may be null
  if (q.R == 0) a.le = reinterpret_cast<const int32_t*>(q.scratch);
  return launch_plan(a, q.scratch, st);
}

// M blocks a plan of R rows over E experts can have: an expert with rows fills its rows / kBM whole blocks and at most
// one more.
static int64_t mblock_bound(int64_t R, int E) { return (R < E ? R : E) + R / kPrefillBlockM; }

int64_t resident_plan_blocks(int64_t R, int E) { return mblock_bound(R, E); }

hipError_t launch_resident_plan(const ResidentPlan& q, hipStream_t st) {
  PlanArgs a{};
  a.ids = q.ids;
  a.map = q.map;
  a.map_base = q.map_base;
  a.map_len = q.map_len;
  a.slot_ptr = q.slot_ptr;
  a.n_slots = q.n_slots;
  a.local = q.local;
  a.err = q.err;
  a.R = q.R;
  a.nl = q.E;
  a.bm = kPrefillBlockM;
  a.nb = mblock_bound(q.R, q.E);
  a.P = a.nb * kPrefillBlockM;
  a.sorted_rows = q.sorted_rows;
  a.block_expert = q.block_expert;
  a.num_padded = q.num_padded;
  a.order = q.order;
  return launch_plan(a, q.scratch, st);
}

// ---------------------------------------------------------------- grouped GEMM
// Block: 256 threads (4 waves) x 128 sorted rows (one expert) x `tpb` tiles of 64 NB weight rows, K in steps of 128 (two
// quantisation groups). Each wave owns 16 NB weight rows of a tile (NB 16-column MFMA B fragments) for all rows of the
// block, so every weight is dequantized exactly once, by the wave that multiplies it, straight into MFMA B registers.
// Gate/up: the first NB / 2 fragments are gate rows, the others the same up rows, so silu(g) * u is formed in
// registers. Column n of fragment j is the wave's weight row NB n + j (gate/up: h column (NB / 2) n + j % (NB / 2)), so
// a lane's fragments hold adjacent outputs and the epilogues store whole pieces.
// K order inside a step: its two groups one after the other, each in MFMA slices 0, 1; lane quad q (lane >> 4) of slice s
// holds elements 16 q + 8 s .. + 7 of the group (packed word 2q + s), of the weight row and of the activation rows alike.
// That is the dense GEMM's order, the same for every tile shape and every number of live rows, so a row's bits depend on
// that row and its record only. A quad loads 16 bytes (four words of one group: quads 0, 1, 2, 3 words 0-3 of the first,
// 0-3 of the second, 4-7 of the first, 4-7 of the second) and neighbouring quads exchange two words by v_permlane16_swap
// (their nibbles: the words sit in a loaded quadruple, which the exchange would copy first; layer at 333 tokens 175.5 us
// against 176.9, 8192 962 against 965). Whole 16-byte pieces in K order, without the exchange, save 1 % of a layer but sum in
// another order; two 8-byte loads instead of the exchange cost 5-9 % of a layer (2048 tokens 302 -> 324 us, 19 tokens
// 69 -> 75).
// Memory paths:
//  * A (activations for gate/up, h for down): direct global -> LDS loads of 16 bytes per lane (four whole 256-byte row
//    pieces per instruction), double-buffered; only the live 16-row fragments are loaded. The two stages are separate
//    LDS objects, so the compiler knows that a pending load into one does not touch reads of the other. 16-byte chunk
//    c of row m sits at chunk position c ^ a_swz(m), the lane that loads a position reads the chunk that belongs
//    there, and the 16 lanes one ds_read_b128 phase serves fall on distinct banks (3.2 M conflict cycles per gate/up
//    launch at 8192 tokens, 1.5 % of the CU cycles).
//  * Packed weights: 16 bytes per lane per step straight into registers, one stage ahead.
//  * Scales and biases: 8 groups (4 steps) of the wave's own rows at a time, direct to LDS, loaded once the last
//    step of the previous 8 groups has read its values.
// A stage holds KS steps: KS rises as the live rows fall (the loads of one stage are in flight while the previous one
// is computed, and a light stage has little to compute), at the same LDS bytes.
// What bounds it (MI355X, inside a layer, 512 experts top-10, counters over the SIMD cycles): at 8192 tokens (H 2048 / I 512)
// gate/up takes 442-450 us, 764-778 TFLOP/s, the matrix units busy 41 % and other VALU (19 instructions per 8 nibbles, most
// of it) 42 %, LDS 15 %; two waves a SIMD overlap the two only in part (ordering one slice's dequantisation between the MFMAs of
// the slice before, with or without wave priorities, changes nothing). 2048 tokens 29 and 37 % with 1.5 waves a SIMD, 333
// tokens (H 2560 / I 640) 14 and 38 %: the dequantisation of records that few rows share, and the launch's tail. The down
// product at 8192 tokens writes 671 MB of out_rows: 297 us. The former kernel (64-wide K steps, activations through
// registers, a barrier per 64 K, four fragments always): gate/up and down 473 + 347 us at 8192 tokens, 165 + 110 at 2048 (now
// 145-159 + 93-99), 28 + 17 at 19 (now 22 + 14).
constexpr int kBM = 128;
constexpr int kStepK = 128;          // K per step: two quantisation groups
constexpr int kRowB = kStepK * 2;    // bytes of one activation row per step
constexpr int kAStage = kBM * kRowB; // one LDS stage of activations: 32 KB
constexpr int kSbG = 8;              // groups per (s, b) table chunk

typedef __bf16 ss_bf16x2 __attribute__((ext_vector_type(2)));
typedef float ss_f32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void ss_lds_void;

// bf16 pair (lo, hi) rounded to nearest even by the hardware conversion.
SS_DEV uint32_t cvt_pk_bf16(float lo, float hi) {
  const ss_bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// 8 nibbles (element e at bits 4e) -> bf16(q * s + b) x 8 as an MFMA operand (pairs low element first).
// A nibble q in a byte of its own is the OCP fp8 e4m3 value q * 2^-9 exactly (q < 8 subnormal, q >= 8 with
// exponent field 1), so one v_cvt_pk_f32_fp8 turns two nibbles into fp32. s9 = s * 2^9 (exact), hence
// (q * 2^-9) * s9 = q * s exactly and the fused multiply-add rounds q * s + b once, as the reference's fp32
// q * s + b does (q * s is exact in fp32: 4-bit by 8-bit mantissas); then one rounding to bf16. (A scale of 2^119
// or more would overflow s9; bf16 weight scales are far below that.) The masks are opaque to the compiler, so it
// keeps them as two v_and_b32 instead of folding them into per-nibble bit-field extracts.
SS_DEV uint32_t and_opaque(uint32_t x, uint32_t m) {
  uint32_t r;
  asm("v_and_b32 %0, %1, %2" : "=v"(r) : "s"(m), "v"(x));
  return r;
}
struct ss_nibbles {
  uint32_t lo, hi;  // n0 n2 n4 n6 / n1 n3 n5 n7, one to a byte
};
SS_DEV ss_nibbles nibbles_of(uint32_t w) { return {and_opaque(w, 0x0F0F0F0Fu), and_opaque(w >> 4, 0x0F0F0F0Fu)}; }
// Lanes of odd quads of a with lanes of even quads of b.
SS_DEV void quad_exchange(ss_nibbles& a, ss_nibbles& b) {
  const auto l = __builtin_amdgcn_permlane16_swap(a.lo, b.lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(a.hi, b.hi, false, false);
  a.lo = l[0];
  b.lo = l[1];
  a.hi = h[0];
  b.hi = h[1];
}
SS_DEV ss_u32x4 dequant8(const ss_nibbles& w, float s9, float bi) {
  const int lo = (int)w.lo, hi = (int)w.hi;
  const auto e02 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, false), e46 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, true);
  const auto e13 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false), e57 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
  ss_u32x4 r;
  r.x = cvt_pk_bf16(__builtin_fmaf(e02[0], s9, bi), __builtin_fmaf(e13[0], s9, bi));
  r.y = cvt_pk_bf16(__builtin_fmaf(e02[1], s9, bi), __builtin_fmaf(e13[1], s9, bi));
  r.z = cvt_pk_bf16(__builtin_fmaf(e46[0], s9, bi), __builtin_fmaf(e57[0], s9, bi));
  r.w = cvt_pk_bf16(__builtin_fmaf(e46[1], s9, bi), __builtin_fmaf(e57[1], s9, bi));
  return r;
}

// out_rows larger than the memory-side cache (256 MB) leave by non-temporal stores: the combine finds them in memory
// either way, and they no longer push the packed weights and h out of the caches. Smaller ones stay plain, so that the
// combine reads them from that cache. Measured (layer, us, plain / non-temporal, two runs of each in turn within 0.2 %,
// H 2048): 3300 tokens (270 MB) 479 / 471, 4096 557 / 548, 5500 708 / 695, 8192 986 / 973; 2600 at H 2560 (266 MB) level,
// 566 / 566; below the line, in an earlier measurement, 2048 (168 MB) 310 / 316.
constexpr int64_t kStreamBytes = 256ll << 20;

struct GemmArgs {
  const uint16_t* a;           // gate/up: x bf16 [T, H]; down: h bf16 [R, I]
  const int32_t* row_token;    // [R] (gate/up)
  const float* row_weight;     // [R] (down)
  const int32_t* sorted_rows;  // [P]
  const int32_t* block_expert; // [P / kBM]
  const int32_t* num_padded;   // [1]
  const int64_t* group_ptr;    // [num_local] record base addresses
  const MBlock* order;         // null, or the M blocks in launch order (then block_expert and group_ptr are unused)
  int topk;                    // with row_token null: row r belongs to token r / topk
  uint16_t* h;                 // gate/up output bf16 [R, I]
  float* out_rows;             // down output fp32 [R, H]
  int64_t R;
  int T, H, I;
  bool stream_out;                 // down: out_rows by non-temporal stores
  int64_t w_off, s_off, b_off;     // gate (or down) pieces
  int64_t w2_off, s2_off, b2_off;  // up pieces (gate/up)
  uint64_t* trace;                 // per-block stamps (start, end, expert << 32 | valid rows, XCC << 32 | HW_ID) or null
};

// LDS barrier for data exchanged through LDS: waits for this wave's LDS operations only. (Fences would also wait for its
// stores to memory: the compiler cannot tell them from pending loads into LDS.)
SS_DEV void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Block index -> (M block, group of N tiles). The M blocks are dealt round-robin to the XCDs (workgroup b runs on XCD
// b % 8), in launch order (plan order for a caller's plan), so every XCD gets an even share of the heavy and the light
// experts' blocks; each XCD takes all N tiles of one M block in a row (they share its activation rows in the XCD's L2).
// Measured on MI355X with the former kernel, contiguous per-XCD ranges of the plan end 140-180 us apart at 2048 tokens,
// and groups of 2, 4 or 8 M blocks per XCD (for the weights they share) change nothing.
SS_DEV bool xcd_tile(int mb, int nt, int& pid_m, int& pid_n) {
  const int b = blockIdx.x, x = b & 7, s = b >> 3;
  const int sm = s / nt;
  pid_m = sm * 8 + x;
  pid_n = s - sm * nt;
  return pid_m < mb;
}

// Every load of this wave issued so far has landed (vmcnt 0; the other counters are left alone). The builtin and not an
// asm statement: the compiler counts it, so it adds no wait of its own where the loaded registers are read, behind
// stores that were issued in between.
SS_DEV void wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" ::: "memory");
}

// Chunk swizzle of activation row m (see above): ds_read_b128 serves lanes 0-3 and 12-15 of one quad with lanes 4-11 of
// its neighbour; both quads' chunk numbers of a slice lie in the same half, so rows 4-11 (mod 16) take the other half of
// the positions.
SS_DEV int a_swz(int m) { return (m & 3) | ((m >> 1) & 4) | (((m << 1) ^ m) & 8); }

constexpr int kZeroRow = (int)0x80000000u;  // a row whose activations are zero (it reads row 0; its h is stored as 0)

struct GemmSmem {
  int a_row[kBM];    // activation row of each position, or kZeroRow
  int out_row[kBM];  // row of h / out_rows, -1 past the valid rows
  float wt[kBM];
};

// `ntile` N tiles from tile0 for the block's NF live 16-row fragments, KS K-steps per LDS stage.
template <bool GU, int NB, int NF, int KS>
SS_DEV void gemm_tiles(const GemmArgs& g, const GemmSmem& sm, uint8_t* a0, uint8_t* a1, uint8_t* lss, uint8_t* lsb,
                       const uint8_t* base, int tile0, int ntile) {
  static_assert(NF * KS <= 8 && (KS == 1 || KS == 2 || KS == 4), "a stage holds kAStage bytes; its chunk is loaded whole");
  constexpr int TN = 64 * NB, HB = NB / 2;  // weight rows per tile; gate (and up) fragments per wave
  constexpr int NQ = NF > 4 ? 2 : NF;       // A fragments read ahead of their MFMAs
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int kdim = GU ? g.H : g.I;
  const int nsteps = kdim / kStepK, G = kdim / 64;
  const int nst = (nsteps + KS - 1) / KS;  // stages per tile
  const int wrow_b = kdim / 2;             // bytes of a packed weight row
  const uint32_t arow_b = kdim * 2;
  // Activations: load instruction c of wave w covers rows 16 c + 4 w + q, position n of each.
  const int ar = 4 * w + q;
  const uint8_t* abase = reinterpret_cast<const uint8_t*>(g.a) + 16 * (n ^ a_swz(ar));
  // Lane offset of fragment 0's 16 bytes from the tile's first row; fragment j adds a uniform offset.
  // Quads 0 and 2 take the pieces of the step's first group, quads 1 and 3 those of its second.
  const uint32_t lw =
      (uint32_t)((GU ? 8 * NB * w + HB * n : 16 * NB * w + NB * n) * wrow_b + 16 * ((q >> 1) | (q & 1) << 1));
  const int64_t tile_w = (int64_t)(GU ? TN / 2 : TN) * wrow_b, tile_s = (int64_t)(GU ? TN / 2 : TN) * G * 2;
  // (s, b) table: lane (q, n) of wave w fills slot 64 w + lane with its wave's row of fragment q (lanes past NB repeat
  // the last fragment's), so a fragment's 16 rows are adjacent slots.
  const int jq = q < NB ? q : NB - 1;
  const bool s_up = GU && jq >= HB;
  const int srow = GU ? 8 * NB * w + HB * n + (jq & (HB - 1)) : 16 * NB * w + NB * n + jq;
  const uint8_t* sptr = base + (s_up ? g.s2_off : g.s_off) + (int64_t)srow * G * 2;
  const uint32_t sb_dist = (uint32_t)(g.b_off - g.s_off);  // from a row's scales to its biases
  // Rows of a multiple of 8 groups are 16-byte aligned: a slot is 16 bytes (8 groups). Otherwise (an odd number of
  // steps) pairs of groups load as dwords: pair p of a slot at 256 p + 4 slot.
  const bool wide = G % 8 == 0;

  uint4 bw[2][KS][NB];
  auto load = [&](int tile, int st, auto p_c) {
    constexpr int P = decltype(p_c)::value;
    uint8_t* ad = P ? a1 : a0;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const int k = st * KS + u;
      if (KS == 1 || k < nsteps) {
#pragma unroll
        for (int c = 0; c < NF; ++c) {
          const uint32_t row = (uint32_t)sm.a_row[16 * c + ar] & 0x7FFFFFFFu;
          __builtin_amdgcn_global_load_lds(abase + k * kRowB + (uint64_t)row * arow_b,
                                           (ss_lds_void*)(ad + (u * NF * 16 + 16 * c + 4 * w) * kRowB), 16, 0, 0);
        }
        uint32_t lv = lw;
        asm volatile("" : "+v"(lv));  // the addresses are formed here, not kept in registers over the loop
        const uint8_t* wt = base + tile * tile_w + 64 * k;
#pragma unroll
        for (int j = 0; j < NB; ++j)
          bw[P][u][j] = ldg16(wt + (GU && j >= HB ? g.w2_off : g.w_off) + (int64_t)(GU ? j & (HB - 1) : j) * wrow_b + lv);
      }
    }
  };
  // groups g0 .. g0 + 7 of the tile's rows into this wave's slots
  auto load_sb = [&](int tile, int g0) {
    const uint8_t* p = sptr + tile * tile_s + 2 * g0;
    if (wide) {
      __builtin_amdgcn_global_load_lds(p, (ss_lds_void*)(lss + 1024 * w), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(p + sb_dist, (ss_lds_void*)(lsb + 1024 * w), 16, 0, 0);
    } else {
#pragma unroll
      for (int d = 0; d < kSbG / 2; ++d)
        if (g0 + 2 * d < G) {
          __builtin_amdgcn_global_load_lds(p + 4 * d, (ss_lds_void*)(lss + 1024 * w + 256 * d), 4, 0, 0);
          __builtin_amdgcn_global_load_lds(p + sb_dist + 4 * d, (ss_lds_void*)(lsb + 1024 * w + 256 * d), 4, 0, 0);
        }
    }
  };
  const int sb_lane = 1024 * w + (wide ? 16 : 4) * n;
  const int sb_j = wide ? 256 : 64, sb_k = wide ? 4 : 256;

  ss_f32x4 acc[NF][NB];
  auto zero = [&]() {
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // Stage st from LDS stage / register set P. When the stage is the last to read the table chunk (`chunk`), its
  // (s, b) values are all in registers before the next chunk (tile ct, group cg) is requested into the same slots.
  auto compute = [&](int st, auto p_c, bool chunk, int ct, int cg) {
    constexpr int P = decltype(p_c)::value;
    const uint8_t* as = (P ? a1 : a0) + n * kRowB;
    int apos = 16 * ((2 * q) ^ a_swz(n));
    asm volatile("" : "+v"(apos));
    uint32_t sp[KS][NB], bp[KS][NB];  // the step's two groups, the first in the low half
#pragma unroll
    for (int u = 0; u < KS; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int at = sb_lane + j * sb_j + ((st * KS + u) & (kSbG / 2 - 1)) * sb_k;
        sp[u][j] = *reinterpret_cast<const uint32_t*>(lss + at);
        bp[u][j] = *reinterpret_cast<const uint32_t*>(lsb + at);
      }
    if (chunk) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      load_sb(ct, cg);
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (u > 0 && st * KS + u >= nsteps) break;
      // Neighbouring quads exchange two words: each then holds words 2 q, 2 q + 1 of the first group, then of the second.
      ss_nibbles wd[4][NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const uint4 v = bw[P][u][j];
        wd[0][j] = nibbles_of(v.x);
        wd[2][j] = nibbles_of(v.z);
        quad_exchange(wd[0][j], wd[2][j]);
        wd[1][j] = nibbles_of(v.y);
        wd[3][j] = nibbles_of(v.w);
        quad_exchange(wd[1][j], wd[3][j]);
      }
      float sc[NB], bi[NB];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s % 2 == 0) {
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            sc[j] = __uint_as_float(s ? sp[u][j] & 0xFFFF0000u : sp[u][j] << 16) * 512.f;  // s * 2^9
            bi[j] = __uint_as_float(s ? bp[u][j] & 0xFFFF0000u : bp[u][j] << 16);
          }
        }
        ss_u32x4 bf[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) bf[j] = dequant8(wd[s][j], sc[j], bi[j]);
        // A fragments a few at a time: the scheduling barriers keep their registers few; the two waves of a SIMD
        // overlap one wave's dequantisation and LDS reads with the other's MFMAs.
        const uint8_t* ap = as + u * NF * 16 * kRowB + (apos ^ (16 * ((s & 1) | (s & 2) << 2)));
#pragma unroll
        for (int i0 = 0; i0 < NF; i0 += NQ) {
          ss_u32x4 av[NQ];
#pragma unroll
          for (int i = 0; i < NQ; ++i) av[i] = *reinterpret_cast<const ss_u32x4*>(ap + (i0 + i) * 16 * kRowB);
#pragma unroll
          for (int i = 0; i < NQ; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i0 + i][j] = ss_mfma(av[i], bf[j], acc[i0 + i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  auto epilogue_as = [&](int tile, auto stream_c) {
    constexpr bool STREAM = decltype(stream_c)::value;
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * q + r;
        const int orow = sm.out_row[m];
        if (orow < 0) continue;
        if (GU) {
          const bool live = sm.a_row[m] >= 0;
          uint32_t hp = 0;
#pragma unroll
          for (int j = 0; j < HB; ++j) {
            const float gv = acc[i][j][r], uv = acc[i][j + HB][r];
            // silu with the hardware exp2 and reciprocal (about 1 ulp each): h is rounded to bf16 next, which
            // hides fp32 differences of a few ulp except at a rounding tie.
            const float sig = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gv * -1.4426950408889634f));
            const float hv = live ? gv * sig * uv : 0.f;
            hp |= (uint32_t)ss_f32_to_bf16(hv) << (16 * j);
          }
          uint16_t* hd = g.h + (int64_t)orow * g.I + tile * (TN / 2) + 8 * NB * w + HB * n;
          if constexpr (NB == 4) *(SS_G uint32_t*)hd = hp;
          else *(SS_G uint16_t*)hd = (uint16_t)hp;
        } else {
          const float wt = sm.wt[m];
          float* od = g.out_rows + (int64_t)orow * g.H + tile * TN + 16 * NB * w + NB * n;
          if constexpr (NB == 4) {
            const ss_f32x4 v = {acc[i][0][r] * wt, acc[i][1][r] * wt, acc[i][2][r] * wt, acc[i][3][r] * wt};
            if constexpr (STREAM) __builtin_nontemporal_store(v, (SS_G ss_f32x4*)od);
            else *(SS_G ss_f32x4*)od = v;
          } else {
            *(SS_G ss_f32x2*)od = ss_f32x2{acc[i][0][r] * wt, acc[i][1][r] * wt};
          }
        }
      }
  };
  auto epilogue = [&](int tile) {
    if constexpr (!GU && NB == 4)
      if (g.stream_out) return epilogue_as(tile, std::true_type{});
    epilogue_as(tile, std::false_type{});
  };

  zero();
  int tile = tile0, st = 0;
  const int nall = ntile * nst;
  constexpr int SPC = kSbG / 2 / KS;  // stages per table chunk
  load_sb(tile, 0);
  load(tile, 0, std::integral_constant<int, 0>{});
  wait_loads();
  lds_barrier();
  // Stage f of all tiles: the next stage's loads, this stage's MFMAs, the wait for those loads, the tile's epilogue
  // behind its last stage (its stores drain under the next stage: without this the non-temporal ones cost time,
  // 979 -> 986 us at 8192 tokens), then the barrier, so that every wave's loads have
  // landed.
  auto stage = [&](int f, auto p_c) {
    constexpr int P = decltype(p_c)::value;
    int t2 = tile, s2 = st + 1;
    if (s2 == nst) {
      s2 = 0;
      ++t2;
    }
    const bool more = f + 1 < nall;
    if (more) load(t2, s2, std::integral_constant<int, P ^ 1>{});
    __builtin_amdgcn_sched_barrier(0);
    compute(st, p_c, more && s2 % SPC == 0, t2, s2 * KS * 2);
    __builtin_amdgcn_sched_barrier(0);
    wait_loads();
    if (st == nst - 1) {
      epilogue(tile);
      zero();
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) lds_barrier();
    tile = t2;
    st = s2;
  };
#pragma unroll 1
  for (int f = 0; f < nall; f += 2) {
    stage(f, std::integral_constant<int, 0>{});
    if (f + 1 < nall) stage(f + 1, std::integral_constant<int, 1>{});
  }
}

template <bool GU, int NB>
__global__ __launch_bounds__(256, 2) void prefill_gemm_kernel(GemmArgs g, int nt, int tpb) {
  __shared__ __attribute__((aligned(256))) uint8_t a0[kAStage];
  __shared__ __attribute__((aligned(256))) uint8_t a1[kAStage];
  __shared__ __attribute__((aligned(256))) uint8_t lss[4096];
  __shared__ __attribute__((aligned(256))) uint8_t lsb[4096];
  __shared__ GemmSmem sm;
  const int tid = threadIdx.x;
  const int mb = g.num_padded[0] / kBM;
  int pid_m, pid_n;
  if (!xcd_tile(mb, nt, pid_m, pid_n)) return;
  int e;
  const uint8_t* base;
  if (g.order) {
    const MBlock b = g.order[pid_m];
    e = b.expert;
    pid_m = b.index;
    base = reinterpret_cast<const uint8_t*>(b.record);
  } else {
    e = g.block_expert[pid_m];
    if (e < 0) return;
    base = reinterpret_cast<const uint8_t*>(g.group_ptr[e]);
  }
  const uint64_t t_start = g.trace ? __builtin_amdgcn_s_memrealtime() : 0;
  bool valid = false;
  if (tid < kBM) {
    const int r = g.sorted_rows[(int64_t)pid_m * kBM + tid];
    valid = r < g.R;
    int row = kZeroRow;
    if (valid) {
      if (GU) {
        const int t = g.row_token ? g.row_token[r] : (int)((uint32_t)r / (uint32_t)g.topk);
        if (t >= 0 && t < g.T) row = t;
      } else {
        row = r;
      }
    }
    sm.a_row[tid] = row;
    sm.out_row[tid] = valid ? r : -1;
    if (!GU) sm.wt[tid] = valid ? g.row_weight[r] : 0.f;
  }
  // Valid rows are a prefix of the block (each expert's rows come first in its padded range).
  const int nvalid = __syncthreads_count(valid);
  const int nf = (nvalid + 15) >> 4;  // live fragments (1..8)
  const int tile0 = pid_n * tpb;
  constexpr int KL = NB == 4 ? 2 : 4;  // with four fragments, four steps of weights do not fit the registers
  if (nf > 6) gemm_tiles<GU, NB, 8, 1>(g, sm, a0, a1, lss, lsb, base, tile0, tpb);
  else if (nf > 4) gemm_tiles<GU, NB, 6, 1>(g, sm, a0, a1, lss, lsb, base, tile0, tpb);
  else if (nf > 2) gemm_tiles<GU, NB, 4, 2>(g, sm, a0, a1, lss, lsb, base, tile0, tpb);
  else if (nf > 1) gemm_tiles<GU, NB, 2, KL>(g, sm, a0, a1, lss, lsb, base, tile0, tpb);
  else gemm_tiles<GU, NB, 1, KL>(g, sm, a0, a1, lss, lsb, base, tile0, tpb);
  // Diagnostics: gate/up blocks at entries [0, 8192), down blocks at [8192, 16384), four per block.
  if (g.trace && tid == 0) {
    const size_t at = (GU ? 0 : 8192) + 4 * (size_t)blockIdx.x;
    if (at + 4 <= (GU ? 8192u : 16384u)) {
      const uint32_t hw = __builtin_amdgcn_s_getreg(4 | (31 << 11));   // HW_ID
      const uint32_t xcc = __builtin_amdgcn_s_getreg(20 | (31 << 11)); // XCC_ID
      g.trace[at] = t_start;
      g.trace[at + 1] = __builtin_amdgcn_s_memrealtime();
      g.trace[at + 2] = ((uint64_t)(uint32_t)e << 32) | (uint32_t)nvalid;
      g.trace[at + 3] = ((uint64_t)xcc << 32) | hw;
    }
  }
}

template <bool GU>
static void launch_gemm(const GemmArgs& g, int nb, int tpb, int64_t mb, hipStream_t st) {
  const int rows = GU ? g.I : g.H, tn = GU ? 32 * nb : 64 * nb;
  const int nt = rows / tn / tpb;
  const dim3 grid((unsigned)(8 * nt * ((mb + 7) / 8)));
  if (nb == 4) hipLaunchKernelGGL((prefill_gemm_kernel<GU, 4>), grid, dim3(256), 0, st, g, nt, tpb);
  else hipLaunchKernelGGL((prefill_gemm_kernel<GU, 2>), grid, dim3(256), 0, st, g, nt, tpb);
}

hipError_t launch_prefill_gemm(const PrefillArgs& p, hipStream_t st) {
  static_assert(kBM == kPrefillBlockM, "one block size for the plan and the GEMM");
  const SsRecord rec = ss_record_layout(p.H, p.I);
  if (p.R == 0) return hipSuccess;
  GemmArgs g{};
  g.row_token = p.row_token;
  g.row_weight = p.row_weight;
  g.sorted_rows = p.sorted_rows;
  g.block_expert = p.block_expert;
  g.num_padded = p.num_padded;
  g.group_ptr = p.group_ptr;
  g.order = p.order;
  g.topk = p.topk;
  g.h = p.h_buf;
  g.out_rows = p.out_rows;
  g.R = p.R;
  g.T = p.T;
  g.H = p.H;
  g.I = p.I;
  g.trace = p.trace;
  // With no token at all every row is a zero row, whose (unused) activations still come from a readable row.
  g.a = p.T > 0 ? p.x : reinterpret_cast<const uint16_t*>(p.out_rows);
  g.w_off = rec.gw;
  g.s_off = rec.gs;
  g.b_off = rec.gb;
  g.w2_off = rec.uw;
  g.s2_off = rec.us;
  g.b2_off = rec.ub;
  // Grids cover the M blocks a plan can have (rounded up to a multiple of 8) times the N tiles; blocks past the
  // device-side count exit at once. The library's own plan has no block without rows and at most one partial block per
  // expert; a caller's may have any number of blocks that padded_rows holds.
  const int64_t mb = p.order ? mblock_bound(p.R, p.num_local) : padded_rows(p.R, p.num_local, kBM) / kBM;
  // Tiles: with few rows per expert most M blocks are light and the chip is short of blocks, so a wave takes two
  // weight fragments instead of four (twice the blocks); with more rows the wider wave reads its activations from LDS
  // half as often. Measured with 512 experts (us, two / four fragments): gate/up R = 190 24 / 27, 3330 (H 2560 /
  // I 640) 85 / 90, 6000 67 / 72, 20480 139 / 124; down R = 190 15 / 17, 480 20 / 20, 3330 55 / 54, 6000 48 / 43.
  // Two down tiles per block (one prologue) pay off once there are blocks to spare: R = 6000 43 / 43, 10000 (H 2560)
  // 95 against 101 with one, 81920 280 against 300.
  const int nb_gu = p.R < 16 * (int64_t)p.num_local ? 2 : 4, nb_d = p.R < 2 * (int64_t)p.num_local ? 2 : 4;
  const int td = p.R >= 8192 && p.H % 512 == 0 ? 2 : 1;
  g.stream_out = p.R * p.H * 4 > kStreamBytes;
  launch_gemm<true>(g, nb_gu, 1, mb, st);
  g.a = p.h_buf;
  g.w_off = rec.dw;
  g.s_off = rec.ds;
  g.b_off = rec.db;
  launch_gemm<false>(g, nb_d, td, mb, st);
  return hipGetLastError();
}

// ---------------------------------------------------------------- combine_rank_order (fused_moe_affine.py:164-172)
// With LAYER also y = bf16(bf16(out) + bf16(bf16(sigmoid(sgl)) * sh)), the roundings of combine_shared_kernel, so the
// sums are not read back (at 8192 tokens the two launches took 160 + 22 us, this one 132). Bound by HBM: T K H 4 bytes
// in, read once and non-temporally (layer, us, plain / non-temporal loads, two runs each: 333 tokens at H 2560 level, 2600
// at H 2560 575 / 566, 2048 326 / 316, 3300 479 / 471, 8192 993 / 973).
template <bool LAYER>
__global__ __launch_bounds__(256) void combine_kernel(const float* __restrict__ rows,
                                                      const int32_t* __restrict__ row_local,
                                                      const uint16_t* __restrict__ sh,
                                                      const uint16_t* __restrict__ sgl, int T, int K, int H,
                                                      float* __restrict__ out, uint16_t* __restrict__ y) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one float4 of one token
  const int h4 = H >> 2;
  if (idx >= (int64_t)T * h4) return;
  const int64_t t = idx / h4, c = idx - t * h4;
  const float4* p = reinterpret_cast<const float4*>(rows) + (t * K) * h4 + c;
  uint2 s2 = make_uint2(0u, 0u);
  float gl = 0.f;
  if (LAYER) {
    s2 = reinterpret_cast<const uint2*>(sh)[idx];
    gl = ss_bf16_to_f32(sgl[t]);
  }
  // Every row is loaded (in bounds) and a skipped row's value replaced by +0 afterwards: a select between a local
  // zero and a loaded value is kept on values, never turned into a load through a selected address.
  auto row = [&](int k) {
    const ss_f32x4 v = __builtin_nontemporal_load((const SS_G ss_f32x4*)(p + (int64_t)k * h4));
    return make_float4(v[0], v[1], v[2], v[3]);
  };
  float4 acc = row(0);
  if (row_local && row_local[t * K] < 0) acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 1; k < K; ++k) {
    const float4 v = row(k);
    const bool skip = row_local && row_local[t * K + k] < 0;
    acc.x = acc.x + (skip ? 0.f : v.x);
    acc.y = acc.y + (skip ? 0.f : v.y);
    acc.z = acc.z + (skip ? 0.f : v.z);
    acc.w = acc.w + (skip ? 0.f : v.w);
  }
  reinterpret_cast<float4*>(out)[idx] = acc;
  if (LAYER) {
    const float sg = ss_round_bf16(1.f / (1.f + ss_expf(-gl)));
    const float rv[4] = {acc.x, acc.y, acc.z, acc.w};
    const uint32_t sv[4] = {s2.x & 0xFFFFu, s2.x >> 16, s2.y & 0xFFFFu, s2.y >> 16};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = ss_f32_to_bf16(ss_round_bf16(rv[e]) + ss_round_bf16(sg * ss_bf16_to_f32(sv[e])));
    reinterpret_cast<uint2*>(y)[idx] = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
  }
}

hipError_t launch_combine(const float* rows, const int32_t* row_local, int T, int K, int H, float* out,
                          hipStream_t st) {
  const int64_t n = (int64_t)T * (H / 4);
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(combine_kernel<false>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rows, row_local,
                     nullptr, nullptr, T, K, H, out, nullptr);
  return hipGetLastError();
}

hipError_t launch_combine_layer(const float* rows, const int32_t* row_local, const uint16_t* sh, const uint16_t* sgl,
                                int T, int K, int H, float* out, uint16_t* y, hipStream_t st) {
  const int64_t n = (int64_t)T * (H / 4);
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(combine_kernel<true>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rows, row_local, sh, sgl,
                     T, K, H, out, y);
  return hipGetLastError();
}

}  // namespace ss
