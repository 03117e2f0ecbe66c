// Prefill MoE: rows sorted into expert-contiguous blocks, a grouped bf16 MFMA GEMM over affine-4bit records
// dequantized into MFMA registers, and the rank-order combine.
//
// Semantics follow kernels/moe_align.py:11-48, kernels/fused_moe_affine.py:39-172 (the reference's prefill path):
//  * moe_align: a stable counting sort of the rows by local expert (rows outside [0, num_local) are skipped); each
//    expert's rows padded to block_m with the sentinel R; every block of block_m positions belongs to one expert.
//    Computed without atomics in any order-dependent place: ranks inside a 256-row chunk by comparison, chunk
//    offsets by a sequential scan per expert.
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
constexpr int kAlignChunk = 256;

int64_t padded_rows(int64_t R, int num_local, int block_m) {
  const int64_t n = R + (int64_t)num_local * (block_m - 1);
  return (n + block_m - 1) / block_m * block_m;
}

// scratch ints: rank [R], chunk offsets [nchunk][num_local], pad_start [num_local + 1], totals [num_local]
int64_t align_scratch_ints(int64_t R, int num_local) {
  const int64_t nch = (R + kAlignChunk - 1) / kAlignChunk;
  return R + nch * num_local + 2 * (int64_t)num_local + 1;
}

SS_DEV int align_key(const int32_t* le, int64_t i, int64_t R, int nl) {
  if (i >= R) return nl + 1;
  const int v = le[i];
  return (v >= 0 && v < nl) ? v : nl;
}

// Per chunk: the rank of each row among the earlier rows of the chunk with the same key, and per-key counts.
// Inside a wave the rank is the number of lower lanes holding the same key (one ballot per distinct key of the
// wave, taken in lane order); the earlier waves of the chunk add their counts of that key from LDS.
__global__ __launch_bounds__(kAlignChunk) void align_count_kernel(const int32_t* __restrict__ le, int64_t R, int nl,
                                                                  int32_t* __restrict__ rank,
                                                                  int32_t* __restrict__ chunk_cnt) {
  extern __shared__ uint8_t sm_cnt[];  // [kAlignChunk / 64 waves][nl + 2]: per-wave counts (<= 64) of every key
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  constexpr int NW = kAlignChunk / 64;
  const int nk = nl + 2;  // keys 0 .. nl + 1 (nl: outside [0, nl), nl + 1: past R)
  const int64_t i = (int64_t)blockIdx.x * kAlignChunk + tid;
  const int key = align_key(le, i, R, nl);
  for (int e = tid; e < NW * nk; e += kAlignChunk) sm_cnt[e] = 0;
  __syncthreads();
  // rank inside the wave: walk the wave's distinct keys in the order of their lowest lane
  int r_in = 0;
  uint64_t todo = ~0ull;
  while (todo) {
    const int l0 = (int)__builtin_ctzll(todo);
    const int k0 = __builtin_amdgcn_readlane(key, l0);
    const uint64_t same = __ballot(key == k0);
    if (key == k0) r_in = __popcll(same & ((1ull << lane) - 1ull));
    if (lane == l0) sm_cnt[w * nk + k0] = (uint8_t)__popcll(same);
    todo &= ~same;
  }
  __syncthreads();
  int r = r_in;
  for (int v = 0; v < w; ++v) r += sm_cnt[v * nk + key];
  if (i < R) rank[i] = r;
  for (int e = tid; e < nl; e += kAlignChunk) {
    int c = 0;
#pragma unroll
    for (int v = 0; v < NW; ++v) c += sm_cnt[v * nk + e];
    chunk_cnt[(int64_t)blockIdx.x * nl + e] = c;
  }
}

__global__ void align_zero_kernel(int nl, int32_t* __restrict__ tot) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < nl) tot[e] = 0;
}

// Per key: exclusive offsets of the key's rows in each chunk (chunk order) and the key's total. One thread per key;
// its nch loads are independent, so they are all in flight at once.
__global__ __launch_bounds__(256) void align_keyscan_kernel(int nl, int nch, int32_t* __restrict__ chunk_cnt,
                                                            int32_t* __restrict__ tot) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= nl) return;
  int run = 0;
  for (int c0 = 0; c0 < nch; c0 += 32) {
    int v[32];
#pragma unroll
    for (int q = 0; q < 32; ++q) v[q] = c0 + q < nch ? chunk_cnt[(int64_t)(c0 + q) * nl + e] : 0;
#pragma unroll
    for (int q = 0; q < 32; ++q) {
      if (c0 + q < nch) chunk_cnt[(int64_t)(c0 + q) * nl + e] = run;
      run += v[q];
    }
  }
  tot[e] = run;
}

// One workgroup: exclusive scan of the padded key sizes -> pad[0 .. nl] (pad[nl] = num_padded), and the expert of
// every block of bm positions (-1 past num_padded).
__global__ __launch_bounds__(1024) void align_padscan_kernel(int nl, int bm, int64_t nb, const int32_t* __restrict__ tot,
                                                             int32_t* __restrict__ pad, int32_t* __restrict__ block_expert,
                                                             int32_t* __restrict__ num_padded) {
  extern __shared__ int ps[];  // [nl + 1]
  __shared__ int part[1024];
  const int tid = threadIdx.x;
  // Each thread sums up to 4 consecutive keys, a Hillis-Steele scan over the 1024 thread totals, then the per-thread
  // prefixes (nl <= 4096).
  int loc[4], sum = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = 4 * tid + q;
    loc[q] = e < nl ? (tot[e] + bm - 1) / bm * bm : 0;
    sum += loc[q];
  }
  part[tid] = sum;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  int run = part[tid] - sum;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = 4 * tid + q;
    if (e < nl) ps[e] = run;
    run += loc[q];
  }
  if (tid == 1023) {
    ps[nl] = part[1023];
    *num_padded = part[1023];
  }
  __syncthreads();
  for (int e = tid; e <= nl; e += 1024) pad[e] = ps[e];
  for (int64_t q = tid; q < nb; q += 1024) {
    const int64_t pos = q * bm;
    // the last key e with ps[e] <= pos (binary search), -1 past the end
    int lo = 0, hi = nl;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (ps[mid] <= pos) lo = mid;
      else hi = mid - 1;
    }
    block_expert[q] = pos < ps[nl] ? lo : -1;
  }
}

// Sentinel R at every position that holds no row: past a key's rows inside its padded range, and past num_padded.
__global__ __launch_bounds__(256) void align_fill_kernel(int64_t R, int nl, int bm, int64_t P,
                                                         const int32_t* __restrict__ pad, const int32_t* __restrict__ tot,
                                                         const int32_t* __restrict__ block_expert,
                                                         int32_t* __restrict__ sorted_rows) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= P) return;
  const int e = block_expert[p / bm];
  if (e < 0 || p - pad[e] >= tot[e]) sorted_rows[p] = (int32_t)R;
}

__global__ __launch_bounds__(kAlignChunk) void align_scatter_kernel(const int32_t* __restrict__ le, int64_t R, int nl,
                                                                    const int32_t* __restrict__ rank,
                                                                    const int32_t* __restrict__ chunk_off,
                                                                    const int32_t* __restrict__ pad,
                                                                    int32_t* __restrict__ sorted_rows) {
  const int64_t i = (int64_t)blockIdx.x * kAlignChunk + threadIdx.x;
  const int key = align_key(le, i, R, nl);
  if (key < nl) sorted_rows[pad[key] + chunk_off[(int64_t)blockIdx.x * nl + key] + rank[i]] = (int32_t)i;
}

hipError_t launch_moe_align(const AlignArgs& a, hipStream_t st) {
  const int nch = (int)((a.R + kAlignChunk - 1) / kAlignChunk);
  int32_t* rank = a.scratch;
  int32_t* chunk = rank + a.R;
  int32_t* pad = chunk + (int64_t)nch * a.num_local;
  int32_t* tot = pad + a.num_local + 1;
  const int64_t P = padded_rows(a.R, a.num_local, a.block_m);
  if (nch > 0) {
    hipLaunchKernelGGL(align_count_kernel, dim3(nch), dim3(kAlignChunk), (size_t)(kAlignChunk / 64) * (a.num_local + 2),
                       st, a.local_expert,
                       a.R, a.num_local, rank, chunk);
    hipLaunchKernelGGL(align_keyscan_kernel, dim3((a.num_local + 255) / 256), dim3(256), 0, st, a.num_local, nch,
                       chunk, tot);
  } else {
    hipLaunchKernelGGL(align_zero_kernel, dim3((a.num_local + 255) / 256), dim3(256), 0, st, a.num_local, tot);
  }
  hipLaunchKernelGGL(align_padscan_kernel, dim3(1), dim3(1024), (size_t)(a.num_local + 1) * 4, st, a.num_local,
                     a.block_m, P / a.block_m, tot, pad, a.block_expert, a.num_padded);
  if (P > 0)
    hipLaunchKernelGGL(align_fill_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, a.R, a.num_local,
                       a.block_m, P, pad, tot, a.block_expert, a.sorted_rows);
  if (nch > 0)
    hipLaunchKernelGGL(align_scatter_kernel, dim3(nch), dim3(kAlignChunk), 0, st, a.local_expert, a.R, a.num_local,
                       rank, chunk, pad, a.sorted_rows);
  return hipGetLastError();
}

// ---------------------------------------------------------------- grouped GEMM
// Block: 256 threads (4 waves) x 128 sorted rows (one expert) x `tpb` tiles of 64 NB weight rows, K in steps of 128 (two
// quantisation groups). Each wave owns 16 NB weight rows of a tile (NB 16-column MFMA B fragments) for all rows of the
// block, so every weight is dequantized exactly once, by the wave that multiplies it, straight into MFMA B registers.
// Gate/up: the first NB / 2 fragments are gate rows, the others the same up rows, so silu(g) * u is formed in
// registers. Column n of fragment j is the wave's weight row NB n + j (gate/up: h column (NB / 2) n + j % (NB / 2)), so
// a lane's fragments hold adjacent outputs and the epilogues store whole pieces.
// K order inside a step: lane quad q (lane >> 4) holds the 16 bytes of packed words 4q .. 4q + 3 of its weight row
// (elements 32 q .. 32 q + 31, one group); MFMA slice s (0..3) uses word 4q + s, and the A fragment of slice s holds
// the same elements of each row. The order is the same for every tile shape and every number of live rows, so a
// row's bits depend on that row and its record only.
// Memory paths:
//  * A (activations for gate/up, h for down): direct global -> LDS loads of 16 bytes per lane (four whole 256-byte row
//    pieces per instruction), double-buffered; only the live 16-row fragments are loaded. The two stages are separate
//    LDS objects, so the compiler knows that a pending load into one does not touch reads of the other. 16-byte chunk
//    c of row m sits at chunk position c ^ a_swz(m), the lane that loads a position reads the chunk that belongs
//    there, and the 16 lanes one ds_read_b128 phase serves fall on distinct banks (1.6 M conflict cycles per gate/up
//    launch at 8192 tokens; with c ^ (m & 15) 23 M).
//  * Packed weights: 16 bytes per lane per step straight into registers, one stage ahead.
//  * Scales and biases: 8 groups (4 steps) of the wave's own rows at a time, direct to LDS, loaded once the last
//    step of the previous 8 groups has read its values.
// A stage holds KS steps: KS rises as the live rows fall (the loads of one stage are in flight while the previous one
// is computed, and a light stage has little to compute), at the same LDS bytes.
// What bounds it (MI355X, 8192 tokens x top-10, H 2048 / I 512, gate/up): 372 us, 924 TFLOP/s; without the loads 330,
// without the dequantisation 315, without either 256, MFMA alone 161: the dequantisation (19 VALU per 8 nibbles) and
// the MFMAs of the two waves of a SIMD overlap only in part (ordering one slice's dequantisation between the MFMAs of
// the slice before, with or without wave priorities, changes nothing). The down product writes 671 MB of out_rows: 280
// us, 195 without the stores. The former kernel (64-wide K steps, activations through registers, a barrier per 64 K,
// four fragments always) took 424 and 325 us, and the pair 245 us at 2048 tokens and 45 at 19 (now 232 and 39).
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
SS_DEV ss_u32x4 dequant8(uint32_t w, float s9, float bi) {
  const int lo = (int)and_opaque(w, 0x0F0F0F0Fu), hi = (int)and_opaque(w >> 4, 0x0F0F0F0Fu);  // n0 n2 n4 n6 / n1 n3 n5 n7
  const auto e02 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, false), e46 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, true);
  const auto e13 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false), e57 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
  ss_u32x4 r;
  r.x = cvt_pk_bf16(__builtin_fmaf(e02[0], s9, bi), __builtin_fmaf(e13[0], s9, bi));
  r.y = cvt_pk_bf16(__builtin_fmaf(e02[1], s9, bi), __builtin_fmaf(e13[1], s9, bi));
  r.z = cvt_pk_bf16(__builtin_fmaf(e46[0], s9, bi), __builtin_fmaf(e57[0], s9, bi));
  r.w = cvt_pk_bf16(__builtin_fmaf(e46[1], s9, bi), __builtin_fmaf(e57[1], s9, bi));
  return r;
}

struct GemmArgs {
  const uint16_t* a;           // gate/up: x bf16 [T, H]; down: h bf16 [R, I]
  const int32_t* row_token;    // [R] (gate/up)
  const float* row_weight;     // [R] (down)
  const int32_t* sorted_rows;  // [P]
  const int32_t* block_expert; // [P / kBM]
  const int32_t* num_padded;   // [1]
  const int64_t* group_ptr;    // [num_local] record base addresses
  uint16_t* h;                 // gate/up output bf16 [R, I]
  float* out_rows;             // down output fp32 [R, H]
  int64_t R;
  int T, H, I;
  int64_t w_off, s_off, b_off;     // gate (or down) pieces
  int64_t w2_off, s2_off, b2_off;  // up pieces (gate/up)
  uint64_t* trace;                 // per-block stamps (start, end, expert << 32 | valid rows, XCC << 32 | HW_ID) or null
};

// LDS barrier for data exchanged through LDS only: waits for this wave's LDS operations, not for its global loads
// in flight (which a workgroup-scope fence would also wait for).
SS_DEV void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Block index -> (M block, group of N tiles). The plan's M blocks are dealt round-robin to the XCDs (workgroup b runs on
// XCD b % 8), in plan order, so every XCD gets an even share of the heavy and the light experts' blocks; each XCD takes
// all N tiles of one M block in a row (they share its activation rows in the XCD's L2). Measured on MI355X, contiguous
// per-XCD ranges of the plan end 140-180 us apart at 2048 tokens, and groups of 2, 4 or 8 M blocks per XCD (for the
// weights they share) change nothing.
SS_DEV bool xcd_tile(int mb, int nt, int& pid_m, int& pid_n) {
  const int b = blockIdx.x, x = b & 7, s = b >> 3;
  const int sm = s / nt;
  pid_m = sm * 8 + x;
  pid_n = s - sm * nt;
  return pid_m < mb;
}

// Chunk swizzle of activation row m (see above): ds_read_b128 serves lanes 0-3 and 12-15 of one quad with lanes 4-11 of
// its neighbour, whose chunk numbers differ in bit 2, so rows 4-11 (mod 16) take the upper half of the positions.
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
  const uint32_t lw = (uint32_t)((GU ? 8 * NB * w + HB * n : 16 * NB * w + NB * n) * wrow_b + 16 * q);
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
  const int sb_lane = 1024 * w + (wide ? 16 : 4) * n + 2 * (q >> 1);
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
    int apos = 16 * ((4 * q) ^ a_swz(n));
    asm volatile("" : "+v"(apos));
    float sc[KS][NB], bi[KS][NB];
#pragma unroll
    for (int u = 0; u < KS; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int at = sb_lane + j * sb_j + ((st * KS + u) & (kSbG / 2 - 1)) * sb_k;
        sc[u][j] = __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t*>(lss + at) << 16) * 512.f;  // s * 2^9
        bi[u][j] = __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t*>(lsb + at) << 16);
      }
    if (chunk) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      load_sb(ct, cg);
    }
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (u > 0 && st * KS + u >= nsteps) break;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        ss_u32x4 bf[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const uint4 v = bw[P][u][j];
          bf[j] = dequant8(s == 0 ? v.x : s == 1 ? v.y : s == 2 ? v.z : v.w, sc[u][j], bi[u][j]);
        }
        // A fragments a few at a time: the scheduling barriers keep their registers few; the two waves of a SIMD
        // overlap one wave's dequantisation and LDS reads with the other's MFMAs.
        const uint8_t* ap = as + u * NF * 16 * kRowB + (apos ^ (16 * s));
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
  auto epilogue = [&](int tile) {
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
          if constexpr (NB == 4)
            stg16(od, make_uint4(__float_as_uint(acc[i][0][r] * wt), __float_as_uint(acc[i][1][r] * wt),
                                 __float_as_uint(acc[i][2][r] * wt), __float_as_uint(acc[i][3][r] * wt)));
          else
            *(SS_G ss_f32x2*)od = ss_f32x2{acc[i][0][r] * wt, acc[i][1][r] * wt};
        }
      }
  };

  zero();
  int tile = tile0, st = 0;
  const int nall = ntile * nst;
  constexpr int SPC = kSbG / 2 / KS;  // stages per table chunk
  load_sb(tile, 0);
  load(tile, 0, std::integral_constant<int, 0>{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  // Stage f of all tiles: the next stage's loads, this stage's MFMAs, the tile's epilogue behind its last stage, then
  // the wait for the loads (every wave's, by the barrier).
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
    if (st == nst - 1) {
      epilogue(tile);
      zero();
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
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
  const int e = g.block_expert[pid_m];
  if (e < 0) return;
  const uint64_t t_start = g.trace ? __builtin_amdgcn_s_memrealtime() : 0;
  const uint8_t* base = reinterpret_cast<const uint8_t*>(g.group_ptr[e]);
  bool valid = false;
  if (tid < kBM) {
    const int r = g.sorted_rows[(int64_t)pid_m * kBM + tid];
    valid = r < g.R;
    int row = kZeroRow;
    if (valid) {
      if (GU) {
        const int t = g.row_token[r];
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
  // An expert with rows fills at most its rows / 128 whole M blocks and one partial one, so the grid covers that bound
  // (rounded up to a multiple of 8) times the N tiles; blocks past the device-side count exit at once.
  const int64_t P = padded_rows(p.R, p.num_local, kBM);
  const int64_t bound = (p.R < p.num_local ? p.R : p.num_local) + p.R / kBM;
  const int64_t mb = bound < P / kBM ? bound : P / kBM;
  // Tiles: with few rows per expert most M blocks are light and the chip is short of blocks, so a wave takes two
  // weight fragments instead of four (twice the blocks); with more rows the wider wave reads its activations from LDS
  // half as often. Measured with 512 experts (us, two / four fragments): gate/up R = 190 24 / 27, 3330 (H 2560 /
  // I 640) 85 / 90, 6000 67 / 72, 20480 139 / 124; down R = 190 15 / 17, 480 20 / 20, 3330 55 / 54, 6000 48 / 43.
  // Two down tiles per block (one prologue) pay off once there are blocks to spare: R = 6000 43 / 43, 10000 (H 2560)
  // 95 against 101 with one, 81920 280 against 300.
  const int nb_gu = p.R < 16 * (int64_t)p.num_local ? 2 : 4, nb_d = p.R < 2 * (int64_t)p.num_local ? 2 : 4;
  const int td = p.R >= 8192 && p.H % 512 == 0 ? 2 : 1;
  launch_gemm<true>(g, nb_gu, 1, mb, st);
  g.a = p.h_buf;
  g.w_off = rec.dw;
  g.s_off = rec.ds;
  g.b_off = rec.db;
  launch_gemm<false>(g, nb_d, td, mb, st);
  return hipGetLastError();
}

// ---------------------------------------------------------------- combine_rank_order (fused_moe_affine.py:164-172)
__global__ __launch_bounds__(256) void combine_kernel(const float* __restrict__ rows,
                                                      const int32_t* __restrict__ row_local, int T, int K, int H,
                                                      float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one float4 of one token
  const int h4 = H >> 2;
  if (idx >= (int64_t)T * h4) return;
  const int64_t t = idx / h4, c = idx - t * h4;
  const float4* p = reinterpret_cast<const float4*>(rows) + (t * K) * h4 + c;
  // Every row is loaded (in bounds) and a skipped row's value replaced by +0 afterwards: a select between a local
  // zero and a loaded value is kept on values, never turned into a load through a selected address.
  float4 acc = p[0];
  if (row_local && row_local[t * K] < 0) acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 1; k < K; ++k) {
    const float4 v = p[(int64_t)k * h4];
    const bool skip = row_local && row_local[t * K + k] < 0;
    acc.x = acc.x + (skip ? 0.f : v.x);
    acc.y = acc.y + (skip ? 0.f : v.y);
    acc.z = acc.z + (skip ? 0.f : v.z);
    acc.w = acc.w + (skip ? 0.f : v.w);
  }
  reinterpret_cast<float4*>(out)[idx] = acc;
}

hipError_t launch_combine(const float* rows, const int32_t* row_local, int T, int K, int H, float* out,
                          hipStream_t st) {
  const int64_t n = (int64_t)T * (H / 4);
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(combine_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rows, row_local, T, K, H,
                     out);
  return hipGetLastError();
}

// group_ptr[e] = slot_ptr[map[map_base + e]] for the resident-pool entry point (0 when absent: such rows are
// skipped by setting their local expert to -1 in the caller's routing).
__global__ void group_ptr_kernel(const int32_t* __restrict__ map, int64_t map_base, int64_t map_len,
                                 const int64_t* __restrict__ slot_ptr, int64_t n_slots, int E, int64_t* gptr,
                                 const int32_t* __restrict__ ids, int64_t R, int32_t* __restrict__ local, int* err) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < E) {
    const int64_t mi = map_base + i;
    const int slot = mi < map_len ? map[mi] : -1;
    gptr[i] = (slot >= 0 && slot < n_slots) ? slot_ptr[slot] : 0;
  }
  if (i < R) {
    const int e = ids[i];
    int le = -1;
    if (e >= 0 && e < E) {
      const int64_t mi = map_base + e;
      const int slot = mi < map_len ? map[mi] : -1;
      if (slot >= 0 && slot < n_slots) le = e;
      else ss_raise(err, SS_ERR_SLOT);
    } else {
      ss_raise(err, SS_ERR_EXPERT_ID);
    }
    local[i] = le;
  }
}

__global__ void row_token_kernel(int64_t R, int K, int32_t* row_token) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < R) row_token[i] = (int32_t)(i / K);
}

hipError_t launch_prefill_tables(const int32_t* map, int64_t map_base, int64_t map_len, const int64_t* slot_ptr,
                                 int64_t n_slots, int E, int64_t* gptr, const int32_t* ids, int64_t R, int K,
                                 int32_t* local, int32_t* row_token, int* err, hipStream_t st) {
  const int64_t n = R > E ? R : E;
  hipLaunchKernelGGL(group_ptr_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, map, map_base, map_len,
                     slot_ptr, n_slots, E, gptr, ids, R, local, err);
  if (R > 0) hipLaunchKernelGGL(row_token_kernel, dim3((unsigned)((R + 255) / 256)), dim3(256), 0, st, R, K, row_token);
  return hipGetLastError();
}

}  // namespace ss
