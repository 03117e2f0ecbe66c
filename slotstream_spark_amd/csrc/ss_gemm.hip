// Dense bf16 GEMM C = bf16(A B^T) for the prefill's plain projections (lin on bf16 weights over a prompt chunk,
// model/layers.py:62-76): the router logits (x W_gate^T), the shared expert's gate/up/gate-logit rows
// (x [W_g; W_u; w_sg]^T) and its down projection (hs W_d^T). A [M][K] and B [N][K] are row-major with K contiguous
// (the torch layout of activations and nn.Linear weights), the dot is accumulated in fp32 by the MFMA unit and
// rounded once to bf16.
//
// Block tile (2 WM 16) x (2 WN 16): four waves in a 2 x 2 arrangement, each owning WM x WN 16 x 16 output fragments
// (v_mfma_f32_16x16x32_bf16). K advances in steps of 64 through four LDS stages filled by direct global -> LDS loads
// of 16 bytes per lane (8 whole 128-byte row pieces per instruction), three steps ahead; every step issues the same
// number of loads, so the wait before a step's barrier is a count (the loads of the next two steps stay in flight).
// The stages are separate LDS objects, so the compiler adds no wait of its own for a load into another stage. In LDS the
// 16-byte chunk c of tile row m sits at position c ^ (m & 7) ^ ((m >> 3) & 1) of the row's 128 bytes, so the 16 rows
// one MFMA operand read touches fall on distinct banks. K order inside a step: lane quad q (lane >> 4) of a fragment
// holds elements 16 q + 8 s .. + 7 of its row for MFMA slice s (0, 1), for A and B alike; it does not depend on the
// tile, so neither do the bits of an output.
// Rows of A past M and of B past N read row 0 (a valid address) and their results are not stored.
//
// What bounds it: the operand bytes each CU takes in (see launch_by_size).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ss_common.hpp"
#include "ss_launch.hpp"

namespace ss {

namespace {

constexpr int kGK = 64;     // K per step
constexpr int kStages = 4;  // LDS stages (K is a multiple of kGK * kStages)

typedef __attribute__((address_space(3))) void ss_lds_void;

// Direct-to-LDS load: lane l's 16 bytes land at lds + 16 l (lds is wave-uniform).
SS_DEV void dma16(const void* src, void* lds) { __builtin_amdgcn_global_load_lds(src, (ss_lds_void*)lds, 16, 0, 0); }

SS_DEV int chunk_pos(int m, int c) { return c ^ (m & 7) ^ ((m >> 3) & 1); }

SS_DEV void gemm_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// s_waitcnt immediate that waits for all but `v` vector-memory operations (gfx9 encoding: vmcnt in bits 3:0 and 15:14;
// export and LDS counts at their maxima, not waited for).
constexpr int vmcnt_only(int v) { return (v & 15) | (7 << 4) | (15 << 8) | ((v >> 4) << 14); }

struct DenseGemmArgs {
  const uint16_t* a;  // [M][lda]
  const uint16_t* b;  // [N][ldb]
  uint16_t* c;        // [M][ldc]
  int M, N, K;
  int64_t lda, ldb, ldc;
  int tiles_n, nsteps, tiles, tiles_per_xcd;
  // The prompt layer's input projections in one launch (LAYER): N tiles [0, tr) are the router rows b -> c, tiles
  // [tr, tr + ts) pairs of shared gate and up rows of sh -> hs = bf16(bf16(silu(g)) * u) [M][Is], the last tile the
  // shared_expert_gate row -> sgl [M].
  const uint16_t* sh;  // [2 Is + 1][ldb]: gate rows, up rows, the shared_expert_gate row
  uint16_t* hs;
  uint16_t* sgl;
  int Is, tr, ts;
};

template <int WM, int WN, bool LAYER>
__global__ __launch_bounds__(256) void dense_gemm_kernel(DenseGemmArgs g) {
  constexpr int BM = 2 * WM * 16, BN = 2 * WN * 16;
  constexpr int LA = BM / 32, LB = BN / 32;  // load instructions per wave and step (8 rows each)
  constexpr int L = LA + LB;
  __shared__ __attribute__((aligned(256))) uint8_t l0[(BM + BN) * 128];
  __shared__ __attribute__((aligned(256))) uint8_t l1[(BM + BN) * 128];
  __shared__ __attribute__((aligned(256))) uint8_t l2[(BM + BN) * 128];
  __shared__ __attribute__((aligned(256))) uint8_t l3[(BM + BN) * 128];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 1, wn = w & 1;
  // Workgroups are dealt to the 8 XCDs round-robin; XCD x takes the contiguous tile range [x per, (x + 1) per), so
  // the N tiles of one M tile share an XCD and its L2 holds that A tile for all of them.
  const int per = g.tiles_per_xcd, T = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (T >= g.tiles) return;  // whole workgroup, before any barrier
  const int tm = T / g.tiles_n, tn = T - tm * g.tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  const bool pairs = LAYER && tn >= g.tr && tn < g.tr + g.ts, gate = LAYER && tn >= g.tr + g.ts;
  const int i0 = pairs ? (tn - g.tr) * (BN / 2) : 0;  // first hs column of a pair tile

  // Load instruction i of wave w covers tile rows 8 (w + 4 i) + lane / 8, position lane % 8 of each: chunk
  // (lane % 8) ^ (lane / 8) ^ (w & 1) (4 i is even).
  const int lr = lane >> 3, lc = (lane & 7) ^ lr ^ (w & 1);
  const uint16_t* asrc[LA];
  const uint16_t* bsrc[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int m = m0 + 8 * (w + 4 * i) + lr;
    asrc[i] = g.a + (size_t)(m < g.M ? m : 0) * g.lda + 8 * lc;
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int r = 8 * (w + 4 * i) + lr;
    if (pairs) {
      // row r of wave column r / (16 WN): its first WN / 2 fragments are gate rows, the others the same up rows
      const int c = r / (16 * WN), j = r / 16 % WN;
      const int col = i0 + c * 8 * WN + (j % (WN / 2)) * 16 + r % 16;
      bsrc[i] = g.sh + (size_t)((j < WN / 2 ? 0 : g.Is) + col) * g.ldb + 8 * lc;
    } else if (gate) {
      bsrc[i] = g.sh + (size_t)(2 * g.Is) * g.ldb + 8 * lc;
    } else {
      const int n = n0 + r;
      bsrc[i] = g.b + (size_t)(n < g.N ? n : 0) * g.ldb + 8 * lc;
    }
  }
  const int nsteps = g.nsteps;
  auto stage_of = [&](auto s_c) {
    constexpr int S = decltype(s_c)::value;
    return S == 0 ? l0 : S == 1 ? l1 : S == 2 ? l2 : l3;
  };
  auto load = [&](int k, auto s_c) {
    uint8_t* st = stage_of(s_c);
    const int kk = k < nsteps ? k : nsteps - 1;  // past the end: the last step again, into a stage that is not read
#pragma unroll
    for (int i = 0; i < LA; ++i)
      dma16(asrc[i] + (size_t)kk * kGK, st + 1024 * (w + 4 * i));
#pragma unroll
    for (int i = 0; i < LB; ++i)
      dma16(bsrc[i] + (size_t)kk * kGK, st + BM * 128 + 1024 * (w + 4 * i));
  };

  const int n = lane & 15, q = lane >> 4;
  ss_f32x4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  const int ro0 = n * 128 + 16 * chunk_pos(n, 2 * q), ro1 = n * 128 + 16 * chunk_pos(n, 2 * q + 1);

  load(0, std::integral_constant<int, 0>{});
  load(1, std::integral_constant<int, 1>{});
  load(2, std::integral_constant<int, 2>{});
  __builtin_amdgcn_sched_barrier(0);
  // Step k (stage S): its loads have landed once at most the 2 L loads of steps k + 1 and k + 2 are in flight; the
  // barrier makes every wave's visible, and frees the stage of step k - 1 for the loads of step k + 3.
  auto step = [&](int k, auto s_c) {
    constexpr int S = decltype(s_c)::value;
    const uint8_t* st = stage_of(s_c);
    // No fence here: a release would wait for every load in flight. The waves write LDS by these loads only, and each
    // has consumed its reads of step k - 1 (MFMA operands) before it arrives.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vmcnt_only(2 * L));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load(k + 3, std::integral_constant<int, (S + 3) % kStages>{});
    __builtin_amdgcn_sched_barrier(0);
    // Both slices' fragments are requested before the first MFMA, so slice 1's LDS reads run under slice 0's MFMAs.
    ss_u32x4 av[2][WM], bv[2][WN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint8_t* p = st + (s ? ro1 : ro0);
#pragma unroll
      for (int j = 0; j < WN; ++j) bv[s][j] = *reinterpret_cast<const ss_u32x4*>(p + BM * 128 + (wn * WN + j) * 2048);
#pragma unroll
      for (int i = 0; i < WM; ++i) av[s][i] = *reinterpret_cast<const ss_u32x4*>(p + (wm * WM + i) * 2048);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = ss_mfma(av[s][i], bv[s][j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll 1
  for (int k = 0; k < nsteps; k += kStages) {
    step(k, std::integral_constant<int, 0>{});
    step(k + 1, std::integral_constant<int, 1>{});
    step(k + 2, std::integral_constant<int, 2>{});
    step(k + 3, std::integral_constant<int, 3>{});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  gemm_barrier();
  // acc[i][j][r]: row 16 i + 4 q + r, column 16 j + n of the wave's fragment grid. The block's C tile goes through
  // LDS (one stage, dead by now) so that it leaves in 16-byte row pieces.
  static_assert(BM * BN * 2 <= (BM + BN) * 128, "the C tile fits one stage");
  uint16_t* ct = reinterpret_cast<uint16_t*>(l0);
  const int cw = pairs ? BN / 2 : BN;  // columns of the output tile
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      uint16_t* row = ct + (wm * WM * 16 + 16 * i + 4 * q + r) * cw + wn * (cw / 2) + n;
      if (pairs) {
#pragma unroll
        for (int j = 0; j < WN / 2; ++j) {
          const float gv = ss_round_bf16(acc[i][j][r]), uv = ss_round_bf16(acc[i][j + WN / 2][r]);
          const float sv = ss_round_bf16(gv / (1.f + ss_expf(-gv)));
          row[16 * j] = (uint16_t)ss_f32_to_bf16(sv * uv);
        }
      } else {
#pragma unroll
        for (int j = 0; j < WN; ++j) row[16 * j] = (uint16_t)ss_f32_to_bf16(acc[i][j][r]);
      }
    }
  gemm_barrier();
  if (gate) {  // column 0 of the tile
    for (int r = tid; r < BM; r += 256)
      if (m0 + r < g.M) g.sgl[m0 + r] = ct[r * BN];
    return;
  }
  uint16_t* out = pairs ? g.hs : g.c;
  const int64_t ldo = pairs ? g.Is : g.ldc;
  const int no = pairs ? g.Is : g.N, c0 = pairs ? i0 : n0, cpr = cw / 8;  // 16-byte pieces per tile row
  for (int idx = tid; idx < BM * cpr; idx += 256) {
    const int r = idx / cpr, c8 = idx - r * cpr;
    const int row = m0 + r, col = c0 + 8 * c8;
    if (row < g.M && col < no)
      *reinterpret_cast<uint4*>(out + (size_t)row * ldo + col) = *reinterpret_cast<const uint4*>(ct + r * cw + 8 * c8);
  }
}

template <int WM, int WN, bool LAYER>
hipError_t launch_tiles(const DenseGemmArgs& g0, hipStream_t st) {
  DenseGemmArgs g = g0;
  constexpr int BM = 2 * WM * 16, BN = 2 * WN * 16;
  g.tiles_n = (g.N + BN - 1) / BN;
  if (LAYER) {
    g.tr = g.tiles_n;
    g.ts = g.Is / (BN / 2);
    g.tiles_n += g.ts + 1;
  }
  g.tiles = ((g.M + BM - 1) / BM) * g.tiles_n;
  g.tiles_per_xcd = (g.tiles + 7) / 8;
  hipLaunchKernelGGL((dense_gemm_kernel<WM, WN, LAYER>), dim3((unsigned)(8 * g.tiles_per_xcd)), dim3(256), 0, st, g);
  return hipGetLastError();
}

// Tile by size. A CU takes in about 33 bytes a cycle, whichever path the loads go, so a tile's time is its operand
// bytes: 32 steps of 12 / 16 / 32 KB take 6.3 / 8.2 / 20 us however few tiles there are, and the largest tile moves the
// fewest bytes per FLOP once it fills the chip without a mostly empty last round. Measured (us, 32 x 64 / 64 x 64 /
// 128 x 128; N columns, K 2048): M 19 N 512 6.3 / 8.2 / 20; M 333 N 1544 11 / 9.0 / 20; M 2048 N 1544 40 / 31 / 22;
// M 4096 N 1032 43 / 34 / 40 (288 large tiles on 256 CUs); M 8192 N 1544 143 / 95 / 86. Before (64 x 64 through
// registers, two launches for the 1544 columns): 18.8, 19.5, 32, -, 92 us.
template <bool LAYER>
hipError_t launch_by_size(const DenseGemmArgs& g, hipStream_t st) {
  const int64_t cols = g.N + (LAYER ? 2 * (int64_t)g.Is + 1 : 0);
  auto tiles = [&](int bm, int bn) { return ((g.M + bm - 1) / bm) * ((cols + bn - 1) / bn); };
  const int64_t large = tiles(128, 128), rounds = (large + 255) / 256;
  if (large >= 192 && 256 * rounds * 5 <= large * 7) return launch_tiles<4, 4, LAYER>(g, st);
  if (tiles(64, 64) > 128) return launch_tiles<2, 2, LAYER>(g, st);
  return launch_tiles<1, 2, LAYER>(g, st);
}

}  // namespace

hipError_t launch_dense_gemm(const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, uint16_t* c, int64_t ldc,
                             int M, int N, int K, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  DenseGemmArgs g{};
  g.a = a;
  g.b = b;
  g.c = c;
  g.M = M;
  g.N = N;
  g.K = K;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.nsteps = K / kGK;
  return launch_by_size<false>(g, st);
}

hipError_t launch_layer_gemm(const uint16_t* x, const uint16_t* router_w, const uint16_t* sh_cat, uint16_t* logits,
                             uint16_t* hs, uint16_t* sgl, int T, int H, int E, int Is, hipStream_t st) {
  if (T == 0) return hipSuccess;
  DenseGemmArgs g{};
  g.a = x;
  g.b = router_w;
  g.c = logits;
  g.M = T;
  g.N = E;
  g.K = H;
  g.lda = g.ldb = H;
  g.ldc = E;
  g.sh = sh_cat;
  g.hs = hs;
  g.sgl = sgl;
  g.Is = Is;
  g.nsteps = H / kGK;
  return launch_by_size<true>(g, st);
}

}  // namespace ss
