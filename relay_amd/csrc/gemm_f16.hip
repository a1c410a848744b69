// Dense fp16 products above the skinny kernels' token range, on the matrix cores:
//
//   y[t, n] = sum_k W16[n, k] * x[t, k]  (+ beta * y[t, n])
//
// The role of relay's cublasGemmEx calls (cuda_backend.cu:726-730). One kernel template: a
// workgroup of WN x WT x WK waves computes BN weight rows x BT tokens in 64-k steps. Both
// operands go from global memory straight into a ring of STAGES LDS buffers (no registers, so
// up to 144 KB per CU are in flight), one barrier per step; the operand reads of the next
// 16-k slice are issued before the MFMAs of the current one, across the barrier too.
//
// What bounds it (MI355X). Few tokens: the weight stream. Many: the L2 -> LDS feed; a copy of
// the kernel with only the loads left takes 85-95% of its time on the 128- and 256-row
// tiles, and a copy without them reaches 1.1-1.38 PFLOP/s. So: 8 waves rather than 4 where
// the tile allows it (a wave's own loads arrive at ~7 GB/s: 256 x 128 at 2048 x 8192 x 8192,
// loads only, 297 us with 4 waves, 261 with 8); WK = 2 splits each step's k between two
// groups of waves, so that 8 waves read the operands of 4 (LDS reads per MFMA as for 4 large
// wave tiles); and the workgroups of an XCD cover a compact block of tiles (below).
#include "../../include/relay_hip.h"
#include "common.h"
#include "lds_ring.h"

#include <algorithm>

namespace relay_hip {
namespace {

constexpr int kMaxF16Split = 8;
// Tiles are dealt to the XCDs as contiguous ranges (workgroup L runs on XCD L % 8) of an order
// that walks kBand row tiles per token tile: the 32 workgroups an XCD runs at a time cover
// about 8 x 4 tiles, whose W and x slices they share through its L2, all in one K range.
// Against token tiles fastest over all of them (2048 tokens, 8192 x 8192, 128 x 128 tiles):
// loads only 340 -> 219 us, the kernel 379 -> 343; level at 512 tokens.
constexpr int kBand = 8;

// kStore: y (or this K range's plane of the workspace). kSilu: W is the fused [gate; up]
// matrix (N = 2 I rows); each 32-row block of the tile holds 16 gate rows and their 16 up
// rows, so g and u of an output are in one lane and act[t, a] = fp16(silu(g) * u) is stored.
enum F16Epilogue { kStore = 0, kSilu = 1 };

template <int BN, int BT, int WN, int WT, int WK, int STAGES, int EPI>
__global__ __launch_bounds__(WN * WT * WK * 64, 1) void gemm_f16_kernel(const half_t* __restrict__ w16, int64_t ldw,
                                                                const half_t* __restrict__ x, float* y, int T, int K,
                                                                int N, float beta, float* ws, int n_row, int n_tok,
                                                                int ksn) {
  constexpr int KS = 64, WAVES = WN * WT * WK, Q = 4 / WK, AN = BN / WN / 32, AT = BT / WT / 32;
  constexpr int ROWS = BN + BT, PIECES = ROWS / 8;  // a piece: 8 rows x 128 bytes, one wave load
  constexpr int LPS = (PIECES + WAVES - 1) / WAVES;             // loads per wave and stage
  constexpr int AHEAD = STAGES - 1;                  // stages issued before the first step
  static_assert(STAGES >= 3, "a stage's loads are spread over the step two stages before its own");
  static_assert(WK == 1 || STAGES * ROWS * 128 >= BN * BT * 4, "the K halves meet in the ring");
  static_assert(BN % (32 * WN) == 0 && BT % (32 * WT) == 0, "tile");
  constexpr int STAGE = ROWS * KS;                  // halves per stage: W rows, then x rows
  __shared__ __attribute__((aligned(1024))) half_t lds[STAGES * STAGE];

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const int wn = w % WN, wt = w / WN % WT, wk = w / (WN * WT);
  const int total = n_row * n_tok * ksn, L = blockIdx.x;
  const int per = total / 8, rem8 = total % 8, xcd = L % 8;
  const int idx = xcd * per + min(xcd, rem8) + L / 8;
  const int rks = n_row * ksn, band = idx / (kBand * n_tok), left = min(kBand, rks - band * kBand);
  const int in = idx - band * kBand * n_tok, tok = in / left, rk = band * kBand + in % left;
  const int kz = rk / n_row, row = rk % n_row;
  const int n0 = row * BN, t0 = tok * BT;
  const int nall = K / KS, sbeg = kz * nall / ksn, nsteps = (kz + 1) * nall / ksn - sbeg;
  const int I = N / 2;  // kSilu only

  // Piece p = w + WAVES * i covers tile rows 8 p .. 8 p + 7 (W rows first, then x rows).
  // Lane l brings 16-byte chunk (l % 8) ^ swz(row) of row 8 p + l / 8: rows are stored with
  // their chunks XOR-permuted by (row >> 1) & 7, which makes the operand reads below cover
  // all 64 banks once per 16 lanes.
  const uint4v wrs = lds_rsrc(w16);
  const uint4v xrs = lds_rsrc(x);
  uint32_t voff[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int r = 8 * min(w + WAVES * i, PIECES - 1) + (lane >> 3);  // tile row
    const int ch = (lane & 7) ^ ((r >> 1) & 7);
    if (r < BN) {
      int64_t n;
      if constexpr (EPI == kSilu) {
        const int a = min(n0 / 2 + (r >> 5) * 16 + (r & 15), I - 1);
        n = (r & 16) ? I + a : a;
      } else {
        n = min(n0 + r, N - 1);
      }
      voff[i] = static_cast<uint32_t>(n * ldw * 2 + ch * 16);
    } else {
      const int t = min(t0 + r - BN, T - 1);
      voff[i] = static_cast<uint32_t>((static_cast<int64_t>(t) * K + ch * 8) * 2);
    }
  }
  const uint32_t lds0 = lds_address(lds);
  // Part `part` of `parts` of stage s's loads into ring buffer `buf`.
  auto issue = [&](int s, int buf, int part, int parts) {
    const uint32_t so = static_cast<uint32_t>((sbeg + s) * KS * 2);
#pragma unroll
    for (int i = 0; i < LPS; ++i) {
      if (i < LPS * part / parts || i >= LPS * (part + 1) / parts) continue;
      const int p = min(w + WAVES * i, PIECES - 1);
      const uint32_t dst = lds0 + static_cast<uint32_t>(buf * STAGE * 2 + p * 1024);
      load_to_lds(p * 8 < BN ? wrs : xrs, voff[i], so, dst);
    }
  };

  float16v acc[AN][AT];
#pragma unroll
  for (int a = 0; a < AN; ++a)
#pragma unroll
    for (int b = 0; b < AT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

  half8 fa[2][AN], fb[2][AT];
  const int sw = (c >> 1) & 7;  // rows of a block are 32-aligned
  const half_t* const la = lds + (wn * AN * 32 + c) * KS;
  const half_t* const lb = lds + (BN + wt * AT * 32 + c) * KS;
  auto read = [&](int buf, int q, int set) {
    const int off = buf * STAGE + (((2 * (wk * Q + q) + h) ^ sw) << 3);
#pragma unroll
    for (int a = 0; a < AN; ++a) fa[set][a] = *reinterpret_cast<const half8*>(la + off + a * 32 * KS);
#pragma unroll
    for (int b = 0; b < AT; ++b) fb[set][b] = *reinterpret_cast<const half8*>(lb + off + b * 32 * KS);
  };
  auto mma = [&](int set) {
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int b = 0; b < AT; ++b) acc[a][b] = mfma32x32x16(fa[set][a], fb[set][b], acc[a][b]);
  };

#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (s < nsteps) issue(s, s, 0, 1);
  wait_stages<LPS, AHEAD - 1>(nsteps - 1);
  ring_barrier();
  read(0, 0, 0);
  int buf = 0;
  for (int s = 0; s < nsteps; ++s) {
    const int pbuf = buf == 0 ? STAGES - 1 : buf - 1, nbuf = buf + 1 == STAGES ? 0 : buf + 1;
    const bool more = s + STAGES - 1 < nsteps;
#pragma unroll
    for (int q = 0; q + 1 < Q; ++q) {
      read(buf, q + 1, (q + 1) & 1);
      if (more) issue(s + STAGES - 1, pbuf, q, Q - 1);
      mma(q & 1);
    }
    if (s + 1 < nsteps) {
      // Every read of stage s has landed in registers, stage s + 1 has landed in LDS (in
      // flight behind it: stages s + 2 .. s + AHEAD - 1 ...); after the barrier both hold
      // for all waves, and stage s's buffer takes stage s + STAGES.
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      wait_stages<LPS, STAGES - 2>(nsteps - 2 - s);
      ring_barrier();
      read(nbuf, 0, 0);
    }
    mma((Q - 1) & 1);
    buf = nbuf;
  }
  if constexpr (WK == 2) {
    // Waves w and w + WN WT hold the two K halves of the same blocks: each keeps every other
    // block and hands the rest over through LDS.
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    ring_barrier();
    float* const xs = reinterpret_cast<float*>(lds) + (w % (WN * WT)) * (AN * AT * 1024) + lane * 4;
#pragma unroll
    for (int i = 0; i < AN * AT; ++i)
      if ((i & 1) != wk)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4v*>(xs + i * 1024 + q * 256) =
              float4v{acc[i / AT][i % AT][4 * q], acc[i / AT][i % AT][4 * q + 1], acc[i / AT][i % AT][4 * q + 2],
                      acc[i / AT][i % AT][4 * q + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    ring_barrier();
#pragma unroll
    for (int i = 0; i < AN * AT; ++i)
      if ((i & 1) == wk)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4v v = *reinterpret_cast<const float4v*>(xs + i * 1024 + q * 256);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i / AT][i % AT][4 * q + r] += v[r];
        }
  }

  // Register 4 q + r of block (a, b) in lane (c, h): row 32 a + 8 q + 4 h + r, token 32 b + c.
#pragma unroll
  for (int b = 0; b < AT; ++b) {
    const int t = t0 + 32 * (wt * AT + b) + c;
    if (t >= T) continue;
#pragma unroll
    for (int a = 0; a < AN; ++a) {
      if (WK == 2 && ((a * AT + b) & 1) != wk) continue;
      const int blk = wn * AN + a;
      if constexpr (EPI == kSilu) {
        half_t* act = reinterpret_cast<half_t*>(y);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int o = n0 / 2 + 16 * blk + 8 * q + 4 * h;
          half_t v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = acc[a][b][4 * q + r], u = acc[a][b][8 + 4 * q + r];
            v[r] = f16_of_product(g / (1.0f + expf(-g)), u);
          }
          half_t* dst = act + static_cast<int64_t>(t) * I + o;
          if (I % 4 == 0 && o + 3 < I) {
            *reinterpret_cast<half4*>(dst) = half4{v[0], v[1], v[2], v[3]};
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (o + r < I) dst[r] = v[r];
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + 32 * blk + 8 * q + 4 * h;
          if (n >= N) continue;
          float4v v = {acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
          float* yp = (ksn > 1 ? ws + static_cast<int64_t>(kz) * T * N : y) + static_cast<int64_t>(t) * N + n;
          if (N % 4 == 0) {
            if (ksn == 1 && beta != 0.0f) v += beta * *reinterpret_cast<const float4v*>(yp);
            *reinterpret_cast<float4v*>(yp) = v;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < N) yp[r] = v[r] + (beta != 0.0f ? beta * yp[r] : 0.0f);
          }
        }
      }
    }
  }
}

template <int BN, int BT, int WN, int WT, int WK, int STAGES, int EPI>
int launch_tile(const half_t* w, int64_t ldw, const half_t* x, float* y, int T, int K, int N, float beta, int ksplit,
                float* ws, hipStream_t s) {
  const int n_row = (N + BN - 1) / BN, n_tok = (T + BT - 1) / BT;
  const int64_t total = static_cast<int64_t>(n_row) * n_tok * ksplit;
  RH_REQUIRE(total < (int64_t(1) << 31), "gemm_f16: grid too large");
  RH_TRY_LAUNCH(hipLaunchKernelGGL((gemm_f16_kernel<BN, BT, WN, WT, WK, STAGES, EPI>), dim3(static_cast<unsigned>(total)),
                                   dim3(WN * WT * WK * 64), 0, s, w, ldw, x, y, T, K, N, beta, ws, n_row, n_tok, ksplit));
  return 0;
}

// The tiles, and a timing model of each, in microseconds, fitted to 4,500 measured (tile,
// split) pairs over 16 matrices (576 x 576 to 4096 x 28672) at 13 T from 16 to 2048 (log-RMS
// error 9%): a workgroup takes (64-k steps of its range) x step + fixed; 256 of them run at a
// time (the two small tiles two to a CU, one alone at `alone` of the pair's rate); the weights
// and partial planes stream at 8 TB/s beside it. The split chosen by the minimum is within
// 2.2% of the measured best on average over those points (worst 42%).
struct F16Tile {
  int rows, toks;
  double step, fixed, alone;
  bool pair;
};
constexpr F16Tile kTiles[] = {
    {64, 64, 0.163, 1.258, 0.670, true},    {128, 64, 0.299, 1.629, 0.782, true},
    {128, 128, 0.467, 3.154, 1.0, false},   {192, 128, 0.607, 5.113, 1.0, false},
    {256, 128, 0.734, 4.892, 1.0, false},   {128, 256, 0.686, 5.017, 1.0, false},
};
constexpr int kNumTiles = 6;

double f16_model_us(int tile, int T, int K, int N, int ks) {
  const F16Tile& c = kTiles[tile];
  const int64_t wgs = static_cast<int64_t>((N + c.rows - 1) / c.rows) * ((T + c.toks - 1) / c.toks) * ks;
  const double w = (K / 64 + ks - 1) / ks * c.step + c.fixed;
  const int64_t rounds = (wgs + 255) / 256;
  const double t = c.pair ? (rounds / 2) * 2.0 * w + (rounds % 2) * w / c.alone : rounds * w;
  const double mem = (2.0 * N * K + 4.0 * ks * T * N) * 1.25e-7;
  return 1.1 + t + mem;
}

struct F16Plan {
  int tile, ks;
  double us;
};

// The fastest tile for a given split, or (ks = 0) the fastest (tile, split) when the product's
// consumer adds the ranges: it then reads ks - 1 further planes, at 5 TB/s.
F16Plan f16_plan(int T, int K, int N, int ks) {
  F16Plan best{0, 1, 0.0};
  const int lo = ks ? ks : 1, hi = ks ? ks : (N % 4 ? 1 : std::min(kMaxF16Split, std::max(1, K / 128)));
  for (int k = lo; k <= hi; ++k)
    for (int i = 0; i < kNumTiles; ++i) {
      const double us = f16_model_us(i, T, K, N, k) + 8e-7 * (k - 1) * T * static_cast<double>(N);
      if (best.us == 0.0 || us < best.us) best = {i, k, us};
    }
  return best;
}

template <int EPI>
int launch_f16(int tile, const half_t* w, int64_t ldw, const half_t* x, float* y, int T, int K, int N, float beta,
               int ksplit, float* ws, hipStream_t s) {
  switch (tile) {
    case 0: return launch_tile<64, 64, 2, 2, 1, 4, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
    case 1: return launch_tile<128, 64, 2, 2, 2, 3, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
    case 2: return launch_tile<128, 128, 4, 2, 1, 4, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
    case 3: return launch_tile<192, 128, 2, 2, 2, 3, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
    case 4: return launch_tile<256, 128, 4, 2, 1, 3, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
    default: return launch_tile<128, 256, 2, 4, 1, 3, EPI>(w, ldw, x, y, T, K, N, beta, ksplit, ws, s);
  }
}

}  // namespace
}  // namespace relay_hip

using namespace relay_hip;

// Byte offsets into W (rows ldw elements apart) and x stay below 2^31.
static bool gemm_f16_offsets_fit(int T, int K, int N, int64_t ldw) {
  return ldw < (int64_t(1) << 30) && N * ldw < (int64_t(1) << 30) && static_cast<int64_t>(T) * K < (int64_t(1) << 30);
}

static int gemm_f16_checks(const void* w16, int64_t ldw, const void* x, int T, int K, int N) {
  RH_REQUIRE(T > 0 && N > 0 && K > 0 && K % 64 == 0, "gemm_f16: K must be a positive multiple of 64");
  RH_REQUIRE(ldw >= K && ldw % 8 == 0, "gemm_f16: ldw must be >= K and a multiple of 8");
  RH_REQUIRE(w16 != nullptr && x != nullptr, "gemm_f16: missing pointer");
  RH_REQUIRE((reinterpret_cast<uintptr_t>(w16) | reinterpret_cast<uintptr_t>(x)) % 16 == 0,
             "gemm_f16: W16 and x must be 16-byte aligned");
  RH_REQUIRE(gemm_f16_offsets_fit(T, K, N, ldw),
             "gemm_f16: T * K or N * ldw too large for 32-bit buffer offsets");
  return 0;
}

extern "C" int rh_gemm_f16_fits(int T, int K, int N) {
  return T > 0 && N > 0 && K > 0 && K % 64 == 0 && gemm_f16_offsets_fit(T, K, N, K);
}

// Where the tile kernel is at least level with hipBLASLt's fastest kernel for the same shape
// (timed on that token count, with the launches that each side needs for its consumer: qkv_post,
// the RMSNorm after o and down, SiLU * mul; us, library / tile). Weights N x K, T tokens:
// - Products whose ranges the consumer adds, below 4 M outputs: 4096 x 4096 at 512 35 / 34, 4096 x
//   14336 at 512 78 / 75, 6144 x 4096 at 560 52 / 49, 2048 x 5632 at 1024 43 / 41; 2048 x 2048 at 768
//   19 / 22 and at 32 9 / 10 (level in whole passes). Past them the library fills the chip with
//   larger tiles: 6144 x 4096 at 1536 84 / 114, 4096 x 14336 186 / 212, 2048 x 5632 at 3072 80 / 93.
// - Plain products only where the plan would not split either; one that has to walk all of K on
//   few workgroups is far behind: 5120 x 13824 at 32 39 / 76, 8192 x 8192 at 64 44 / 62. (LM heads of fewer
//   outputs stay here although the library is ahead, 32000 x 2048 at 32 25 / 31, 128256 x 4096 at 17 161 /
//   182: under 1% of a pass, and its choice by timing adds 17-75 ms to a program's first one.)
// - SiLU in the epilogue, below 10 M outputs, and with K <= 2048 always: 11264 x 2048 at 512 41 / 32,
//   at 2048 115 / 105, 28672 x 4096 at 256 83 / 76, at 384 100 / 125.
//   Not with 100 M weights and more at up to 64 tokens: that is a stream of weights, which the
//   library reads at 6 TB/s and this kernel at 5: 28672 x 4096 at 32 44 / 47, 27648 x 5120 at 64 57 / 64.
extern "C" int rh_gemm_f16_pays(int T, int K, int N, int form) {
  if (!rh_gemm_f16_fits(T, K, N)) return 0;
  const int64_t weights = static_cast<int64_t>(N) * K, outputs = static_cast<int64_t>(T) * N;
  if (form == RH_F16_SILU) return (outputs < 10000000 || K <= 2048) && (T > 64 || weights < 100000000);
  return outputs < 4000000 && (form == RH_F16_RANGES || f16_plan(T, K, N, 0).ks == 1);
}

extern "C" int rh_gemm_f16(const void* w16, int64_t ldw, const void* x, float* y, int T, int K, int N, float beta,
                           void* stream) {
  if (T == 0) return 0;
  if (int rc = gemm_f16_checks(w16, ldw, x, T, K, N)) return rc;
  RH_REQUIRE(y != nullptr && reinterpret_cast<uintptr_t>(y) % 16 == 0, "gemm_f16: y must be 16-byte aligned");
  return launch_f16<kStore>(f16_plan(T, K, N, 1).tile, static_cast<const half_t*>(w16), ldw,
                            static_cast<const half_t*>(x), y, T, K, N, beta, 1, nullptr,
                            static_cast<hipStream_t>(stream));
}

extern "C" int rh_gemm_f16_tile(int T, int K, int N, int ksplit) {
  if (T < 1 || K <= 0 || K % 64 || N <= 0 || ksplit < 1 || ksplit > kMaxF16Split) return -1;
  const F16Tile& t = kTiles[f16_plan(T, K, N, ksplit).tile];
  return t.rows * 1000 + t.toks;
}

extern "C" int rh_gemm_f16_partials_plan(int T, int K, int N) {
  if (T < 1 || K <= 0 || K % 64 || N <= 0) return -1;
  return f16_plan(T, K, N, 0).ks;
}

extern "C" int rh_gemm_f16_partials(const void* w16, int64_t ldw, const void* x, int T, int K, int N, int ksplit,
                                    float* workspace, void* stream) {
  if (T == 0) return 0;
  if (int rc = gemm_f16_checks(w16, ldw, x, T, K, N)) return rc;
  RH_REQUIRE(ksplit >= 2 && ksplit <= kMaxF16Split && ksplit <= K / 64 && workspace && N % 4 == 0,
             "gemm_f16_partials: ksplit in 2..8 (at most K / 64), a workspace and N a multiple of 4");
  RH_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "gemm_f16_partials: workspace must be 16-byte aligned");
  return launch_f16<kStore>(f16_plan(T, K, N, ksplit).tile, static_cast<const half_t*>(w16), ldw,
                            static_cast<const half_t*>(x), nullptr, T, K, N, 0.0f, ksplit, workspace,
                            static_cast<hipStream_t>(stream));
}

// K ranges of the fused gate_up product whose consumer merges them (rh_w8_merge_silu), or 1:
// SiLU in the product's own epilogue, which saves the consumer's launch (3 us) and its reads.
extern "C" int rh_gemm_f16_gate_up_plan(int T, int K, int I) {
  if (T < 1 || K <= 0 || K % 64 || I <= 0) return -1;
  if (I % 8) return 1;
  const F16Plan whole = f16_plan(T, K, 2 * I, 1), split = f16_plan(T, K, 2 * I, 0);
  return split.ks > 1 && split.us + 3.0 + 1.6e-6 * T * I < whole.us ? split.ks : 1;
}

extern "C" int rh_gemm_f16_gate_up_silu(const void* w16, int64_t ldw, const void* x, void* act, int T, int K, int I,
                                        void* stream) {
  if (T == 0) return 0;
  RH_REQUIRE(I > 0, "gemm_f16_gate_up_silu: I must be positive");
  if (int rc = gemm_f16_checks(w16, ldw, x, T, K, 2 * I)) return rc;
  RH_REQUIRE(act != nullptr && reinterpret_cast<uintptr_t>(act) % 8 == 0, "gemm_f16_gate_up_silu: act must be aligned");
  return launch_f16<kSilu>(f16_plan(T, K, 2 * I, 1).tile, static_cast<const half_t*>(w16), ldw,
                           static_cast<const half_t*>(x), static_cast<float*>(act), T, K, 2 * I, 0.0f, 1, nullptr,
                           static_cast<hipStream_t>(stream));
}
