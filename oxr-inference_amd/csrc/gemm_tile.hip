// Tiled bf16 GEMM Y = X * W^T for more than 64 token rows (gfx950).
//
// csrc/gemm.hip streams a weight past at most 64 token rows held in registers; more rows cost it one pass
// over the weight per 64, and every wave re-reads its token rows.  Here a workgroup of 8 waves owns a
// BM x BN tile of Y and both operands pass through LDS, shared by the waves:
// * Stages of KC (64 or 128) k go from memory straight into a ring of LDS slots (16-byte
//   global_load_lds, 1 KiB blocks).  A block of a packed operand is one MFMA fragment block (contiguous in
//   memory and in LDS); a block of a row-major operand is 8 rows of 128 bytes, whose 16-byte chunks are
//   stored rotated (chunk c of row r at c ^ (r / 2 % 8)) so that a fragment's 16 rows fall in distinct
//   banks.  Both forms keep a 16-row piece of 64 k in 2 KiB, so they differ only in lane offsets.
// * One barrier per stage: a wave waits until its own blocks of the stage have landed (the vector memory
//   counter is in order, so "at most the later stages' blocks outstanding"), the barrier makes that true of
//   every wave and ends the previous stage's reads, and that slot is refilled while this stage is multiplied.
// * Within a stage fragments are read two products ahead, with a scheduling barrier per step: left alone
//   the compiler reads each fragment right before its use and waits for the LDS latency 16 times a stage
//   (256 x 256 tile, K = 2048, 4096 x 4096: 65 us; read ahead 56).
// What bounds it.  Large tiles (4096 rows): the matrix cores are busy 61 to 64% of the CU cycles (256 x 256) and 55%
// (256 x 128), LDS reads 23 to 28%; the rest is stage barriers and waits that two waves per SIMD do not cover.
// 4 waves of 128 x 128 read a quarter less LDS but leave one wave per SIMD: 71 us against 56.  Small tiles (up to
// 256 rows): matrix cores 28 to 38%, LDS 28%; the chain of stages waits on memory (see kPer below).
#include <algorithm>

#include "gemm_tile.h"

namespace oxr {
namespace {

enum Epilogue { kStore = 0, kSiluMul = 1, kAddResidual = 3, kPartial = 4 };

struct KernelArgs {
  const bf16_t* x;
  const bf16_t* w;
  bf16_t* y;
  float* part;
  int64_t ldx, k, n, ldy;
  int m, tiles_m, tiles_n, k_slice, part_k;
  int x_packed, w_packed, y_packed;
};

// silu(v) rounded to bf16, for v that is a bf16 value: the bits of bf16(v / (1 + expf(-v))) with a correctly
// rounded divide for every such v (checked over all of them), in 9 instructions instead of about 45; in the
// 256 x 256 tile the epilogue's exponentials and divides took a quarter of the time (61 us a round of tiles
// against 47 without them).  The factors 1/4 keep the reciprocal of the largest denominators normal.
__device__ __forceinline__ float silu_bf16(float v) {
  const float e = __builtin_amdgcn_exp2f(-1.4426950408889634f * v);
  const float d = fmaf(e, 0.25f, 0.25f);
  float q = __builtin_amdgcn_rcpf(d);
  q = fmaf(fmaf(-d, q, 1.0f), q, q);
  return (0.25f * v) * (d < 1e38f ? q : 0.0f);
}

// kParts: the sum over k is formed as args.part_k-long partial sums added in order, as the waves of
// csrc/gemm.hip's kernel form it (same bits); otherwise it is one chain of products.
template <int BM, int BN, int WM, int WN, int STAGES, int KC, bool kParts, int EPI>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(1, 2))) void gemm_tile_kernel(KernelArgs a) {
  constexpr int kWaves = WM * WN;
  constexpr int kTM = BM / WM / 16, kTN = BN / WN / 16;  // 16-row tiles of a wave
  constexpr int kSub = KC / 64;  // 64-k pieces of a stage
  constexpr int kLX = BM / 8 / kWaves, kLW = BN / 8 / kWaves, kL = kSub * (kLX + kLW);
  constexpr int kStageBytes = (BM + BN) * 2 * KC;
  static_assert(BM / 8 % kWaves == 0 && BN / 8 % kWaves == 0, "blocks must divide evenly over the waves");
  static_assert((STAGES - 2) * kL <= 63, "the vector memory counter holds 63");
  static_assert(EPI != kSiluMul || kTN % 2 == 0, "gate and up tiles pair up in a wave");
  extern __shared__ __align__(1024) char lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;

  // Tile of this workgroup: consecutive workgroups go to the 8 XCDs in turn; each XCD takes a contiguous
  // range of tiles, 8 token tiles by column tiles, so that operands are shared in its L2.
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
  int id = xcd * (total >> 3) + min(xcd, total & 7) + slot;
  const int per_split = a.tiles_m * a.tiles_n;
  const int split = id / per_split;
  id -= split * per_split;
  constexpr int kGroup = 8;
  const int group = id / (kGroup * a.tiles_n);
  const int gm = min(kGroup, a.tiles_m - group * kGroup);
  const int in = id - group * kGroup * a.tiles_n;
  const int tm = group * kGroup + in % gm, tn = in / gm;
  const int m0 = tm * BM;
  constexpr int kCols = EPI == kSiluMul ? BN / 2 : BN;  // output columns per workgroup
  const int64_t n0 = (int64_t)tn * kCols;
  const int64_t k0 = (int64_t)split * a.k_slice;

  // First weight row of the tile's 16-row piece jt (gate and up pieces alternate per wave for kSiluMul).
  auto w_row = [&](int jt) -> int64_t {
    if constexpr (EPI == kSiluMul) {
      const int wv = jt / kTN, jj = jt % kTN;
      int64_t c = n0 + 16 * (wv * (kTN / 2) + jj % (kTN / 2));
      c = min(c, (a.n - 1) & ~(int64_t)15);
      return jj >= kTN / 2 ? c + a.n : c;
    }
    return min(n0 + 16 * jt, (a.n - 1) & ~(int64_t)15);
  };

  // Byte offsets of this lane's 16 bytes in each of the wave's blocks, from the operands' slices.
  const int64_t x_step = a.x_packed ? 2048 : 128, w_step = a.w_packed ? 2048 : 128;
  const char* xb = (const char*)(a.x + (a.x_packed ? (int64_t)m0 * a.k + 16 * k0 : (int64_t)m0 * a.ldx + k0));
  const int64_t x_last = a.m - 1 - m0;  // the tile's last row in the matrix
  uint32_t xo[kLX];
#pragma unroll
  for (int u = 0; u < kLX; ++u) {
    const int j = kLX * wave + u;
    if (a.x_packed) {
      xo[u] = (uint32_t)(min<int64_t>(j >> 1, x_last >> 4) * a.k * 32 + (j & 1) * 1024 + lane * 16);
    } else {
      const int row = 8 * j + (lane >> 3);
      xo[u] = (uint32_t)(min<int64_t>(row, x_last) * a.ldx * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7)));
    }
  }
  const char* wb[kLW];
  uint32_t wo[kLW];
#pragma unroll
  for (int u = 0; u < kLW; ++u) {
    const int j = kLW * wave + u;
    const int64_t row0 = w_row(j >> 1);
    if (a.w_packed) {
      wb[u] = (const char*)(a.w + row0 * a.k + 16 * k0 + (j & 1) * 512);
      wo[u] = lane * 16;
    } else {
      const int rr = 8 * (j & 1) + (lane >> 3);
      const int64_t last = (EPI == kSiluMul && row0 >= a.n ? 2 * a.n : a.n) - 1 - row0;
      wb[u] = (const char*)(a.w + row0 * a.k + k0);
      wo[u] = (uint32_t)(min<int64_t>(rr, last) * a.k * 2 + 16 * ((lane & 7) ^ ((rr >> 1) & 7)));
    }
  }

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // Block u (of kL) of the next stage into ring slot `buf`; the last one steps the operands on.
  auto issue1 = [&](int buf, int u) __attribute__((always_inline)) {
    const int sub = u / (kLX + kLW), v = u % (kLX + kLW);
    const uint32_t at = lds0 + buf * kStageBytes + sub * (BM + BN) * 128;
    if (v < kLX) dma_block(xb, xo[v], at + (kLX * wave + v) * 1024);
    else dma_block(wb[v - kLX], wo[v - kLX], at + BM * 128 + (kLW * wave + v - kLX) * 1024);
    if (v == kLX + kLW - 1) {
      xb += x_step;
#pragma unroll
      for (int w = 0; w < kLW; ++w) wb[w] += w_step;
    }
  };
  auto issue = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kL; ++u) issue1(buf, u);
  };

  // Fragment of k32 step i in a 16-row piece (2 KiB of LDS).
  const int wm = wave / WN, wn = wave % WN;
  const int sw = 16 * (g ^ ((r >> 1) & 3)), hi = 64 * ((r >> 3) & 1);
  int xf[2], wf[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int rows = r * 128 + sw + ((64 * i) ^ hi);
    xf[i] = wm * kTM * 2048 + (a.x_packed ? 1024 * i + 16 * lane : rows);
    wf[i] = BM * 128 + wn * kTN * 2048 + (a.w_packed ? 1024 * i + 16 * lane : rows);
  }

  f32x4 acc[kTM][kTN];
#pragma unroll
  for (int i = 0; i < kTM; ++i)
#pragma unroll
    for (int j = 0; j < kTN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 sum[kParts ? kTM : 1][kParts ? kTN : 1];  // finished partial sums
  int part_left = a.part_k / KC;
  bool first_part = true;
  const int stages = a.k_slice / KC;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < stages) issue(s);

  int buf = 0;
  for (int c = 0; c < stages; ++c) {
    // Stage c has landed once at most the later stages' blocks are outstanding.
    const int later = min(STAGES - 2, stages - 1 - c);
    if constexpr (STAGES == 2) {
      wait_vm<0>();
    } else {
      constexpr int kMost = STAGES - 2;
      switch (later) {
        case 0: wait_vm<0>(); break;
        case 1: wait_vm<kL>(); break;
        case 2: wait_vm<std::min(2, kMost) * kL>(); break;
        case 3: wait_vm<std::min(3, kMost) * kL>(); break;
        case 4: wait_vm<std::min(4, kMost) * kL>(); break;
        case 5: wait_vm<std::min(5, kMost) * kL>(); break;
        default: wait_vm<kMost * kL>(); break;
      }
    }
    asm volatile("s_barrier" ::: "memory");
    const bool more = c + STAGES - 1 < stages;
    const int fill = buf == 0 ? STAGES - 1 : buf - 1;
    // Steps of one 16-token piece times the wave's weight pieces; fragments are read two steps ahead, the
    // next k32 step's weight fragments during this one's steps.
    constexpr int kSteps = kTM * 2 * kSub;
    const char* at = lds + buf * kStageBytes;
    u32x4 xv[kSteps], wv[2 * kSub][kTN];
    auto read_x = [&](int q) __attribute__((always_inline)) {
      const int k32 = q / kTM;
      xv[q] = *reinterpret_cast<const u32x4*>(at + (k32 >> 1) * (BM + BN) * 128 + xf[k32 & 1] + 2048 * (q % kTM));
    };
    auto read_w = [&](int k32, int t) __attribute__((always_inline)) {
      wv[k32][t] = *reinterpret_cast<const u32x4*>(at + (k32 >> 1) * (BM + BN) * 128 + wf[k32 & 1] + 2048 * t);
    };
#pragma unroll
    for (int t = 0; t < kTN; ++t) read_w(0, t);
    read_x(0);
    read_x(1);
    __builtin_amdgcn_sched_barrier(0);
    // The next stage's blocks: one a step for the large tiles, all in the first step for the others, whose chain
    // of stages waits on memory (one 128 x 128 tile alone takes as long as a launch of 192): MLP at 256 rows
    // 46.4-46.9 us one a step, 45.7-46.0 at once; a prompt's projections on the large tiles 367.7-368.4 / 369.
    constexpr int kPer = kParts ? kL : (kL + kSteps - 1) / kSteps;
#pragma unroll
    for (int q = 0; q < kSteps; ++q) {
      if (q + 2 < kSteps) read_x(q + 2);
      const int k32 = q / kTM, t = q % kTM;
      if (k32 + 1 < 2 * kSub) {
        constexpr int kOver = kTM > 1 ? kTM - 1 : 1;
        if (t < kOver) {
#pragma unroll
          for (int f = t * kTN / kOver; f < (t + 1) * kTN / kOver; ++f) read_w(k32 + 1, f);
        }
      }
      if (more) {
#pragma unroll
        for (int u = q * kPer; u < (q + 1) * kPer; ++u)
          if (u < kL) issue1(fill, u);
      }
#pragma unroll
      for (int j = 0; j < kTN; ++j) acc[t][j] = mfma_16x16x32(wv[k32][j], xv[q], acc[t][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kParts) {
      if (--part_left == 0) {
        part_left = a.part_k / KC;
#pragma unroll
        for (int t = 0; t < kTM; ++t)
#pragma unroll
          for (int j = 0; j < kTN; ++j) {
            sum[t][j] = first_part ? acc[t][j] : sum[t][j] + acc[t][j];
            acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        first_part = false;
      }
    }
    buf = buf + 1 == STAGES ? 0 : buf + 1;
  }
  if constexpr (kParts) {
#pragma unroll
    for (int t = 0; t < kTM; ++t)
#pragma unroll
      for (int j = 0; j < kTN; ++j) acc[t][j] = sum[t][j];
  }

  // Epilogue: lane (r, g) holds columns 4g .. 4g + 3 of a tile for token r.
  if constexpr (EPI == kPartial) {
#pragma unroll
    for (int t = 0; t < kTM; ++t) {
      const int tok = m0 + 16 * (wm * kTM + t) + r;
      if (tok >= a.m) continue;
#pragma unroll
      for (int j = 0; j < kTN; ++j) {
        const int64_t col = n0 + 16 * (wn * kTN + j) + 4 * g;
        if (col < a.n)  // n is a multiple of 4
          *reinterpret_cast<f32x4*>(a.part + ((int64_t)split * a.m + tok) * a.n + col) = acc[t][j];
      }
    }
  } else {
    constexpr int kOut = EPI == kSiluMul ? kTN / 2 : kTN;
    float any = 0.f;  // NaN if any output is
#pragma unroll
    for (int t = 0; t < kTM; ++t) {
      const int tok = m0 + 16 * (wm * kTM + t) + r;
      if (tok >= a.m) continue;
#pragma unroll
      for (int j = 0; j < kOut; ++j) {
        const int64_t col = n0 + 16 * (wn * kOut + j) + 4 * g;
        bf16_t* dst = a.y + (a.y_packed ? packed_offset(tok, col, a.n) : (int64_t)tok * a.ldy + col);
        const bool whole = col + 3 < a.n;
        // bf16 outputs in pairs (hardware rounding to nearest even).
        uint32_t pair[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float lo = acc[t][j][2 * e], hi = acc[t][j][2 * e + 1];
          if constexpr (EPI == kSiluMul) {
            const f32x4 up = acc[t][kOut + j];
            const uint32_t v = pack_bf_hw(lo, hi), u = pack_bf_hw(up[2 * e], up[2 * e + 1]);
            const uint32_t sl = pack_bf_hw(silu_bf16(lo_bf(v)), silu_bf16(hi_bf(v)));
            lo = lo_bf(sl) * lo_bf(u);
            hi = hi_bf(sl) * hi_bf(u);
          } else if constexpr (EPI == kAddResidual) {
            const uint32_t v = pack_bf_hw(lo, hi);
            uint32_t old = 0u;
            if (whole) {
              old = reinterpret_cast<const uint32_t*>(dst)[e];
            } else {
              for (int i = 0; i < 2; ++i)
                if (col + 2 * e + i < a.n) old |= (uint32_t)dst[2 * e + i] << (16 * i);
            }
            lo = lo_bf(v) + lo_bf(old);
            hi = hi_bf(v) + hi_bf(old);
          }
          pair[e] = pack_bf_hw(lo, hi);
          any = __builtin_elementwise_maximum(__builtin_elementwise_maximum(any, lo), hi);
        }
        if (whole) {
          *reinterpret_cast<u32x2*>(dst) = u32x2{pair[0], pair[1]};
        } else {
          for (int e = 0; e < 4; ++e)
            if (col + e < a.n) dst[e] = (bf16_t)((pair[e >> 1] >> (16 * (e & 1))) & 0xffffu);
        }
      }
    }
    // The hardware's rounding keeps a NaN's payload; the 64-row kernel's NaN is canonical, so the lane's are made so.
    if (any != any) {
      for (int t = 0; t < kTM; ++t) {
        const int tok = m0 + 16 * (wm * kTM + t) + r;
        if (tok >= a.m) break;
        for (int c = 0; c < 4 * kOut; ++c) {
          const int64_t col = n0 + 16 * (wn * kOut + (c >> 2)) + 4 * g + (c & 3);
          bf16_t* dst = a.y + (a.y_packed ? packed_offset(tok, col, a.n) : (int64_t)tok * a.ldy + col);
          if (col < a.n && (*dst & 0x7fffu) > 0x7f80u) *dst = (bf16_t)0x7fc0u;
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int STAGES, int KC, bool kParts, int EPI>
int launch(const TileArgs& t, int parts, hipStream_t s) {
  constexpr size_t lds = (size_t)STAGES * (BM + BN) * 2 * KC;
  const auto kernel = gemm_tile_kernel<BM, BN, WM, WN, STAGES, KC, kParts, EPI>;
  static std::atomic<uint64_t> lds_allowed{0};
  const int st = allow_dynamic_lds(lds_allowed, (const void*)kernel, (int)lds);
  if (st) return st;
  constexpr int kCols = EPI == kSiluMul ? BN / 2 : BN;
  const int64_t tiles_m = (t.m + BM - 1) / BM, tiles_n = (t.n + kCols - 1) / kCols;
  const int k_slice = (int)(t.k / t.k_splits);
  const KernelArgs a{t.x, t.w, t.y, t.part, t.ldx, t.k, t.n, t.ldy, (int)t.m, (int)tiles_m, (int)tiles_n, k_slice,
                     k_slice / parts, t.x_packed, t.w_packed, t.y_packed};
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n * t.k_splits)), dim3(64 * WM * WN), lds, s, a);
  return OXR_LAUNCH_STATUS();
}

template <int EPI>
int dispatch(const TileArgs& t, int tile, int parts, hipStream_t s) {
  if constexpr (EPI != kPartial) {  // partial sums are never one chain
    if (tile == 0) return launch<256, 256, 2, 4, 2, 64, false, EPI>(t, parts, s);
    if (tile == 1) return launch<256, 128, 4, 2, 3, 64, false, EPI>(t, parts, s);
  }
  switch (tile) {
    case 2: return launch<128, 128, 4, 2, 4, 64, true, EPI>(t, parts, s);
    case 3: return launch<128, 64, 4, 2, 3, 128, true, EPI>(t, parts, s);
    case 4: return launch<64, 64, 4, 2, 4, 128, true, EPI>(t, parts, s);
    default: return OXR_ERR_UNSUPPORTED;
  }
}

// Tile with the least estimated time: rounds of tiles over the 256 CUs (one workgroup each: LDS) times the
// time of a tile, which is a cost per 64 k and a fixed one (pipeline fill, epilogue; more for SiLU * mul).
// Measured on MI355X, us: one tile of K = 2048 and K = 6144 by itself 48 / 121, 29 / 72, 22 / 55, 13 / 33 and
// 10 / 25 from the largest tile to the smallest.  At 256 rows the 12288-row gate_up weight takes 23 / 30 / 32
// with 128 x 128 / 128 x 64 / 64 x 64 tiles (192, 384 and 768 of them) and 51 / 30 with the two large ones;
// the 4096-row qkv weight 21 / 12 / 10 (64, 128 and 256 tiles); 4096 rows of gate_up 183 (256 x 256) / 204 /
// 266.  The large tiles sum k in one chain, so they serve only the calls without partial sums (one_chain).
struct TileCost {
  int bm, bn;
  float per_k64, fixed, fixed_silu;
};
constexpr TileCost kTiles[] = {{256, 256, 1.2f, 13.f, 18.f},
                               {256, 128, 0.75f, 9.f, 9.f},
                               {128, 128, 0.51f, 5.f, 5.5f},
                               {128, 64, 0.29f, 3.5f, 5.f},
                               {64, 64, 0.21f, 3.2f, 4.f}};
int pick_tile(const TileArgs& t, int epilogue, bool one_chain) {
  int best = 2;
  float best_time = 0.f;
  for (int i = one_chain ? 0 : 2; i < 5; ++i) {
    const TileCost& c = kTiles[i];
    const int64_t cols = epilogue == kSiluMul ? c.bn / 2 : c.bn;
    const int64_t tiles = ((t.m + c.bm - 1) / c.bm) * ((t.n + cols - 1) / cols) * t.k_splits;
    const float time = (float)((tiles + 255) / 256) * ((float)(t.k / t.k_splits / 64) * c.per_k64 +
                                                       (epilogue == kSiluMul ? c.fixed_silu : c.fixed));
    if (i == (one_chain ? 0 : 2) || time < best_time) {
      best = i;
      best_time = time;
    }
  }
  return best;
}

}  // namespace

bool gemm_tile_supported(const TileArgs& t) {
  // A tile's row offsets are 32-bit, its workgroups at most 2^31 - 1 (counted for the smallest tile).
  constexpr int64_t kMaxStride = (int64_t)1 << 22;
  return t.ldx <= kMaxStride && t.k <= kMaxStride && t.m <= 0x7fffffff &&
         ((t.m + 63) / 64) * ((t.n + 31) / 32) * t.k_splits <= 0x7fffffff;
}

int launch_gemm_tile(const TileArgs& t, int epilogue, int parts, bool one_chain, hipStream_t s) {
  if (one_chain) parts = 1;
  const int tile = pick_tile(t, epilogue, one_chain);
  switch (epilogue) {
    case kStore: return dispatch<kStore>(t, tile, parts, s);
    case kSiluMul: return dispatch<kSiluMul>(t, tile, parts, s);
    case kAddResidual: return dispatch<kAddResidual>(t, tile, parts, s);
    case kPartial: return dispatch<kPartial>(t, tile, parts, s);
    default: return OXR_ERR_INVALID_ARG;
  }
}

}  // namespace oxr
