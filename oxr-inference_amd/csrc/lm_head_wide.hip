// LM head for 33 to 256 token rows (packed weight), gfx950.
//
// At 256 rows the head does 159 GFLOP on a 622 MB weight, at the ridge of the matrix cores and HBM (about
// 100 us each on this card), so both have to run at their rate at once.  One persistent workgroup of 8 waves
// per CU owns a balanced contiguous range of 32-row vocab tiles, taken 8 at a time (a group); all token rows
// times a group are multiplied with 32x32x16 products, wave (wm, wn) taking half of the token rows and two
// vocab tiles (128 accumulators at 256 rows).
// * Both operands pass through LDS in 32-k stages (1 KiB blocks of the packed layouts, 16-byte
//   global_load_lds): a ring of 4 stages of token rows and 6 or 8 of weight.  Waves 0-3 issue the weight's
//   blocks and waves 4-7 the token rows': the vector memory counter is in order, so a wave that loaded both
//   could not wait for a young token-row block without waiting for every older weight block, which is
//   requested up to 6 stages ahead because it comes from HBM.
// * The barrier at the start of stage c says that stage c + 1 has landed, so stage c's last products already
//   read the next stage's first fragments and no LDS latency shows at the barrier.
// * A range's last group often has few tiles (18 or 19 tiles a CU at vocab 151,936: 8 + 8 + 2 or 3).  With at
//   most 4 each wave takes one tile, which halves the group's products.
// * Epilogue per group: bf16 logits as 16-byte stores (two lanes' halves exchanged), and the running best of
//   each token as one 32-bit integer (signed bf16 key, column) per lane: 4 instructions a logit.
//
// Kernel alone at vocab 151,936, hidden 2048, ids only, us: 256 rows 165 (185 with logits), 96 rows 119, 64 rows
// 104 (6.0 TB/s).  Up to 128 rows the HBM stream bounds it; the weight is loaded non-temporally there (64 rows: 111
// without).  At 256 rows the parts by themselves take 96 (products: the clock falls from 2.5 to 2.0 GHz under
// them), 45 (fragment reads) and 118 (loads); what is left is that a wave whose loads wait to be issued does not
// multiply.  Neither the ring's depth, nor wave priorities, nor non-temporal weight loads (171) move it.
//
// Each logit is one chain of products over k in ascending order, whatever the number of rows.
#include "lm_head_wide.h"

#include <type_traits>

#include "argmax_key.h"

namespace oxr {
namespace {

typedef short i16x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;
constexpr int kGroup = 8;    // vocab tiles per group
constexpr int kXSlots = 4;   // stages of token rows in LDS
constexpr int kWBytes = kGroup * 2048;  // a stage of weight: 32 rows x 32 k per tile

// Two packed bf16 values as signed 16-bit keys: ordered like the values, -0 equal to +0 (no NaN).
__device__ __forceinline__ uint32_t key_pair(uint32_t p) {
  const i16x2 v = __builtin_bit_cast(i16x2, p);
  const i16x2 s = v >> 15;
  return __builtin_bit_cast(uint32_t, (i16x2)(((v & (i16x2)(0x7fff)) ^ s) - s));
}

// TT: 32-token tiles (2, 4 or 8; rows past M are padding whose results nobody reads).
// kMask: weight blocks past the range's end are not read.  Where the loads bound the kernel they cost what the others
// do: 32,000 vocab rows are 4 tiles a CU, half a group (128 token rows 44.2 us, so 39.6; 151,936 rows 64 token rows
// ids only 109.9 / 107.1).  At 256 token rows it makes no difference, and where a CU has one tile the mask is the
// longer way to its next load (1000 vocab rows 31.0 / 32.3).
template <int TT, bool kMask>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void lm_head_wide_kernel(
    const bf16_t* __restrict__ xp, int M, const bf16_t* __restrict__ w, int K, int64_t N,
    bf16_t* __restrict__ logits, int wide_stores, uint64_t* __restrict__ best_out) {
  constexpr int kTT = TT / 2;             // token tiles per wave
  constexpr int kXBytes = TT * 2048;      // a stage of token rows
  constexpr int kWSlots = TT == 8 ? 6 : 8;
  constexpr int kXL = TT * 2 / 4;         // token-row blocks per stage of each of waves 4-7
  constexpr int kWL = kGroup * 2 / 4;     // weight blocks per stage of each of waves 0-3
  extern __shared__ __align__(1024) char lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int wm = wave >> 2, wn = wave & 3;
  const int64_t nt32 = (N + 31) / 32, w_last = (N + 15) / 16 - 1;
  const int64_t lo = (int64_t)blockIdx.x * nt32 / gridDim.x, hi = (int64_t)(blockIdx.x + 1) * nt32 / gridDim.x;
  const int groups = (int)((hi - lo + kGroup - 1) / kGroup);
  const int steps = K / 32;  // stages of a group

  // Loads.  Waves 0-3: blocks 4 wave .. + 3 of a weight stage (tile b / 2, 16-row half b % 2); waves 4-7:
  // blocks of a token-row stage (16-row piece b).  Every stage issues the same number of loads: stages past the last
  // group repeat it, tiles past the range's end are loaded with no lane active (kMask) or re-read its last one.
  const bool weight_wave = wave < 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const char* src[4];
  uint32_t lanes[2] = {~0u, ~0u};  // of the loads of each of the wave's tiles: all or none
  int load_step = 0, load_group = 0, load_slot = 0;
  auto sources = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (weight_wave) {
        const int b = kWL * wave + u;
        const int64_t vt = lo + (int64_t)min(load_group, groups - 1) * kGroup + (b >> 1);
        src[u] = (const char*)(w + min(2 * min(vt, hi - 1) + (b & 1), w_last) * (K * 16));
        lanes[u >> 1] = __builtin_amdgcn_readfirstlane(vt < hi ? ~0u : 0u);
      } else {
        const int b = kXL * (wave - 4) + u % kXL;
        src[u] = (const char*)(xp + (int64_t)min(b, (M + 15) / 16 - 1) * (K * 16));
      }
    }
  };
  const uint32_t lane_off = lane * 16;
  const int my_slots = weight_wave ? kWSlots : kXSlots, my_bytes = weight_wave ? kWBytes : kXBytes;
  const uint32_t my_ring = lds0 + (weight_wave ? kXSlots * kXBytes + kWL * wave * 1024 : kXL * (wave - 4) * 1024);
  auto issue1 = [&](int u) __attribute__((always_inline)) {
    const uint32_t at = my_ring + load_slot * my_bytes + u * 1024;
    if (TT < 8 && weight_wave) dma_block_nt<kMask>(src[u], lane_off, at, lanes[u >> 1]);
    else if (u < kXL || weight_wave) dma_block(src[u], lane_off, at);
  };
  auto issued = [&]() __attribute__((always_inline)) {
    load_slot = load_slot + 1 == my_slots ? 0 : load_slot + 1;
    if (++load_step == steps) {
      load_step = 0;
      ++load_group;
      sources();
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) src[u] += 1024;
    }
  };
  // Stage c + 1 has landed when at most the stages requested after it are outstanding.
  auto wait_next = [&]() __attribute__((always_inline)) {
    if (weight_wave) wait_vm<(kWSlots - 3) * kWL>();
    else wait_vm<(kXSlots - 3) * kXL>();
    asm volatile("s_barrier" ::: "memory");
  };

  sources();
  for (int s = 0; s < my_slots - 1; ++s) {
#pragma unroll
    for (int u = 0; u < 4; ++u) issue1(u);
    issued();
  }

  // Fragment of k16 step kk of a stage: lane (n, h) reads row n of a 32-row tile (two 1 KiB blocks).
  const int frag = (n >> 4) * 1024 + h * 256 + (n & 15) * 16;
  const int x_off = wm * kTT * 2048 + frag;
  u32x4 xf[2][kTT], wf[2][2];
  int x_slot = 0, w_slot = 0;
  auto tiles_of = [&](int gi) { return (int)min(hi - lo - (int64_t)gi * kGroup, (int64_t)kGroup); };
  auto w_off_of = [&](bool half) { return kXSlots * kXBytes + (half ? wn : 2 * wn) * 2048 + frag; };

  wait_next();
  bool half = tiles_of(0) <= kGroup / 2;
  int w_off = w_off_of(half);
#pragma unroll
  for (int tt = 0; tt < kTT; ++tt) xf[0][tt] = *reinterpret_cast<const u32x4*>(lds + x_off + 2048 * tt);
#pragma unroll
  for (int v = 0; v < 2; ++v) wf[0][v] = *reinterpret_cast<const u32x4*>(lds + w_off + 2048 * v);

  f32x16 acc[kTT][2];
  uint64_t best[kTT];
#pragma unroll
  for (int tt = 0; tt < kTT; ++tt) best[tt] = 0;

  // The stages of one group, NV vocab tiles per wave; next_w_off: the next group's.
  auto run_group = [&](auto nv, int next_w_off) __attribute__((always_inline)) {
    constexpr int NV = decltype(nv)::value;
#pragma unroll
    for (int tt = 0; tt < kTT; ++tt)
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[tt][v][e] = 0.f;
    for (int s = 0; s < steps; ++s) {
      wait_next();
      const char* xa = lds + x_slot * kXBytes + x_off;
      const char* wa = lds + w_slot * kWBytes + w_off;
      x_slot = (x_slot + 1) & (kXSlots - 1);
      w_slot = w_slot + 1 == kWSlots ? 0 : w_slot + 1;
      const char* xn = lds + x_slot * kXBytes + x_off;
      const char* wnx = lds + w_slot * kWBytes + (s + 1 == steps ? next_w_off : w_off);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        // While k16 step kk is multiplied, the fragments of the next (kk = 1: the next stage's first) are read.
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) {
          if (tt == 0) {
#pragma unroll
            for (int v = 0; v < 2; ++v)
              wf[kk ^ 1][v] = *reinterpret_cast<const u32x4*>((kk ? wnx : wa + 512) + 2048 * v);
          }
          xf[kk ^ 1][tt] = *reinterpret_cast<const u32x4*>((kk ? xn : xa + 512) + 2048 * tt);
          if (kk == 0) {
#pragma unroll
            for (int u = tt * 4 / kTT; u < (tt + 1) * 4 / kTT; ++u) issue1(u);
            if (tt == kTT - 1) issued();
          }
#pragma unroll
          for (int v = 0; v < NV; ++v) acc[tt][v] = mfma_32x32x16(wf[kk][v], xf[kk][tt], acc[tt][v]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };

  // Lane (n, h) holds logits of vocab rows 32 vt + 8 m4 + 4h + j (element 4 m4 + j) for token 32 tt + n.
  auto finish_group = [&](auto nv, int gi) __attribute__((always_inline)) {
    constexpr int NV = decltype(nv)::value;
    const int64_t vt0 = lo + (int64_t)gi * kGroup + NV * wn, row0 = 32 * vt0;  // this wave's first tile, row
    int key[kTT];
#pragma unroll
    for (int tt = 0; tt < kTT; ++tt) key[tt] = (int)0x80000000;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int64_t vt = vt0 + v;
      if (vt >= hi) break;  // wave-uniform
      const bool whole = 32 * vt + 32 <= N;
#pragma unroll
      for (int tt = 0; tt < kTT; ++tt) {
        const f32x16& a = acc[tt][v];
        const int tok = 32 * (wm * kTT + tt) + n;
        uint32_t p[4][2];
        float m = a[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) m = __builtin_elementwise_maximum(m, a[e]);  // NaN if any is
        if (whole && !__builtin_amdgcn_ballot_w64(m != m)) {
#pragma unroll
          for (int m4 = 0; m4 < 4; ++m4)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              p[m4][q] = pack_bf_hw(a[4 * m4 + 2 * q], a[4 * m4 + 2 * q + 1]);
              const uint32_t k2 = key_pair(p[m4][q]);
              const int col = 63 - (32 * v + 8 * m4 + 2 * q);  // within the wave's rows; 4h is added at the end
              key[tt] = max(key[tt], max((int)((k2 << 16) | (uint32_t)col), (int)((k2 & 0xffff0000u) | (uint32_t)(col - 1))));
            }
        } else {
#pragma unroll
          for (int m4 = 0; m4 < 4; ++m4)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              p[m4][q] = pack_bf(a[4 * m4 + 2 * q], a[4 * m4 + 2 * q + 1]);
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const uint32_t b16 = (p[m4][q] >> (16 * e)) & 0xffffu;
                const uint32_t k16 = (b16 & 0x7fffu) > 0x7f80u ? 0x7fffu : key_pair(b16) & 0xffffu;  // NaN largest
                const int c = 32 * v + 8 * m4 + 2 * q + e;
                if (row0 + c + 4 * h < N) key[tt] = max(key[tt], (int)((k16 << 16) | (uint32_t)(63 - c)));
              }
            }
        }
        if (logits == nullptr || tok >= M) continue;
        bf16_t* row = logits + (int64_t)tok * N + 32 * vt;
        if (wide_stores && whole) {
          // Lane h = 0 gets rows 8 m4 .. + 7 of its token for the even m4, lane h = 1 for the odd.
#pragma unroll
          for (int m4 = 0; m4 < 4; m4 += 2) {
            const auto r0 = __builtin_amdgcn_permlane32_swap(p[m4][0], p[m4 + 1][0], false, false);
            const auto r1 = __builtin_amdgcn_permlane32_swap(p[m4][1], p[m4 + 1][1], false, false);
            st128(row + 8 * (m4 + h), u32x4{r0[0], r1[0], r0[1], r1[1]});
          }
        } else {
#pragma unroll
          for (int m4 = 0; m4 < 4; ++m4) {
            const int c = 8 * m4 + 4 * h;
            if (32 * vt + c + 3 < N) {
              *reinterpret_cast<u32x2*>(row + c) = u32x2{p[m4][0], p[m4][1]};
            } else {
              for (int j = 0; j < 4; ++j)
                if (32 * vt + c + j < N) row[c + j] = (bf16_t)((p[m4][j >> 1] >> (16 * (j & 1))) & 0xffffu);
            }
          }
        }
      }
    }
#pragma unroll
    for (int tt = 0; tt < kTT; ++tt) {
      if (key[tt] == (int)0x80000000) continue;
      const int k = key[tt] >> 16;
      const uint32_t bits = k >= 0 ? (uint32_t)k : 0x8000u | (uint32_t)(-k);
      const uint64_t b = argmax_key(bits << 16, (uint32_t)(row0 + 63 - (key[tt] & 63) + 4 * h));
      best[tt] = b > best[tt] ? b : best[tt];
    }
  };

  constexpr std::integral_constant<int, 1> one{};
  constexpr std::integral_constant<int, 2> two{};
  for (int gi = 0; gi < groups; ++gi) {
    const bool next_half = gi + 1 < groups && tiles_of(gi + 1) <= kGroup / 2;
    const int next = w_off_of(gi + 1 < groups ? next_half : half);
    if (half) {
      run_group(one, next);
      finish_group(one, gi);
    } else {
      run_group(two, next);
      finish_group(two, gi);
    }
    half = next_half;
    w_off = next;
  }

  // Best key per token: the two lane halves, then the 4 waves of a token half through LDS (every load into
  // it has landed after this wait and barrier).
  wait_vm<0>();
  __syncthreads();
  uint64_t* const keys = reinterpret_cast<uint64_t*>(lds);  // [4][32 TT]
#pragma unroll
  for (int tt = 0; tt < kTT; ++tt) {
    const uint32_t olo = __shfl_xor((uint32_t)best[tt], 32, kWave);
    const uint32_t ohi = __shfl_xor((uint32_t)(best[tt] >> 32), 32, kWave);
    const uint64_t o = ((uint64_t)ohi << 32) | olo;
    if (h == 0) keys[wn * 32 * TT + 32 * (wm * kTT + tt) + n] = o > best[tt] ? o : best[tt];
  }
  __syncthreads();
  if (tid < M) {
    uint64_t b = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) b = keys[q * 32 * TT + tid] > b ? keys[q * 32 * TT + tid] : b;
    best_out[(int64_t)blockIdx.x * M + tid] = b;
  }
}

template <int TT, bool kMask>
int launch(const bf16_t* xp, int M, const bf16_t* w, int64_t K, int64_t N, bf16_t* logits, uint64_t* best, int grid,
           hipStream_t s) {
  constexpr int lds = kXSlots * TT * 2048 + (TT == 8 ? 6 : 8) * kWBytes;
  const auto kernel = lm_head_wide_kernel<TT, kMask>;
  static std::atomic<uint64_t> lds_allowed{0};
  const int st = allow_dynamic_lds(lds_allowed, (const void*)kernel, lds);
  if (st) return st;
  const int wide_stores = logits != nullptr && (uintptr_t)logits % 16 == 0 && N % 8 == 0;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * kWaves), lds, s, xp, M, w, (int)K, N, logits, wide_stores,
                     best);
  return OXR_LAUNCH_STATUS();
}

}  // namespace

int launch_lm_head_wide(const bf16_t* xp, int M, const bf16_t* w, int64_t K, int64_t N, bf16_t* logits,
                        uint64_t* best, int grid, hipStream_t s) {
  const bool mask = (N + 31) / 32 > grid;
  if (M <= 64) return (mask ? launch<2, true> : launch<2, false>)(xp, M, w, K, N, logits, best, grid, s);
  if (M <= 128) return (mask ? launch<4, true> : launch<4, false>)(xp, M, w, K, N, logits, best, grid, s);
  return launch<8, false>(xp, M, w, K, N, logits, best, grid, s);
}

}  // namespace oxr
