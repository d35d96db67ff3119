// Attention of few queries on many keys (decoding: at most 16 queries a head), fp16 in and out, fp32 accumulation.
//
// Bound by reading K and V once.  The prompt kernels give every wave 32 queries of its own and share a key tile between
// waves; with one query three of four waves would multiply copies of it.  Here the waves share the queries and cut
// the KEYS: a wave walks every fourth 32-key tile of its workgroup's part of the keys on its own, from copies straight into
// its own LDS (global_load_lds, 16 bytes a lane), with no barrier in the loop, and the four running (maximum, sum, O)
// meet once at the end.  What is in flight is what the rate depends on: a compute unit has 64 to 128 KB of copies on the
// way (its share of 6 TB/s times a microsecond or two of latency is 25 to 50 KB).
//
// Products on v_mfma_f32_16x16x32_f16, both transposed so that a lane has one query: S^T = K Q^T (A: keys, from LDS rows,
// B: the resident queries), O^T = V^T P^T (A: V^T by the transposing LDS read, B: the weights as they come out of the
// first product, the contraction taking the keys in the order a lane holds them).
//
// Measured (microseconds, with the 4-wave prompt kernel before): 1 query a head, 256 heads of 128, 4096 keys 116 -> 91 -> 77
// with copies that leave no lines in the caches (7.0 TB/s; nothing but such copies reaches 7.1); 8 heads, 32768 keys 41 -> 26; 16 queries,
// 24 heads of 128, 1753 keys 34 -> 10.
//
// The keys of a head are cut over workgroups (parts) where heads alone do not fill the chip; attn_merge_kernel
// (flash_attn.hip) merges what the parts leave.
#include <algorithm>

#include "fa_common.h"
#include "ftk_common.h"

namespace ftk {

constexpr int kDecKeys = 32;     // keys of a tile
constexpr int kDecWaves = 4;
// The reference before any score: finite, so that a tile whose scores are all -inf weighs nothing (-inf - -inf is a NaN).
// Every finite score is above it or equal to it, and 2^(kNoRef - score) is zero.
constexpr float kNoRef = -3.402823466e38f;

// LDS slots of a row's 16-byte chunks: chunk c of row r sits in slot c ^ decode_swizzle(r).  The 16 lanes that an LDS
// read of 16 bytes serves together hold one chunk of 16 rows; these are then 16 different places of the 256-byte bank line.
template <int D>
__device__ __forceinline__ int decode_swizzle(int row) {
  if (D == 128) return row & 15;
  if (D == 64) return (row >> 1) & 7;
  return (row >> 2) & 3;
}

template <int D>
struct DecodeShape {
  static constexpr int TILE = kDecKeys * D * 2;                 // bytes of a K or V tile
  static constexpr int COPIES = TILE / 1024;                    // 1 KB copies of a tile
  static constexpr int STAGES = D >= 96 ? 2 : 4;                // tiles of a wave's ring
  static constexpr size_t LDS = (size_t)kDecWaves * STAGES * 2 * TILE;
};

// ONCE: K and V are too large for the caches to keep from call to call (launch_decode).
template <int D, bool ONCE>
__global__ __launch_bounds__(kDecWaves * 64) void flash_decode_kernel(const _Float16* __restrict__ Q, const _Float16* __restrict__ K,
                                                                      const _Float16* __restrict__ V, _Float16* __restrict__ O, int Sq,
                                                                      int Skv, float scale_log2e, int nparts, int part_keys,
                                                                      float* __restrict__ part_o, float* __restrict__ part_ml) {
  using S = DecodeShape<D>;
  constexpr int KS = D / 32;            // k steps of S^T
  constexpr int DT = D / 16;            // tiles of O^T
  constexpr int CH = D / 8;             // 16-byte chunks of a row
  constexpr int STAGES = S::STAGES;
  using lds_v4s = __attribute__((address_space(3))) v4s;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const int bh = blockIdx.x / nparts, part = blockIdx.x - bh * nparts;
  const int first = part * part_keys, last = min(Skv, first + part_keys);
  const int ntiles = (last - first + kDecKeys - 1) / kDecKeys;
  const _Float16* const Kg = K + (size_t)bh * Skv * D;
  const _Float16* const Vg = V + (size_t)bh * Skv * D;
  unsigned char* const ring = smem + wave * (STAGES * 2 * S::TILE);

  // copies: a copy fills 64 slots in a row; slot p is row p / CH, and holds the chunk the swizzle gives it.  Rows past the
  // last key repeat it (their weights are zero).
  auto issue = [&](int t, int stage) __attribute__((always_inline)) {
    const int key0 = first + t * kDecKeys;
    unsigned char* const dst = ring + stage * (2 * S::TILE);
    const char* const kb = reinterpret_cast<const char*>(Kg + (size_t)key0 * D);
    const char* const vb = reinterpret_cast<const char*>(Vg + (size_t)key0 * D);
    const int most = Skv - 1 - key0;
#pragma unroll
    for (int i = 0; i < S::COPIES; ++i) {
      const int p = 64 * i + lane, row = p / CH, slot = p - row * CH;
      const unsigned off = (unsigned)(min(row, most) * (2 * D) + (slot ^ decode_swizzle<D>(row)) * 16);
      if constexpr (ONCE) {
        lds_dma16_once(kb, off, dst + 1024 * i);
        lds_dma16_once(vb, off, dst + S::TILE + 1024 * i);
      } else {
        lds_dma16(kb, off, dst + 1024 * i);
        lds_dma16(vb, off, dst + S::TILE + 1024 * i);
      }
    }
  };

  // the queries are asked for before the first tiles and pre-multiplied by scale * log2 e behind them; rows past the
  // last repeat it
  v8h qf[KS];
  const _Float16* const q0 = Q + ((size_t)bh * Sq + min(m, Sq - 1)) * D + 8 * kg;
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const v8h*>(q0 + 32 * s);
  asm volatile("" ::: "memory");

  v4f o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = v4f{0.f, 0.f, 0.f, 0.f};
  float ref = kNoRef, l = 0.0f;

  // this wave's tiles: wave, wave + 4, ...
  const int mine = ntiles > wave ? (ntiles - wave + kDecWaves - 1) / kDecWaves : 0;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (i < mine) issue(wave + kDecWaves * i, i);
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[s][e] = (_Float16)((float)qf[s][e] * scale_log2e);
  int stage = 0;
  for (int i = 0; i < mine; ++i) {
    const int t = wave + kDecWaves * i;
    // the stage the tile before used is free: everything read from it has been used
    if (i + STAGES - 1 < mine) {
      issue(t + kDecWaves * (STAGES - 1), stage == 0 ? STAGES - 1 : stage - 1);
      __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * S::COPIES * (STAGES - 1)) & 15) | (((2 * S::COPIES * (STAGES - 1)) >> 4) << 14));
    } else {
      __builtin_amdgcn_s_waitcnt(0x0F70);   // the last few: vmcnt(0)
    }
    asm volatile("" ::: "memory");
    const unsigned char* const kt = ring + stage * (2 * S::TILE);
    const unsigned char* const vt = kt + S::TILE;
    v4f sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int row = 16 * h + m;
        const v8h a = *reinterpret_cast<const v8h*>(kt + row * (2 * D) + (((4 * s + kg) ^ decode_swizzle<D>(row)) * 16));
        sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qf[s], sc[h], 0, 0, 0);
      }
    }
    // lane (query m, kg) has keys 16 h + 4 kg + r
    if (first + t * kDecKeys + kDecKeys > last) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (first + t * kDecKeys + 16 * h + 4 * kg + r >= last) sc[h][r] = -INFINITY;
    }
    // the reference maximum moves only when a score is above it by 2^8 in the weights
    float mx = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])), fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    if (__builtin_amdgcn_ballot_w64(!(mx <= ref + 8.0f)) != 0) {
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float moved = fmaxf(ref, mx);
      const float alpha = __builtin_amdgcn_exp2f(ref - moved);
      ref = moved;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;
    }
    v8h p;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[4 * h + r] = (_Float16)__builtin_amdgcn_exp2f(sc[h][r] - ref);
        l += (float)p[4 * h + r];
      }
    // O^T: lane group kg contracts keys 4 kg .. +3 and 16 + 4 kg .. +3; 16 lanes hand in a block of 4 keys x 16 columns
    const int a4 = (lane & 15) >> 2, b4 = lane & 3;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      v4s half[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 16 * h + 4 * kg + a4;
        const unsigned char* src = vt + row * (2 * D) + (((2 * dt + (b4 >> 1)) ^ decode_swizzle<D>(row)) * 16) + 8 * (b4 & 1);
        half[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src));
      }
      typedef short v8s __attribute__((ext_vector_type(8)));
      const v8s both = {half[0][0], half[0][1], half[0][2], half[0][3], half[1][0], half[1][1], half[1][2], half[1][3]};
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, both), p, o[dt], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    stage = stage == STAGES - 1 ? 0 : stage + 1;
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // ---- the four waves meet: O as [wave][tile][lane] in LDS, (ref, l) behind it
  __syncthreads();
  v4f* const so = reinterpret_cast<v4f*>(smem);
  float* const sml = reinterpret_cast<float*>(smem + kDecWaves * DT * 64 * sizeof(v4f));   // [wave][query][2]
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) so[(wave * DT + dt) * 64 + lane] = o[dt];
  if (kg == 0) {
    sml[(wave * 16 + m) * 2] = ref;
    sml[(wave * 16 + m) * 2 + 1] = l;
  }
  __syncthreads();
  const int q = tid & 15;
  if (q >= Sq) return;
  float top = kNoRef, sum = 0.0f, w[kDecWaves];
#pragma unroll
  for (int i = 0; i < kDecWaves; ++i) top = fmaxf(top, sml[(i * 16 + q) * 2]);
#pragma unroll
  for (int i = 0; i < kDecWaves; ++i) {
    w[i] = __builtin_amdgcn_exp2f(sml[(i * 16 + q) * 2] - top);
    sum += w[i] * sml[(i * 16 + q) * 2 + 1];
  }
  const float inv = 1.0f / sum;
  for (int g = tid >> 4; g < D / 4; g += kDecWaves * 4) {   // columns 4 g .. +3: tile g / 4, lane group g % 4
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kDecWaves; ++i) {
      const v4f v = so[(i * DT + (g >> 2)) * 64 + 16 * (g & 3) + q];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += w[i] * v[r];
    }
    if (nparts == 1) {
      const v4h out = {(_Float16)(acc[0] * inv), (_Float16)(acc[1] * inv), (_Float16)(acc[2] * inv), (_Float16)(acc[3] * inv)};
      *reinterpret_cast<v4h*>(O + ((size_t)bh * Sq + q) * D + 4 * g) = out;
    } else {
      *reinterpret_cast<v4f*>(part_o + (((size_t)bh * nparts + part) * Sq + q) * D + 4 * g) = acc;
    }
  }
  if (nparts > 1 && tid < 16) {
    float* ml = part_ml + 2 * (((size_t)bh * nparts + part) * Sq + q);
    ml[0] = top;
    ml[1] = sum;
  }
}

// How the keys of bh heads are cut: the number of parts (1: not at all) and the keys of a part, a multiple of four tiles.
// A compute unit holds one workgroup at a time (its LDS), so what is weighed is rounds of workgroups times the steps of a
// workgroup, a tile for each of its four waves: 64 KB at D 128, 2.6 us at a compute unit's share of 6 TB/s (2.3 at the 7 that copies which leave no lines behind reach), against
// about 3 us that a workgroup and 4 us that the merge (a launch) cost beside that.
int decode_parts(long long bh, int Skv, int D, int cus, int* part_keys) {
  const int groups = (Skv + kDecWaves * kDecKeys - 1) / (kDecWaves * kDecKeys);   // a tile for each wave
  int best = 1;
  double best_cost = 1e30;
  for (int n = 1; n <= 64 && n <= groups; ++n) {
    const int per = (groups + n - 1) / n, parts = (groups + per - 1) / per;
    if (parts != n) continue;
    const double rounds = (double)((bh * n + cus - 1) / cus);
    const double cost = rounds * (3.0 + per * (2.6 * D / 128)) + (n > 1 ? 4.0 : 0.0);
    if (cost < 0.97 * best_cost) {   // more parts are more workspace: not for a rounding of the rounds
      best_cost = cost;
      best = n;
    }
  }
  const int per = (groups + best - 1) / best;
  *part_keys = best == 1 ? Skv : per * kDecWaves * kDecKeys;
  return best;
}

template <int D, bool ONCE>
static int launch(const void* Q, const void* K, const void* V, void* O, int BH, int Sq, int Skv, float scale, int nparts, int part_keys,
                  float* part_o, float* part_ml, hipStream_t s) {
  static DeviceOnce attr_once;
  unsigned attr_bit;
  if (attr_once.pending(&attr_bit)) {
    FTK_HIP(hipFuncSetAttribute((const void*)flash_decode_kernel<D, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)DecodeShape<D>::LDS));
    attr_once.done(attr_bit);
  }
  hipLaunchKernelGGL((flash_decode_kernel<D, ONCE>), dim3((unsigned)(BH * nparts)), dim3(kDecWaves * 64), DecodeShape<D>::LDS, s, (const _Float16*)Q,
                     (const _Float16*)K, (const _Float16*)V, (_Float16*)O, Sq, Skv, scale * 1.4426950408889634f, nparts, part_keys, part_o,
                     part_ml);
  return check_launch("flash_decode_kernel");
}

// From 128 MB of keys and values upwards, half of what the last-level cache holds, the copies leave no lines behind (ONCE): a program that
// attends to several such caches in turn, a layer each, finds nothing of the next one there, and lines that displace others cost time.  us,
// plain copies and these: 16 x 16 heads, 4096 keys of 128, 537 MB 90.9, 77.1; 10 x 8 heads, 3116 keys, just below the line, three and more in turn
// 26.7, 23.6, alone 22.8, 22.6.  The price is a single cache of up to the size of the last-level one that is read again and again, and two of half of it (3 x 12
// heads, 13619 keys, 251 MB alone 40.4, 41.2 to 43.3, two in turn 48.0, 42.2, six 48.1, 43.5; 20 x 32, 1560 of 64, 256 MB 40.8, 43.6 and 49.3, 44.6; 5 x 12,
// 9000 of 96, 207 MB 33.6, 34.8 and 40.5, 35.9; 6 x 12, 5000 of 96, 138 MB 23.9, 24.2 and 24.8, 25.3, six 28.4, 26.1); smaller ones would pay it as soon as a
// few fit together (6 x 32 heads, 1267 keys of 96, 93 MB, two in turn 15.7, 17.0, six 19.0, 17.6).  (Only V's copies without lines from 128
// to 256 MB: 40.4, 40.7, 44.3 for the 251 MB, 42.7, 42.6, 46.4 for the 256, 34.1, 34.0, 36.4 for 223 in place of 33.4, 34.5, 35.5: no better over all.)
constexpr long long kDecOnceBytes = 128LL << 20;

// nparts workgroups per head, each leaving its part in part_o / part_ml when nparts > 1 (see attn_merge_kernel).
int launch_decode(const void* Q, const void* K, const void* V, void* O, int BH, int Sq, int Skv, int D, float scale, int nparts,
                  int part_keys, float* part_o, float* part_ml, hipStream_t s) {
  const bool once = 4LL * BH * Skv * D >= kDecOnceBytes;
  auto with = [&](auto d_c) {
    constexpr int d = decltype(d_c)::value;
    return once ? launch<d, true>(Q, K, V, O, BH, Sq, Skv, scale, nparts, part_keys, part_o, part_ml, s)
                : launch<d, false>(Q, K, V, O, BH, Sq, Skv, scale, nparts, part_keys, part_o, part_ml, s);
  };
  switch (D) {
    case 32: return with(std::integral_constant<int, 32>{});
    case 64: return with(std::integral_constant<int, 64>{});
    case 96: return with(std::integral_constant<int, 96>{});
    default: return with(std::integral_constant<int, 128>{});
  }
}

}  // namespace ftk
