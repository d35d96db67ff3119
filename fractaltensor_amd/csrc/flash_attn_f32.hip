// Non-causal flash attention with fp32 Q, K, V and O on the fp16 matrix pipe of gfx950: every product of two
// fp32 numbers is formed as three fp16 products of split operands, accumulated in fp32.
//
// The reference's attention program computes in fp32 (examples/flash_attention/flash_attention.py:14-91 with
// kaleido.float32 blocks, flash_attention_utils.py:20-24).  fp32 MFMAs move two k per 16 passes where fp16
// MFMAs move sixteen per 8, so, as in the stacked LSTM, an fp32 product is cheaper as three fp16 ones:
//   v * 2^e = top + rest,  top = fp16(v * 2^e),  rest = fp16(v * 2^e - top),
// and top * top, top * rest and rest * top go into one fp32 accumulator; rest * rest, 2^-22 of a product, is
// dropped.  What shares a power-of-two scale 2^e (its largest magnitude lands in [2^14, 2^15)): a row of Q, all
// of K of one (batch, head), all of V of one (batch, head) (DIRECT: a tile of K, V up to the tile), and the fixed
// 2^7 for the softmax weights p in [0, 2^8).  The two planes hold an element to within 2^-40 of its group's largest magnitude (2^-29 where the
// matrix unit flushes an fp16 subnormal: the remainder of an element below 2^-17 of the largest is one), which is
// what a sum of products is accurate to anyway: 22 significant bits of its own are kept by every element within
// 2^-17 of the largest.
//
// Launches, where the attention kernel does not cut K and V itself (DIRECT): the largest |K| and |V| per (batch, head)
// and the split of K and V into planes [row][top D | rest D] in the workspace, in one launch where heads are small, else in two; the attention kernel, which splits its rows of Q (times scale * log2 e)
// itself, in registers.  A plane row is an fp16 row of 2 D
// elements, so tiles, copies and fragment reads are those of the fp16 kernel at twice the head dimension
// (fa_common.h), and the contractions are its transposed ones: S^T = K Q^T, O^T += V^T P^T, a lane owns one query
// row, the running maximum and sum are lane-local.  The reference that the weights are taken against follows the
// running maximum lazily: it moves only when a score exceeds it by more than 8 bits (kLazyBits), so weights reach
// 2^8 at most and O's accumulators (accumulation registers, which vector instructions reach only through moves)
// are rescaled once per row block on ordinary data rather than whenever one of a wave's 32 rows finds a new
// maximum (every other half tile).
#include <algorithm>
#include <type_traits>

#include "fa_common.h"

namespace ftk {

typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kF32Top = 14;             // a scale group's largest magnitude lands in [2^14, 2^15)
constexpr float kF32PBits = 7.0f;        // 2^7: the scale of the softmax weights in their fp16 planes
constexpr float kLazyBits = 7.99f;      // how far a score may exceed the softmax reference: weights below 2^8, below 65504 in their plane
// s_waitcnt immediate: at most n vector memory operations outstanding (n < 64), the other counters left alone
constexpr int vmcnt_at_most(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// the power of two that brings a largest magnitude with these float bits into [2^14, 2^15), and its inverse
__device__ __forceinline__ void split_scale(unsigned max_bits, float* scale, float* inv) {
  const int eb = min(max((int)((max_bits >> 23) & 0xff), 15), 254 - kF32Top);
  *scale = __uint_as_float((unsigned)(127 + kF32Top + 127 - eb) << 23);
  *inv = __uint_as_float((unsigned)(eb - kF32Top) << 23);
}

// What undoes the scales of a row of Q and of K in a score.  Above zero also where both scales stand at their bound, as those of a row of zeros and
// of keys of zeros do (a sample shorter than its batch): a masked key's score of -inf times zero would be a NaN.  A raw score is below 2^38, so what
// is raised here was below 2^-88 and stays there.
__device__ __forceinline__ float undo_scales(float q_undo, float k_undo) { return fmaxf(q_undo * k_undo, 0x1p-126f); }

__device__ __forceinline__ int clamped_eb(int eb) { return min(max(eb, 15), 254 - kF32Top); }   // the exponent field that split_scale goes by

// The two launches of larger heads: largest |x| of every chunk of every (batch, head) of K and V, as float bits (which order like
// the magnitudes), grid (chunks, BH, 2), per_bh a multiple of 4; then the planes, whose workgroups take the largest of a head's chunks.
// (With one word a head, cleared by a launch and raised by atomics, the three took 24 us at 16 heads of 1280 keys of 128.)
constexpr int kMaxChunks = 64;
__global__ __launch_bounds__(256) void attn_f32_absmax_kernel(const float* K, const float* V, unsigned* chunk_bits, size_t per_bh, int BH) {
  __shared__ unsigned wave_max[4];
  const float* x = (blockIdx.z ? V : K) + (size_t)blockIdx.y * per_bh;
  unsigned m = 0;
#pragma unroll 4
  for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < per_bh; i += (size_t)gridDim.x * 1024) {
    const float4 v = *reinterpret_cast<const float4*>(x + i);
    m = max(max(m, __float_as_uint(fabsf(v.x))), max(__float_as_uint(fabsf(v.y)), max(__float_as_uint(fabsf(v.z)), __float_as_uint(fabsf(v.w)))));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    chunk_bits[((size_t)blockIdx.z * BH + blockIdx.y) * gridDim.x + blockIdx.x] = max(max(wave_max[0], wave_max[1]), max(wave_max[2], wave_max[3]));
}

// One word a head from the words of its chunks, a wave to each: where the workspace has no room for these beside the planes they
// stand in the planes of V, which the launch behind this one writes.  A few microseconds; with a workgroup or a few to a head for
// the whole preparation, as small heads have, the call took 3329 us in place of 2252 at 2 heads of 64 k keys of 128, 4079 in place of 2345 at 4.
__global__ __launch_bounds__(64) void attn_f32_largest_kernel(const unsigned* chunk_bits, int chunks, unsigned* bits) {
  unsigned m = (int)threadIdx.x < chunks ? chunk_bits[(size_t)blockIdx.x * chunks + threadIdx.x] : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if (threadIdx.x == 0) bits[blockIdx.x] = m;
}

// Eight neighbouring floats of a row into its planes [top D | rest D].
template <int D>
__device__ __forceinline__ void split_eight(const float* X, _Float16* planes, long long chunk, float scale) {
  constexpr int CPR = D / 8;
  const long long row = chunk / CPR;
  const int c = (int)(chunk - row * CPR);
  const float4 a = *reinterpret_cast<const float4*>(X + row * D + 8 * c), b = *reinterpret_cast<const float4*>(X + row * D + 8 * c + 4);
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  v8h top, rest;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = v[e] * scale;
    top[e] = (_Float16)s;
    rest[e] = (_Float16)(s - (float)top[e]);
  }
  _Float16* const dst = planes + row * (2 * D) + 8 * c;
  *reinterpret_cast<v8h*>(dst) = top;
  *reinterpret_cast<v8h*>(dst + D) = rest;
}

// Planes under each head's scale, grid (workgroups of a head, BH, 2: K, V), eight floats to a thread; clears the counters.  chunk_bits: the
// words of each head's chunks, or bits itself, with one word a head (which then gets the value it has).
template <int D>
__global__ __launch_bounds__(256) void attn_f32_split_kernel(const float* K, const float* V, _Float16* kplanes, _Float16* vplanes, unsigned* bits,
                                                            const unsigned* chunk_bits, int chunks, int Skv, int BH, int counters) {
  const bool is_v = blockIdx.z != 0;
  const int group = is_v * BH + blockIdx.y, lane = threadIdx.x & 63;
  unsigned m = lane < chunks ? chunk_bits[(size_t)group * chunks + lane] : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) bits[group] = m;
    if (group == 0)
      for (int i = threadIdx.x; i < counters; i += 256) bits[2 * BH + i] = 0;
  }
  float scale, inv;
  split_scale(m, &scale, &inv);
  const size_t head = (size_t)blockIdx.y * Skv * D;
  const float* const X = (is_v ? V : K) + head;
  _Float16* const planes = (is_v ? vplanes : kplanes) + 2 * head;
  const int all = Skv * (D / 8);
  for (int i = blockIdx.x * 256 + threadIdx.x; i < all; i += gridDim.x * 256) split_eight<D>(X, planes, i, scale);
}

// Largest magnitude and planes in one launch, for heads that a compute unit reads in a microsecond or two: each of a
// head's `parts` workgroups finds the head's largest magnitude for itself (the others find the rows in their XCD's L2) and
// writes its share of the planes.  (Three launches, with a clear in front, took 11 us whatever the size: B 2, 8 heads, 1024
// keys of 32.)
constexpr int kPlanesThreads = 512;
template <int D>
__global__ __launch_bounds__(kPlanesThreads) void attn_f32_planes_kernel(const float* K, const float* V, _Float16* kplanes, _Float16* vplanes,
                                                                         unsigned* bits, int Skv, int BH, int parts, int counters) {
  __shared__ unsigned wave_max[kPlanesThreads / 64];
  if (blockIdx.x == 0)   // the counters behind the magnitudes
    for (int i = threadIdx.x; i < counters; i += kPlanesThreads) bits[2 * BH + i] = 0;
  const int id = xcd_consecutive(blockIdx.x, gridDim.x);
  const int group = id / parts, part = id - group * parts;   // group: (batch, head) of K, then of V
  const bool is_v = group >= BH;
  const size_t head = (size_t)(is_v ? group - BH : group) * Skv * D;
  const float* const X = (is_v ? V : K) + head;
  _Float16* const planes = (is_v ? vplanes : kplanes) + 2 * head;
  const int quads = Skv * (D / 4);
  unsigned m = 0;
#pragma unroll 8
  for (int i = threadIdx.x; i < quads; i += kPlanesThreads) {
    const float4 v = *reinterpret_cast<const float4*>(X + 4 * (size_t)i);
    m = max(max(m, __float_as_uint(fabsf(v.x))), max(__float_as_uint(fabsf(v.y)), max(__float_as_uint(fabsf(v.z)), __float_as_uint(fabsf(v.w)))));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPlanesThreads / 64; ++w) m = max(m, wave_max[w]);
  if (part == 0 && threadIdx.x == 0) bits[group] = m;
  float scale, inv;
  split_scale(m, &scale, &inv);
  const int chunks = Skv * (D / 8);
  for (int i = part * kPlanesThreads + threadIdx.x; i < chunks; i += parts * kPlanesThreads) split_eight<D>(X, planes, i, scale);
}

// Bytes a part of a block of 128 query rows leaves in the workspace.
constexpr int f32_partial_bytes(int D) { return 128 * D * 4 + 4 * 64 * 8; }

// DIRECT: Kp and Vp are K and V themselves, no launch in front.  Each workgroup cuts a tile's fp32 rows into their planes on the way to LDS
// (they are as long as the planes), K under a scale of the tile's own, V under that of the largest value of the group's tiles so
// far: no magnitude of a whole head is needed first, and no element has fewer bits than under its head's scale.  Every query block pays for
// it again: f32_split has the line.  The error against float64 is that of the other form, also with keys that differ by 2^20.  At D 128 it takes
// all 512 registers and two spilled ones (12 bytes of scratch a lane); on the grids that f32_split gives it, it is the faster form as it is.
// 4 waves x 32 query rows per workgroup.  Two workgroups to a compute unit at head sizes up to 64 (B 4, 16 heads, 1024 keys of 64: 88
// -> 77 us with a bound of 256 registers, of which the compiler had taken a few more), one above: the accumulators of O,
// both planes of Q and the scores take some 400 registers at D = 128.  K and V tiles of 64 keys, both double buffered.  A wave
// works through the tiles in halves of 32 keys, and with one wave per SIMD the softmax of a half has no other
// wave's MFMAs to run beside: it is cut in two, the maxima under the P V MFMAs of the half before and the weights
// under the score MFMAs of the half after (the comments in the kernel give the order).
// KG > 1 (two groups at head sizes up to 64, whose registers allow two waves per SIMD; four at 32): the groups share the query rows,
// each walks its part of the keys with tiles of its own in LDS, and the first takes in the others' results at the end.
// PART: nparts workgroups share a block of query rows, each with its share of the tiles.  Each leaves its unnormalised
// accumulators, reference and sum in the workspace (write-through: a block's workgroups may sit on several XCDs), and the one
// that finds itself the last by the block's counter takes all of them in, in the order of their keys, so that the result does
// not depend on who was last, and stores the block.
// LDS layout of the tiles of four key groups at head size 32 (padded, they take 172 KB): V rows without padding, the planes of
// every second pair of rows exchanged, so that four rows of a plane fall on different banks.
struct FaFourGroups : FaLayout<64> {
  static constexpr int VRS = 128, VTB = FA_KT * VRS;
};
template <int D, int KG> using F32Tiles = typename std::conditional<KG == 4, FaFourGroups, FaLayout<2 * D>>::type;

template <int D, int KG, int WAVES, bool PART, bool DIRECT>
__global__ __launch_bounds__(KG * WAVES * 64, KG == 1 && D <= 64 ? 2 : 1) void flash_attn_f32_kernel(const float* __restrict__ Q,
                                                                const void* __restrict__ Kp,
                                                                const void* __restrict__ Vp, float q_mul,
                                                                const unsigned* __restrict__ kv_bits, float* __restrict__ O,
                                                                int Sq, int Skv_whole, int nqb, int BH, int nparts,
                                                                int* __restrict__ counters, unsigned char* __restrict__ partials) {
  using L = F32Tiles<D, KG>;          // a plane row is an fp16 row of 2 D elements
  constexpr bool SWZ = KG == 4;
  static_assert(!SWZ || D == 32, "four key groups at head size 32");
  constexpr int DS = D / 16;          // k steps of S^T
  constexpr int DT = D / 32;          // d tiles of O^T
  constexpr int RB = 4 * D;           // bytes per plane row in global memory
  constexpr int KRS = L::KRS, VRS = L::VRS, KTB = L::KTB, VTB = L::VTB;
  constexpr int KCP = (KTB / 1024 + WAVES - 1) / WAVES, VCP = (VTB / 1024 + WAVES - 1) / WAVES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) % WAVES);   // within its key group
  const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((tid >> 6) / WAVES);
  constexpr int GROUP_LDS = 2 * (KTB + VTB);
  unsigned char* const Kb = smem + group * GROUP_LDS;   // [2][KTB]
  unsigned char* const Vb = Kb + 2 * KTB;               // [2][VTB]
  const int j = lane & 31;
  const int hh = lane >> 5;
  const int id = xcd_consecutive(blockIdx.x, gridDim.x);   // a head's query blocks share an XCD
  const int block = PART ? id / nparts : id, part = PART ? id - block * nparts : 0;
  const int bh = block / nqb;
  const int qb = block - bh * nqb;
  const int q_base = qb * (WAVES * 32) + wave * 32;

  // the workgroup's tiles of keys: the first `long_parts` parts have one more than the others
  const int all_tiles = (Skv_whole + FA_KT - 1) / FA_KT, each = PART ? all_tiles / nparts : all_tiles, long_parts = PART ? all_tiles - each * nparts : 0;
  const int tile_first = part * each + min(part, long_parts);
  const int key_part = tile_first * FA_KT;
  const int Skv_all = PART && part + 1 < nparts ? (each + (part < long_parts ? 1 : 0)) * FA_KT : Skv_whole - key_part;   // its keys
  // the groups have neighbouring shares of the tiles, the first ones one more where they do not divide (never fewer than one each)
  const int part_tiles = (Skv_all + FA_KT - 1) / FA_KT, share = part_tiles / KG, long_groups = part_tiles - share * KG;
  const int most_tiles = share + (long_groups > 0 ? 1 : 0);
  const int key_first = (group * share + min(group, long_groups)) * FA_KT;
  const int Skv = KG == 1 ? Skv_all : group + 1 < KG ? (share + (group < long_groups ? 1 : 0)) * FA_KT : Skv_all - key_first;   // the keys this group sees
  // (a row of fp32 and its two planes are as long)
  const _Float16* Kg = static_cast<const _Float16*>(Kp) + ((size_t)bh * Skv_whole + key_part + key_first) * (2 * D);
  const _Float16* Vg = static_cast<const _Float16*>(Vp) + ((size_t)bh * Skv_whole + key_part + key_first) * (2 * D);
  float* Og = O + (size_t)bh * Sq * D;

  // DIRECT: a tile's fp32 rows through registers, eight neighbouring floats of FN rows of K and of V to a lane.  Asked for a tile
  // ahead; its largest magnitudes meet in LDS at the barrier in the middle of the tile before, behind which every wave cuts its
  // rows into their planes in LDS.
  constexpr int CPR8 = D / 8, FN = DIRECT ? D / (8 * WAVES) : 1;
  __shared__ unsigned tile_max[DIRECT ? KG : 1][DIRECT ? WAVES : 1][2];
  float4 fk[FN][2], fv[FN][2];
  auto fetched = [&](auto i_c, int* row, int* c) __attribute__((always_inline)) {
    const int x = 64 * (wave + WAVES * decltype(i_c)::value) + lane;
    *row = x / CPR8;
    *c = x - *row * CPR8;
  };
  [[maybe_unused]] auto fetch = [&](int kt) __attribute__((always_inline)) {
    const int last = Skv - 1 - kt * FA_KT;   // rows past the end re-read the last key; their scores are masked
    const float* const kb = reinterpret_cast<const float*>(Kg) + (size_t)kt * FA_KT * D;
    const float* const vb = reinterpret_cast<const float*>(Vg) + (size_t)kt * FA_KT * D;
    static_for<FN>([&](auto i_c) __attribute__((always_inline)) {
      constexpr int i = decltype(i_c)::value;
      int row, c;
      fetched(i_c, &row, &c);
      const unsigned at = (unsigned)(min(row, last) * D + 8 * c);
      fk[i][0] = *reinterpret_cast<const float4*>(kb + at);
      fk[i][1] = *reinterpret_cast<const float4*>(kb + at + 4);
      fv[i][0] = *reinterpret_cast<const float4*>(vb + at);
      fv[i][1] = *reinterpret_cast<const float4*>(vb + at + 4);
    });
  };
  // the wave's largest magnitudes of the rows it fetched
  [[maybe_unused]] auto publish_max = [&]() __attribute__((always_inline)) {
    auto wave_max = [&](const float4 (&f)[FN][2]) __attribute__((always_inline)) -> unsigned {
      float m = 0.0f;
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(f[i][h].x), "v"(f[i][h].y));
          asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(f[i][h].z), "v"(f[i][h].w));
        }
      // within rows of 16 lanes, then over the four rows
      unsigned b = __float_as_uint(m);
      b = max(b, (unsigned)__builtin_amdgcn_mov_dpp((int)b, 0x128, 0xf, 0xf, true));
      b = max(b, (unsigned)__builtin_amdgcn_mov_dpp((int)b, 0x124, 0xf, 0xf, true));
      b = max(b, (unsigned)__builtin_amdgcn_mov_dpp((int)b, 0x122, 0xf, 0xf, true));
      b = max(b, (unsigned)__builtin_amdgcn_mov_dpp((int)b, 0x121, 0xf, 0xf, true));
      return max(max((unsigned)__builtin_amdgcn_readlane((int)b, 0), (unsigned)__builtin_amdgcn_readlane((int)b, 16)),
                 max((unsigned)__builtin_amdgcn_readlane((int)b, 32), (unsigned)__builtin_amdgcn_readlane((int)b, 48)));
    };
    const unsigned mk = wave_max(fk), mv = wave_max(fv);
    if (lane == 0) {
      tile_max[group][wave][0] = mk;
      tile_max[group][wave][1] = mv;
    }
  };
  // Planes into buffer buf: K under the tile's own scale (k_undo: what undoes it), V under that of the largest magnitude of the
  // group's tiles so far (v_eb: its exponent field), which O follows when it comes to the tile.
  [[maybe_unused]] float k_undo = 0.0f;
  [[maybe_unused]] int v_eb = 0;
  [[maybe_unused]] auto put_planes = [&](int buf) __attribute__((always_inline)) {
    unsigned mk = 0, mv = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      mk = max(mk, tile_max[group][w][0]);
      mv = max(mv, tile_max[group][w][1]);
    }
    mk = (unsigned)__builtin_amdgcn_readfirstlane((int)mk);
    mv = (unsigned)__builtin_amdgcn_readfirstlane((int)mv);
    v_eb = max(v_eb, (int)(mv >> 23));
    float k_scale, v_scale_now, unused;
    split_scale(mk, &k_scale, &k_undo);
    split_scale((unsigned)v_eb << 23, &v_scale_now, &unused);
    auto put = [&](const float4 (&f)[2], float scale, unsigned char* top_at, unsigned char* rest_at) __attribute__((always_inline)) {
      const float v[8] = {f[0].x, f[0].y, f[0].z, f[0].w, f[1].x, f[1].y, f[1].z, f[1].w};
      v4u top, rest;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const v2f x = {v[2 * e] * scale, v[2 * e + 1] * scale};
        const unsigned tu = __builtin_bit_cast(unsigned, __builtin_convertvector(x, v2h));
        unsigned ru;
        asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]\n\tv_fma_mixhi_f16 %0, %1, -1.0, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=&v"(ru) : "v"(tu), "v"(x[0]), "v"(x[1]));
        top[e] = tu;
        rest[e] = ru;
      }
      *reinterpret_cast<v4u*>(top_at) = top;
      *reinterpret_cast<v4u*>(rest_at) = rest;
    };
    static_for<FN>([&](auto i_c) __attribute__((always_inline)) {
      constexpr int i = decltype(i_c)::value;
      int row, c;
      fetched(i_c, &row, &c);
      unsigned char* const k_at = Kb + buf * KTB + row * KRS + 16 * c;
      put(fk[i], k_scale, k_at, k_at + 2 * D);
      unsigned char* const v_at = Vb + buf * VTB + row * VRS + 16 * c;
      const int swapped = SWZ ? 64 * ((row >> 1) & 1) : 0;   // (SWZ: planes of 64 bytes)
      put(fv[i], v_scale_now, v_at + swapped, v_at + (SWZ ? 64 - swapped : 2 * D));
    });
  };
  if constexpr (DIRECT) fetch(0);

  // The lane's query row: the fp32 row is read, multiplied by q_mul (scale * log2 e: a score leaves the matrix unit in
  // exponent units), brought under the row's own power-of-two scale and split into the two planes here, in registers
  // (a lane and its partner 32 lanes on hold the row's two halves of every 16 columns).
  const int qrow = min(q_base + j, Sq - 1);
  v8h qt[DS], qr[DS];
  float s_mul;                     // what a score is multiplied by to undo the scales
  [[maybe_unused]] float q_undo;   // the query row's part of it
  {
    const float* qsrc = Q + ((size_t)bh * Sq + qrow) * D + 8 * hh;
    float4 x[DS][2];
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      x[s][0] = *reinterpret_cast<const float4*>(qsrc + 16 * s);
      x[s][1] = *reinterpret_cast<const float4*>(qsrc + 16 * s + 4);
    }
    unsigned m = 0;
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        x[s][h].x *= q_mul; x[s][h].y *= q_mul; x[s][h].z *= q_mul; x[s][h].w *= q_mul;
        m = max(max(m, __float_as_uint(fabsf(x[s][h].x))), max(__float_as_uint(fabsf(x[s][h].y)),
                                                               max(__float_as_uint(fabsf(x[s][h].z)), __float_as_uint(fabsf(x[s][h].w)))));
      }
    m = max(m, (unsigned)__shfl_xor((int)m, 32));   // the row's largest magnitude, as float bits
    float q_scale, q_inv;
    split_scale(m, &q_scale, &q_inv);
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float v[4] = {x[s][h].x * q_scale, x[s][h].y * q_scale, x[s][h].z * q_scale, x[s][h].w * q_scale};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const _Float16 top = (_Float16)v[e];
          qt[s][4 * h + e] = top;
          qr[s][4 * h + e] = (_Float16)(v[e] - (float)top);
        }
      }
    q_undo = q_inv;
    s_mul = 1.0f;
    if constexpr (!DIRECT) {
      float k_scale, k_inv;
      split_scale(kv_bits[bh], &k_scale, &k_inv);
      s_mul = undo_scales(q_inv, k_inv);
    }
  }
  [[maybe_unused]] float v_scale, v_inv;
  if constexpr (!DIRECT) split_scale(kv_bits[BH + bh], &v_scale, &v_inv);

  v16f om[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) om[dt][r] = 0.0f;

  // copies: as in the fp16 kernel, copy c of a tile fills LDS bytes [1024 c, 1024 c + 1024) of the padded tile
  unsigned k_src[KCP], v_src[VCP];
#pragma unroll
  for (int i = 0; i < KCP; ++i) {
    const int x = 1024 * (wave + WAVES * i) + 16 * lane;
    const int row = min(x / KRS, FA_KT - 1), col = x % KRS;
    k_src[i] = row * RB + (col < RB ? col : 0);
  }
#pragma unroll
  for (int i = 0; i < VCP; ++i) {
    const int x = 1024 * (wave + WAVES * i) + 16 * lane;
    const int row = min(x / VRS, FA_KT - 1), col = x % VRS;
    if constexpr (SWZ) v_src[i] = row * RB + (col ^ (64 * ((row >> 1) & 1)));
    else v_src[i] = row * RB + (col < RB ? col : 0);
  }
  // (a whole tile takes the copies' offsets as they are; the last tile of a ragged row of keys clamps each)
  auto copy_rows = [&](auto n_c, auto bytes_c, const unsigned (&src)[decltype(n_c)::value], const _Float16* rows, int key0,
                       unsigned char* dst) __attribute__((always_inline)) {
    constexpr int N = decltype(n_c)::value, COPIES = decltype(bytes_c)::value / 1024;
    if (key0 + FA_KT <= Skv) {
      static_for<N>([&](auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if (WAVES * i + WAVES - 1 < COPIES || wave + WAVES * i < COPIES) lds_dma16(rows, src[i], dst + 1024 * (wave + WAVES * i));
      });
    } else {
      static_for<N>([&](auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if (wave + WAVES * i < COPIES) {
          unsigned off = src[i];
          const unsigned last = (unsigned)(Skv - 1 - key0), row = off / RB;   // rows past the end re-read the last key; their scores are masked
          if (row > last) off -= (row - last) * RB;
          lds_dma16(rows, off, dst + 1024 * (wave + WAVES * i));
        }
      });
    }
  };
  auto copy_k = [&](int kt, int buf) __attribute__((always_inline)) {
    copy_rows(std::integral_constant<int, KCP>{}, std::integral_constant<int, KTB>{}, k_src, Kg + (size_t)kt * FA_KT * (2 * D), kt * FA_KT,
              Kb + buf * KTB);
  };
  auto copy_v = [&](int kt, int buf) __attribute__((always_inline)) {
    copy_rows(std::integral_constant<int, VCP>{}, std::integral_constant<int, VTB>{}, v_src, Vg + (size_t)kt * FA_KT * (2 * D), kt * FA_KT,
              Vb + buf * VTB);
  };
  // every wave issues at least this many copies of a K tile, of a V tile (wave 0 may issue one more)
  constexpr int KC_MIN = KTB / 1024 / WAVES, VC_MIN = VTB / 1024 / WAVES;

  const int k_lane = j * KRS + 16 * hh;
  const int v_lane = (4 * hh + ((lane & 15) >> 2)) * VRS + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
  [[maybe_unused]] const int v_first = SWZ ? 64 * (((lane & 15) >> 3) & 1) : 0;   // where the rows this lane names (4 hh + its quarter) have their values
  using lds_v4s = __attribute__((address_space(3))) v4s;
  typedef short v8s __attribute__((ext_vector_type(8)));
  // A-operand of the P V product: step s (16 keys) and d tile dt of one half tile; plane 0 = values, 1 = remainders
  auto read_v = [&](const unsigned char* vbase, int s, int dt, int plane) __attribute__((always_inline)) {
    const unsigned char* p0 = vbase + 16 * s * VRS + 64 * dt;
    if constexpr (SWZ) p0 += plane ? 64 - v_first : v_first;
    else p0 += plane * (2 * D);
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p0));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p0 + 8 * VRS));
    const v8s both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(v8h, both);
  };

  const v16f zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // One wave per SIMD has only its own vector instructions to put beside its MFMAs, so the softmax of a half is cut in
  // two and each part runs under the MFMAs of another product:
  //   the scores of half h                  beside  the weights of half h - 1 (exp2, the split into planes)
  //   the P V product of half h - 1         beside  the raw scores and the maximum of half h
  // and then the reference moves if it has to (rarely, see kLazyBits) and O is rescaled.
  //
  // State between the two: raw[], the scores of the half before in the matrix unit's units (times s_mul: exponent
  // units), and m_ref, the reference they are taken against; pt / pr, the weights whose product is still to come.
  float raw[16];
  float m_ref = -INFINITY, l_run = 0.0f;   // l_run: the sum of the weights, in their planes' scale
  v8h pt[2], pr[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) { pt[s][e] = (_Float16)0.0f; pr[s][e] = (_Float16)0.0f; }
#pragma unroll
  for (int r = 0; r < 16; ++r) raw[r] = -INFINITY;   // in front of the first half: weights of zero

  // weights of pair k (two neighbouring scores) of the half before: p * 2^7 = exp2(raw * s_mul - m_ref + kF32PBits), its two planes
  float lsum = 0.0f;
  unsigned ptu[8], pru[8];
  auto weight_pair = [&](auto k_c, float bias) __attribute__((always_inline)) {
    constexpr int k = decltype(k_c)::value;
    const float s0 = __builtin_amdgcn_exp2f(fmaf(raw[2 * k], s_mul, bias)), s1 = __builtin_amdgcn_exp2f(fmaf(raw[2 * k + 1], s_mul, bias));
    lsum += s0 + s1;
    const v2f sv = {s0, s1};
    const v2h top = __builtin_convertvector(sv, v2h);
    unsigned tu = __builtin_bit_cast(unsigned, top), ru;
    // the remainders, s - top rounded to fp16: one mixed-precision fma each (the fp16 value read as fp32 times -1, plus
    // s; the difference is exact in fp32) instead of a conversion back, a subtraction and a conversion
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]\n\tv_fma_mixhi_f16 %0, %1, -1.0, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=&v"(ru) : "v"(tu), "v"(s0), "v"(s1));
    // pinned to its place: left alone, the compiler moves the arithmetic to where the weights are read, out from under the MFMAs
    asm volatile("" : "+v"(tu), "+v"(ru), "+v"(lsum));
    ptu[k] = tu;
    pru[k] = ru;
  };
  // the weights of key step h of the half (pairs 4 h .. 4 h + 3) as the P V product's fragments
  auto weights_done = [&](int h) __attribute__((always_inline)) {
    pt[h] = __builtin_bit_cast(v8h, v4u{ptu[4 * h], ptu[4 * h + 1], ptu[4 * h + 2], ptu[4 * h + 3]});
    pr[h] = __builtin_bit_cast(v8h, v4u{pru[4 * h], pru[4 * h + 1], pru[4 * h + 2], pru[4 * h + 3]});
  };
  // With an even number of d tiles the P V product uses the weights of the first key step (pairs 0..3) alone for its
  // first half: only those are formed beside the scores, pairs 4..7 beside the first half of the product itself, and
  // the maxima of the next scores beside its second half -- a wave that is alone on its SIMD hides some four vector
  // instructions per MFMA, so the vector work is dealt out as evenly as the order allows.
  constexpr bool kDefer = DT % 2 == 0;
  constexpr int kPairsBesideScores = kDefer ? 4 : 8;
  float bias = 0.0f;   // what a raw score times s_mul is offset by in the weights' exponent (set where a half's weights begin)

  // Fragments live across the two products: each requests the other's first ones before it ends, so that no product
  // begins by waiting for LDS (a read takes some hundreds of cycles under this load).
  v8h kf_t[4], kf_r[4];   // K fragments (values, remainders) of a k step, four sets in turn
  v8h vf_t[4], vf_r[4];   // V fragments of a (key step, d tile) group, two pairs of groups in turn
  auto read_k = [&](const unsigned char* kbase, int s, int set) __attribute__((always_inline)) {
    kf_t[set] = *reinterpret_cast<const v8h*>(kbase + 32 * s);
    kf_r[set] = *reinterpret_cast<const v8h*>(kbase + 2 * D + 32 * s);
  };
  auto read_group = [&](const unsigned char* pvbase, int g, int set) __attribute__((always_inline)) {
    vf_t[set] = read_v(pvbase, g / DT, g % DT, 0);
    vf_r[set] = read_v(pvbase, g / DT, g % DT, 1);
  };

  // The scores of 32 keys (one half of a tile): value x value and the two mixed products, all into am.  A step's
  // K fragments are requested three steps ahead; PRELOADED: those of steps 0 and 1 by the product before.
  // Beside the MFMAs: the weights of the half before, a share with every step; the copies of a whole tile that is
  // on its way (COPY 1: K of tile ckt, 2: V of tile ckt; 0: none), a share with every step and no branch among them;
  // and at the end the first V fragments of the product that follows (rows at pvbase).
  auto scores = [&](auto preloaded_c, auto copy_c, int ckt, int cbuf, const unsigned char* kbase, const unsigned char* pvbase,
                    v16f& am) __attribute__((always_inline)) {
    constexpr bool PRELOADED = decltype(preloaded_c)::value;
    constexpr int COPY = decltype(copy_c)::value;
    constexpr int NCOPY = COPY == 1 ? KCP : VCP;
    if constexpr (!PRELOADED) {
      read_k(kbase, 0, 0);
      read_k(kbase, 1, 1);
    }
    if constexpr (DS > 2) read_k(kbase, 2, 2);
    bias = m_ref > -INFINITY ? kF32PBits - m_ref : 0.0f;   // (no reference before the first half: every raw score is -inf)
    lsum = 0.0f;
    const _Float16* crows = (COPY == 1 ? Kg : Vg) + (size_t)ckt * FA_KT * (2 * D);
    unsigned char* cdst = COPY == 1 ? Kb + cbuf * KTB : Vb + cbuf * VTB;
    __builtin_amdgcn_sched_barrier(0);
    static_for<DS>([&](auto s_c) __attribute__((always_inline)) {
      constexpr int s = decltype(s_c)::value, b = s % 4;
      am = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf_t[b], qt[s], s == 0 ? zero16 : am, 0, 0, 0);
      if constexpr (s + 3 < DS) read_k(kbase, s + 3, (s + 3) % 4);
      if constexpr (s >= DS - 2) read_group(pvbase, s - (DS - 2), s - (DS - 2));
      am = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf_t[b], qr[s], am, 0, 0, 0);
      am = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf_r[b], qt[s], am, 0, 0, 0);
      static_for<kPairsBesideScores * (s + 1) / DS - kPairsBesideScores * s / DS>([&](auto j_c) __attribute__((always_inline)) {
        weight_pair(std::integral_constant<int, kPairsBesideScores * s / DS + decltype(j_c)::value>{}, bias);
      });
      // the order within the step: MFMA, the reads, and the vector instructions in three shares behind the three MFMAs
      // (the first share holds the two exp2, four issue slots each)
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, s >= DS - 2 ? 4 : 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (COPY != 0) {
        static_for<NCOPY * (s + 1) / DS - NCOPY * s / DS>([&](auto j_c) __attribute__((always_inline)) {
          constexpr int i = NCOPY * s / DS + decltype(j_c)::value, COPIES = (COPY == 1 ? KTB : VTB) / 1024;
          const unsigned src = COPY == 1 ? k_src[i % KCP] : v_src[i % VCP];
          if (WAVES * i + WAVES - 1 < COPIES || wave + WAVES * i < COPIES) lds_dma16(crows, src, cdst + 1024 * (wave + WAVES * i));
        });
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    weights_done(0);
    if constexpr (!kDefer) {
      weights_done(1);
      l_run += lsum;
    }
  };

  // The P V product of the half whose weights are in pt / pr (V rows at pvbase), and beside it (MAXIMA) the raw
  // scores and the maximum of the half whose products are in am; then the reference moves if a score exceeds it
  // by more than kLazyBits, and O and the sum are brought to the new one.  Groups (key step, d tile: 3 MFMAs) are
  // taken two at a time, in an order in which no MFMA adds to the result of the one before it; a pair's V fragments are
  // requested under the pair before.
  // (DIRECT: the V rows at pvbase are under the scale of exponent field pend_eb, O under that of o_eb)
  [[maybe_unused]] int o_eb = 0, pend_eb = 0;
  auto pv_and_maxima = [&](auto maxima_c, auto next_k_c, auto mask_c, const unsigned char* pvbase, const unsigned char* next_kbase,
                           const v16f& am, int key0) __attribute__((always_inline)) {
    if constexpr (DIRECT) {
      if (pend_eb != o_eb) {
        const float by = ldexpf(1.0f, clamped_eb(o_eb) - clamped_eb(pend_eb));
        o_eb = pend_eb;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) om[dt][r] *= by;
      }
    }
    // MAXIMA false: the product alone, behind the last half, all of whose weights are there; MASK: the half is ragged
    constexpr bool MAXIMA = decltype(maxima_c)::value, NEXT_K = decltype(next_k_c)::value, MASK = decltype(mask_c)::value;
    constexpr bool DEFER = kDefer && MAXIMA;
    constexpr int NG = 2 * DT, NM = 3 * NG;
    constexpr int M0 = DEFER ? NM / 2 : 0, MN = NM - M0;   // the slots that hold the maxima
    // (the first pair's fragments were requested by the scores before; NEXT_K: the last slots request the K fragments
    // of steps 0 and 1 of the scores that follow, rows at next_kbase)
    float mx = -INFINITY;
    [[maybe_unused]] const int lim = Skv - key0 - 4 * hh;   // score r belongs to a key past the end when 8 (r >> 2) + (r & 3) >= lim
    static_for<NM>([&](auto i_c) __attribute__((always_inline)) {
      constexpr int i = decltype(i_c)::value, pair = i / 6, k = i % 6, g0 = 2 * pair, g1 = g0 + 1;
      constexpr int b0 = (pair & 1) * 2, b1 = b0 + 1, nb = ((pair + 1) & 1) * 2;
      constexpr int sk0 = g0 / DT, dt0 = g0 % DT, sk1 = g1 / DT, dt1 = g1 % DT;
      if constexpr ((k == 1 || k == 3) && g0 + 2 < NG) read_group(pvbase, g0 + 2 + (k == 3), nb + (k == 3));   // the next pair's fragments
      if constexpr (NEXT_K && g0 + 2 >= NG && (k == 1 || k == 3)) read_k(next_kbase, k == 3, k == 3);
      if constexpr (k == 0) om[dt0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_t[b0], pt[sk0], om[dt0], 0, 0, 0);
      if constexpr (k == 1) om[dt1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_t[b1], pt[sk1], om[dt1], 0, 0, 0);
      if constexpr (k == 2) om[dt0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_t[b0], pr[sk0], om[dt0], 0, 0, 0);
      if constexpr (k == 3) om[dt1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_t[b1], pr[sk1], om[dt1], 0, 0, 0);
      if constexpr (k == 4) om[dt0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_r[b0], pt[sk0], om[dt0], 0, 0, 0);
      if constexpr (k == 5) om[dt1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf_r[b1], pt[sk1], om[dt1], 0, 0, 0);
      if constexpr (DEFER && i < M0) {   // the weights of the second key step (pairs 4..7), wanted by this product's second half
        static_for<4 * (i + 1) / M0 - 4 * i / M0>([&](auto j_c) __attribute__((always_inline)) {
          weight_pair(std::integral_constant<int, 4 + 4 * i / M0 + decltype(j_c)::value>{}, bias);
        });
        if constexpr (i == M0 - 1) {
          weights_done(1);
          l_run += lsum;
        }
      }
      if constexpr (MAXIMA && i >= M0) {
#pragma unroll
        for (int r = 16 * (i - M0) / MN; r < 16 * (i - M0 + 1) / MN; ++r) {
          raw[r] = am[r];
          if constexpr (MASK) {
            if (8 * (r >> 2) + (r & 3) >= lim) raw[r] = -INFINITY;
          }
          mx = fmaxf(mx, raw[r]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (MAXIMA) {
      if constexpr (DIRECT) s_mul = undo_scales(q_undo, k_undo);   // (from here on `raw` is of the tile that `am` is of)
      mx = max_with_other_half(mx) * s_mul;   // finite: the half holds at least one key; s_mul > 0
      if (__builtin_amdgcn_ballot_w64(mx > m_ref + kLazyBits) != 0) {   // a row of the wave moves its reference
        const bool moves = mx > m_ref + kLazyBits;
        const float m_new = moves ? mx : m_ref;
        const float alpha = moves ? __builtin_amdgcn_exp2f(m_ref - m_new) : 1.0f;   // 0 the first time (m_ref = -inf)
        m_ref = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) om[dt][r] *= alpha;
      }
    }
  };

  // A tile's K rows are last read by the scores of its second half and its V rows one half later, beside the next
  // tile's first maxima: K of tile kt + 1 is requested beside the scores of tile kt's first half, V of tile kt + 1
  // beside those of its second half, behind the barrier in the middle of the tile.  Copies complete in the order of their issue, so each of the two barriers waits for the
  // older of the two requests only.
  const int ntiles = (Skv + FA_KT - 1) / FA_KT;
  if constexpr (DIRECT) {
    publish_max();
    __syncthreads();
    put_planes(0);
    o_eb = pend_eb = v_eb;
  } else {
    copy_k(0, 0);
    copy_v(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  }
  __syncthreads();

  const unsigned char* pend_v = Vb + v_lane;   // the V rows of the half whose product is still to come (first: zero weights on tile 0)
  for (int kt = 0; kt < ntiles; ++kt) {
    const int buf = kt & 1;
    const bool more = kt + 1 < ntiles;
    const bool whole_next = !DIRECT && (kt + 2) * FA_KT <= Skv;   // a tile follows and all of its 64 keys exist
    [[maybe_unused]] const int tile_eb = v_eb;   // the scale of V of tile kt
    if constexpr (DIRECT) {
      if (more) fetch(kt + 1);
    }
    {   // first half; beside its scores, K of tile kt + 1 is requested (K[buf ^ 1] was last read before the barrier that ended tile kt - 1)
      v16f am;
      const unsigned char* kbase = Kb + buf * KTB + k_lane;
      if (whole_next) {
        scores(std::false_type{}, std::integral_constant<int, 1>{}, kt + 1, buf ^ 1, kbase, pend_v, am);
      } else {
        if (!DIRECT && more) copy_k(kt + 1, buf ^ 1);   // the last, ragged tile: each copy clamps its rows
        scores(std::false_type{}, std::integral_constant<int, 0>{}, 0, 0, kbase, pend_v, am);
      }
      if (kt * FA_KT + 32 <= Skv) pv_and_maxima(std::true_type{}, std::true_type{}, std::false_type{}, pend_v, kbase + 32 * KRS, am, kt * FA_KT);
      else pv_and_maxima(std::true_type{}, std::true_type{}, std::true_type{}, pend_v, kbase + 32 * KRS, am, kt * FA_KT);
      pend_v = Vb + buf * VTB + v_lane;
    }
    // V of tile kt has landed in every wave (asked for half a tile ago or more); V[buf ^ 1] has been read for the last time
    if constexpr (DIRECT) {
      if (more) publish_max();
    } else {
      if (more) __builtin_amdgcn_s_waitcnt(vmcnt_at_most(KC_MIN));
      else __builtin_amdgcn_s_waitcnt(0x0F70);
    }
    __syncthreads();
    const float k_undo_now = k_undo;
    if constexpr (DIRECT) {
      pend_eb = tile_eb;   // pend_v is now the tile's
      if (more) put_planes(buf ^ 1);
    }
    const float k_undo_next = k_undo;
    k_undo = k_undo_now;   // of the tile whose second half follows
    if (kt * FA_KT + 32 < Skv) {   // second half (a tile that is followed by another has one); beside its scores, V of tile kt + 1 is requested
      v16f am;
      const unsigned char* kbase = Kb + buf * KTB + k_lane + 32 * KRS;
      if (whole_next) {
        scores(std::true_type{}, std::integral_constant<int, 2>{}, kt + 1, buf ^ 1, kbase, pend_v, am);
      } else {
        if (!DIRECT && more) copy_v(kt + 1, buf ^ 1);
        scores(std::true_type{}, std::integral_constant<int, 0>{}, 0, 0, kbase, pend_v, am);
      }
      if (kt * FA_KT + 64 <= Skv) pv_and_maxima(std::true_type{}, std::false_type{}, std::false_type{}, pend_v, nullptr, am, kt * FA_KT + 32);
      else pv_and_maxima(std::true_type{}, std::false_type{}, std::true_type{}, pend_v, nullptr, am, kt * FA_KT + 32);
      pend_v = Vb + buf * VTB + v_lane + 32 * VRS;
    }
    // K of tile kt + 1 has landed; K[buf] has been read for the last time
    if (!DIRECT && more) __builtin_amdgcn_s_waitcnt(vmcnt_at_most(VC_MIN));
    k_undo = k_undo_next;
    __syncthreads();
  }
  {   // the last half's weights, then its product
    bias = kF32PBits - m_ref;
    lsum = 0.0f;
    static_for<8>([&](auto k_c) __attribute__((always_inline)) { weight_pair(k_c, bias); });
    weights_done(0);
    weights_done(1);
    l_run += lsum;
    read_group(pend_v, 0, 0);
    read_group(pend_v, 1, 1);
    const v16f none = zero16;
    pv_and_maxima(std::false_type{}, std::false_type{}, std::false_type{}, pend_v, nullptr, none, 0);
  }
  if (KG > 1 && ntiles < most_tiles) {   // the last tile of the groups that have one more
    __syncthreads();
    __syncthreads();
  }
  __syncthreads();   // LDS is reused below
  float l = l_run + __shfl_xor(l_run, 32);
  if constexpr (KG > 1) {
    // the other groups leave their accumulators, references and sums in their part of LDS, by lane; the first takes them in by
    // the rule of an online softmax
    auto oo = [&](int g) __attribute__((always_inline)) { return reinterpret_cast<v4f*>(smem + g * GROUP_LDS) + wave * (DT * 4 * 64) + lane; };
    auto oml = [&](int g) __attribute__((always_inline)) {
      return reinterpret_cast<float2*>(smem + g * GROUP_LDS + WAVES * (DT * 4 * 64 * 16)) + wave * 64 + lane;
    };
    static_assert(WAVES * (DT * 4 * 64 * 16 + 64 * 8) <= GROUP_LDS, "a group's result fits its tiles' place");
    if (group > 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) oo(group)[(4 * dt + g) * 64] = v4f{om[dt][4 * g], om[dt][4 * g + 1], om[dt][4 * g + 2], om[dt][4 * g + 3]};
      *oml(group) = make_float2(m_ref, l);
      if (DIRECT && lane == 0) tile_max[group][wave][0] = (unsigned)o_eb;
    }
    __syncthreads();
    if (!PART && group > 0) return;
    if (group == 0) {
#pragma unroll
      for (int other = 1; other < KG; ++other) {
        const float2 ml = *oml(other);
        const float m = fmaxf(m_ref, ml.x);
        float wm = __builtin_amdgcn_exp2f(m_ref - m), wo = __builtin_amdgcn_exp2f(ml.x - m);
        l = wm * l + wo * ml.y;
        m_ref = m;
        if constexpr (DIRECT) {   // the two groups' O under the scale of the larger values
          const int eb = __builtin_amdgcn_readfirstlane((int)tile_max[other][wave][0]), most = max(o_eb, eb);
          wm = ldexpf(wm, clamped_eb(o_eb) - clamped_eb(most));
          wo = ldexpf(wo, clamped_eb(eb) - clamped_eb(most));
          o_eb = most;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const v4f o = oo(other)[(4 * dt + g) * 64];
#pragma unroll
            for (int k = 0; k < 4; ++k) om[dt][4 * g + k] = wm * om[dt][4 * g + k] + wo * o[k];
          }
      }
    }
  }
  if constexpr (PART) {
    static_assert(WAVES == 4, "a partial result is that of 128 query rows");
    __shared__ int arrived;
    constexpr int PB = f32_partial_bytes(D), ML = PB - WAVES * 64 * 8;   // a part's accumulators, then its references and sums
    const auto mine = __builtin_amdgcn_make_buffer_rsrc(partials + (size_t)block * nparts * PB, 0, (unsigned)(nparts * PB), 0x00020000);
    constexpr int kAgent = 16;   // sc1
    const unsigned o_at = (unsigned)(wave * (DT * 4 * 64) + lane) * 16, ml_at = (unsigned)(ML + (wave * 64 + lane) * 8);
    if (group == 0) {
#pragma unroll
      for (int i = 0; i < 4 * DT; ++i) {
        const v4f o = {om[i / 4][4 * (i % 4)], om[i / 4][4 * (i % 4) + 1], om[i / 4][4 * (i % 4) + 2], om[i / 4][4 * (i % 4) + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, o), mine, o_at, part * PB + i * 1024, kAgent);
      }
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, make_float2(m_ref, l)), mine, ml_at, part * PB, kAgent);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    if (tid == 0) arrived = __hip_atomic_fetch_add(counters + block, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != nparts - 1 || group > 0) return;
    auto sum_of = [&](int p) __attribute__((always_inline)) {
      return __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(mine, ml_at, p * PB, kAgent));
    };
    auto piece = [&](int p, int i) __attribute__((always_inline)) {
      return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(mine, o_at, p * PB + i * 1024, kAgent));
    };
    // several parts' loads on their way at once: one after the other they take a microsecond each
    constexpr int AT_ONCE = D == 32 ? 8 : D == 64 ? 4 : 2;
    for (int p0 = 0; p0 < nparts; p0 += AT_ONCE) {
      v2f ml[AT_ONCE];
      v4f o[AT_ONCE][4 * DT];
#pragma unroll
      for (int a = 0; a < AT_ONCE; ++a) {
        const int p = min(p0 + a, nparts - 1);
        ml[a] = sum_of(p);
#pragma unroll
        for (int i = 0; i < 4 * DT; ++i) o[a][i] = piece(p, i);
      }
#pragma unroll
      for (int a = 0; a < AT_ONCE; ++a) {
        if (p0 + a >= nparts) break;
        const bool first = p0 + a == 0;   // (the state so far is this part's own, and in the sum already)
        const float m = first ? ml[a][0] : fmaxf(m_ref, ml[a][0]);
        const float wm = first ? 0.0f : __builtin_amdgcn_exp2f(m_ref - m), wo = first ? 1.0f : __builtin_amdgcn_exp2f(ml[a][0] - m);
        l = first ? ml[a][1] : wm * l + wo * ml[a][1];
        m_ref = m;
#pragma unroll
        for (int i = 0; i < 4 * DT; ++i)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float so_far = om[i / 4][4 * (i % 4) + k];
            om[i / 4][4 * (i % 4) + k] = first ? o[a][i][k] : wm * so_far + wo * o[a][i][k];
          }
      }
    }
  }

  // ---- normalise and store: the wave turns its 32 x D tile round through the LDS nobody reads any more (the
  // barrier above ended the last tile), so that whole rows leave as consecutive bytes
  constexpr int ORS = 4 * D + 16;
  constexpr int LPR = D / 4;   // 16-byte chunks per row
  unsigned char* const ot = smem + wave * (32 * ORS);
  if constexpr (DIRECT) split_scale((unsigned)o_eb << 23, &v_scale, &v_inv);
  const float fin = v_inv / l;   // l in the scale of the weights' planes, as O's accumulators
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float4 o;
      o.x = om[dt][4 * g + 0] * fin;
      o.y = om[dt][4 * g + 1] * fin;
      o.z = om[dt][4 * g + 2] * fin;
      o.w = om[dt][4 * g + 3] * fin;
      *reinterpret_cast<float4*>(ot + j * ORS + 4 * (32 * dt + 8 * g + 4 * hh)) = o;
    }
#pragma unroll
  for (int idx = lane; idx < 32 * LPR; idx += 64) {
    const int r = idx / LPR, c = idx - r * LPR;
    const v4u piece = *reinterpret_cast<const v4u*>(ot + r * ORS + 16 * c);
    const int row = q_base + r;
    if (row < Sq) __builtin_nontemporal_store(piece, reinterpret_cast<v4u*>(Og + (size_t)row * D + 4 * c));
  }
}

static size_t round256f(size_t v) { return (v + 255) / 256 * 256; }

// How the work is laid out: waves (of 32 query rows) and key groups of a workgroup, and workgroups that share a block's keys.
struct F32Split {
  int waves, groups, parts;
  bool direct;   // the attention kernel cuts K and V into planes itself
};
static F32Split f32_split(long long BH, int Sq, int Skv, int D, int cus) {
  const int tiles = (Skv + FA_KT - 1) / FA_KT;
  // What the planes in a launch or two of their own cost beyond the attention kernel's, and what cutting them itself costs that (us): for
  // every tile of a wave more, for each query block again, and most where the wave is alone on its SIMD and has no registers left.
  // Fitted to 137 grids of 2 to 96 heads, 64 to 2048 queries and keys.  us with planes and without: 16 heads S 1024 D 32 20.0, 17.9; 12 heads
  // S 96 D 64 10.7, 7.9; 64 heads S 448 D 64 28.3, 20.4; 68 heads S 243 D 96 24.8, 19.1; 69 heads S 186 D 128 25.2, 19.9; the other
  // way round 24 heads S 1728 D 64 85.8, 89.3; 12 heads S 1536 D 128 72, 105.
  const float planes_us = 2.7f + 0.3e-6f * 8.0f * (float)BH * (float)Skv * (float)D;
  // (chain: tiles of a wave; per_simd: waves that a SIMD gets in turn or at once)
  auto direct_us = [&](int chain, long long per_simd) {
    const float tile = D == 32 ? (per_simd == 1 ? 0.33f : 0.15f) : D == 64 ? (per_simd == 1 ? 0.6f : 0.23f) : D == 96 ? 0.7f : 1.45f;
    return tile * (float)chain * (float)per_simd;
  };
  const long long blocks = (long long)((Sq + 127) / 128) * BH;
  if (blocks > 2 * cus) return {4, 1, 1, direct_us(tiles, (blocks + cus - 1) / cus) < planes_us};
  // Time in tenths of what a wave that shares its SIMD needs for a tile (1.05, 1.35, 1.7, 1.9 us by head size).  Two waves of a SIMD
  // hardly overlap, so what counts is the tiles that a SIMD works through; one that has only one wave takes a fifth longer.  What
  // parts leave in the workspace and the last one takes in costs 1.4, 1.6, 2.2, 2.6 us and 0.55, 0.7, 0.85, 1.05 us a part: as much as
  // 35 tenths with four to six parts, at every head size.  Over 580 grids of 1 to 64 heads, 32 to 4096 queries and 128 to 8192
  // keys the split chosen takes 2.5, 3.3, 0.7 and 1.6 % longer in the mean than the best one of all for the grid, a quarter at the most; 25
  // tenths serve as well, with 20 or 50 it is up to 1 % more.
  const int merge = 35, blocks128 = (int)blocks, blocks64 = (Sq + 63) / 64 * (int)BH;
  const float tenths = 1.0f / (D == 32 ? 0.105f : D == 64 ? 0.135f : D == 96 ? 0.17f : 0.19f);
  // What a split saves that cuts K and V itself counts for it (parts do not: their counters are cleared by the launch in front), but
  // for longer chains of sums than the cheapest split has without that it is not taken.
  struct Found {
    F32Split split;
    int cost, chain;
  };
  Found plain = {{4, 1, 1, false}, 1 << 30, 0}, best = plain;
  auto consider = [&](int waves, int groups, int parts) {
    const int workgroups = (waves == 4 ? blocks128 : blocks64) * parts, shares = groups * parts;
    const int resident = D <= 64 && groups == 1 ? 2 : 1;   // workgroups of a compute unit, by registers and LDS
    if (shares > 1 && (tiles < shares || workgroups > resident * cus)) return;
    const int chain = (tiles + shares - 1) / shares, per_simd = std::max(1, (workgroups + cus - 1) / cus * groups * waves / 4);
    const int cost = chain * (D > 64 ? 12 * per_simd : per_simd == 1 ? 12 : 10 * per_simd) + (parts > 1 ? merge : 0) + (groups > 1 ? 2 * groups : 0);
    const float saved = parts > 1 ? 0.0f : planes_us - direct_us(chain, per_simd);
    const bool direct = saved > 0.0f;
    const int without = cost - (direct ? (int)(saved * tenths) : 0);
    if (cost < plain.cost) plain = {{waves, groups, parts, direct}, cost, chain};
    if (without < best.cost) best = {{waves, groups, parts, direct}, without, chain};
  };
  consider(4, 1, 1);
  if (D <= 64) {
    consider(4, 2, 1);
    consider(2, 2, 1);
  }
  if (D == 32) consider(2, 4, 1);
  for (int parts = 2; parts <= 16; ++parts) {
    consider(4, 1, parts);
    if (D <= 64) consider(4, 2, parts);
  }
  return best.chain <= plain.chain ? best.split : plain.split;
}

struct F32Layout {
  size_t bits, chunks, kp, vp, partials, total;
  bool chunked;   // room for the largest magnitudes of chunks of a head
};
static F32Layout f32_layout(long long bh, int nqb, int parts, bool chunked, int Skv, int D) {
  F32Layout w;
  w.chunked = chunked;
  const size_t counters = parts > 1 ? (size_t)bh * nqb : 0;
  w.bits = 0;   // and the counters
  w.chunks = round256f(((size_t)2 * bh + counters) * sizeof(unsigned));
  w.kp = w.chunks + (chunked ? round256f((size_t)2 * bh * kMaxChunks * sizeof(unsigned)) : 0);
  w.vp = w.kp + round256f((size_t)bh * Skv * 2 * D * sizeof(_Float16));
  w.partials = w.vp + round256f((size_t)bh * Skv * 2 * D * sizeof(_Float16));
  w.total = w.partials + (parts > 1 ? round256f((size_t)bh * nqb * parts * f32_partial_bytes(D)) : 0);
  return w;
}

template <int D, int KG, int WAVES, bool PART, bool DIRECT = false>
static int launch_fa_f32_blocks(const float* Q, const void* kp, const void* vp, unsigned* bits, float* O, int BH, int Sq, int Skv,
                                float scale, int parts, char* partials, int lds_max, hipStream_t s) {
  using L = F32Tiles<D, KG>;
  const size_t lds = std::max((size_t)KG * 2 * (L::KTB + L::VTB), (size_t)WAVES * 32 * (4 * D + 16));
  if ((int)lds > lds_max) return fail(FTK_ERR_DEVICE, "ftk_flash_attn_f32: D=%d needs %zu bytes of LDS, the device offers %d", D, lds, lds_max);
  const int nqb = (Sq + 32 * WAVES - 1) / (32 * WAVES);
  const long long blocks = (long long)nqb * BH * parts;
  if (blocks > 0x7fffffffLL) return fail(FTK_ERR_UNSUPPORTED_SHAPE, "ftk_flash_attn_f32: grid too large");
  static DeviceOnce attr_once;
  unsigned attr_bit;
  if (attr_once.pending(&attr_bit)) {
    FTK_HIP(hipFuncSetAttribute((const void*)flash_attn_f32_kernel<D, KG, WAVES, PART, DIRECT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_once.done(attr_bit);
  }
  hipLaunchKernelGGL((flash_attn_f32_kernel<D, KG, WAVES, PART, DIRECT>), dim3((unsigned)blocks), dim3(KG * WAVES * 64), lds, s, Q, kp, vp, scale * 1.4426950408889634f,
                     (const unsigned*)bits, O, Sq, Skv, nqb, BH, parts, bits ? reinterpret_cast<int*>(bits + 2 * BH) : nullptr, reinterpret_cast<unsigned char*>(partials));
  return check_launch("flash_attn_f32_kernel");
}

template <int D>
static int launch_fa_f32(const float* Q, const float* K, const float* V, float* O, int BH, int Sq, int Skv, float scale, char* ws,
                         const F32Layout& w, const F32Split& split, const DeviceProps& dp, hipStream_t s) {
  unsigned* bits = reinterpret_cast<unsigned*>(ws + w.bits);
  _Float16* kp = reinterpret_cast<_Float16*>(ws + w.kp);
  _Float16* vp = reinterpret_cast<_Float16*>(ws + w.vp);
  const size_t per_bh = (size_t)Skv * D, head_bytes = per_bh * sizeof(float);
  // One launch while heads are small and what all its workgroups read for the largest magnitudes stays below 96 MB (a few
  // microseconds of L2); up to two workgroups to a compute unit (B 4, 16 heads, 1024 keys of 64: four parts each, 134 MB, were slower
  // than the launches below).
  const size_t all_heads = 2 * (size_t)BH * head_bytes, most_read = (size_t)96 << 20;
  const int parts = (int)std::max<size_t>(1, std::min({512 / (2 * (size_t)BH), per_bh / (8 * kPlanesThreads), most_read / all_heads}));
  const int counters = split.parts > 1 ? BH * ((Sq + 127) / 128) : 0;
  int rc = FTK_OK;
  if (split.direct) {
    // no planes
  } else if (head_bytes <= 512 * 1024 && all_heads * parts <= most_read) {
    hipLaunchKernelGGL(attn_f32_planes_kernel<D>, dim3((unsigned)(2 * BH * parts)), dim3(kPlanesThreads), 0, s, K, V, kp, vp, bits, Skv, BH, parts,
                       counters);
    rc = check_launch("attn_f32_planes_kernel");
    if (rc) return rc;
  } else {
    const int chunks = (int)std::min<size_t>({(size_t)std::max(1, 2048 / (2 * BH)), (per_bh + 4095) / 4096, kMaxChunks});
    unsigned* const chunk_bits = reinterpret_cast<unsigned*>(ws + (w.chunked ? w.chunks : w.vp));   // (8 bytes a chunk, of 16 KB of V's planes or a whole head's)
    hipLaunchKernelGGL(attn_f32_absmax_kernel, dim3(chunks, BH, 2), dim3(256), 0, s, K, V, chunk_bits, per_bh, BH);
    rc = check_launch("attn_f32_absmax_kernel");
    if (rc) return rc;
    if (!w.chunked) {
      hipLaunchKernelGGL(attn_f32_largest_kernel, dim3(2 * BH), dim3(64), 0, s, (const unsigned*)chunk_bits, chunks, bits);
      rc = check_launch("attn_f32_largest_kernel");
      if (rc) return rc;
    }
    const int wgs = (int)std::min<size_t>(std::max(1, 4096 / (2 * BH)), (per_bh / 8 + 255) / 256);
    hipLaunchKernelGGL(attn_f32_split_kernel<D>, dim3(wgs, BH, 2), dim3(256), 0, s, K, V, kp, vp, bits, (const unsigned*)(w.chunked ? chunk_bits : bits),
                       w.chunked ? chunks : 1, Skv, BH, counters);
    rc = check_launch("attn_f32_split_kernel");
    if (rc) return rc;
  }
  char* const partials = ws + w.partials;
  auto run = [&](auto groups_c, auto waves_c, auto part_c) {
    if constexpr (!decltype(part_c)::value) {
      if (split.direct)
        return launch_fa_f32_blocks<D, decltype(groups_c)::value, decltype(waves_c)::value, false, true>(Q, K, V, nullptr, O, BH, Sq, Skv, scale, 1, nullptr,
                                                                                                         dp.lds_optin, s);
    }
    return launch_fa_f32_blocks<D, decltype(groups_c)::value, decltype(waves_c)::value, decltype(part_c)::value>(
        Q, kp, vp, bits, O, BH, Sq, Skv, scale, split.parts, partials, dp.lds_optin, s);
  };
  std::integral_constant<int, 1> one;
  std::integral_constant<int, 2> two;
  std::integral_constant<int, 4> four;
  if constexpr (D == 32) {
    if (split.groups == 4) return run(four, two, std::false_type{});
  }
  if constexpr (D <= 64) {
    if (split.groups == 2 && split.waves == 2) return run(two, two, std::false_type{});
    if (split.groups == 2) return split.parts > 1 ? run(two, four, std::true_type{}) : run(two, four, std::false_type{});
  }
  return split.parts > 1 ? run(one, four, std::true_type{}) : run(one, four, std::false_type{});
}

}  // namespace ftk

extern "C" size_t ftk_flash_attn_f32_workspace_bytes(int B, int Hd, int Sq, int Skv, int D) {
  if (B <= 0 || Hd <= 0 || Sq <= 0 || Skv <= 0 || D <= 0) return 0;
  const ftk::DeviceProps* dp = nullptr;   // (without a device no call follows)
  const long long bh = (long long)B * Hd, nqb = (Sq + 127) / 128;
  const int parts = ftk::device_props(&dp) == FTK_OK ? ftk::f32_split(bh, Sq, Skv, D, dp->cus).parts : 1;
  return ftk::f32_layout(bh, (int)nqb, parts, true, Skv, D).total;
}

extern "C" int ftk_flash_attn_f32(const float* Q, const float* K, const float* V, float* O, int B, int Hd, int Sq, int Skv, int D,
                                  float scale, void* workspace, size_t workspace_bytes, ftk_stream_t stream) {
  using namespace ftk;
  const char* who = "ftk_flash_attn_f32";
  if (!Q || !K || !V || !O) return fail(FTK_ERR_INVALID_ARGUMENT, "%s: Q, K, V, O must be non-NULL", who);
  if (B <= 0 || Hd <= 0 || Sq <= 0 || Skv <= 0 || D <= 0) return fail(FTK_ERR_INVALID_ARGUMENT, "%s: B, Hd, Sq, Skv, D must be positive", who);
  if (D != 32 && D != 64 && D != 96 && D != 128) return fail(FTK_ERR_UNSUPPORTED_SHAPE, "%s: D=%d must be 32, 64, 96 or 128", who, D);
  if ((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) | reinterpret_cast<uintptr_t>(O)) % 16)
    return fail(FTK_ERR_INVALID_ARGUMENT, "%s: Q, K, V, O must be 16-byte aligned", who);   // rows are read and written 16 bytes at a time
  if (!(scale > 0.0f) || !(scale < INFINITY)) return fail(FTK_ERR_INVALID_ARGUMENT, "%s: scale must be positive and finite", who);
  const long long bh = (long long)B * Hd;
  if (bh > (1LL << 16)) return fail(FTK_ERR_UNSUPPORTED_SHAPE, "%s: B*Hd=%lld too large", who, bh);
  if ((long long)Skv * D >= (1LL << 31) || (long long)Sq * D >= (1LL << 31)) return fail(FTK_ERR_UNSUPPORTED_SHAPE, "%s: a head is too large", who);
  const int nqb = (Sq + 127) / 128;
  F32Layout w = f32_layout(bh, nqb, 1, false, Skv, D);
  if (!workspace || workspace_bytes < w.total)
    return fail(FTK_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, w.total, workspace ? workspace_bytes : (size_t)0);
  if (reinterpret_cast<uintptr_t>(workspace) % 256) return fail(FTK_ERR_INVALID_ARGUMENT, "%s: workspace must be 256-byte aligned", who);
  const DeviceProps* dp = nullptr;
  int rc = device_props(&dp);
  if (rc) return rc;
  F32Split split = f32_split(bh, Sq, Skv, D, dp->cus);
  // what a workspace smaller than the query asks for has no room for is done without
  const F32Layout cut = f32_layout(bh, nqb, split.parts, true, Skv, D), whole = f32_layout(bh, nqb, 1, true, Skv, D);
  if (workspace_bytes >= cut.total) w = cut;
  else if (workspace_bytes >= whole.total) w = whole;
  if (workspace_bytes < cut.total && split.parts > 1) split = {4, D <= 64 && bh * nqb <= dp->cus && Skv > 2 * FA_KT ? 2 : 1, 1, false};
  // An O that takes the place of K or V (or of part of them) is written when every row of theirs has gone into the planes
  auto over_o = [&](const float* kv) {
    const uintptr_t o = reinterpret_cast<uintptr_t>(O), at = reinterpret_cast<uintptr_t>(kv);
    const size_t row = (size_t)bh * D * sizeof(float);
    return o < at + row * Skv && at < o + row * Sq;
  };
  if (over_o(K) || over_o(V)) split.direct = false;
  hipStream_t s = (hipStream_t)stream;
  char* ws = reinterpret_cast<char*>(workspace);
  switch (D) {
    case 32: return launch_fa_f32<32>(Q, K, V, O, (int)bh, Sq, Skv, scale, ws, w, split, *dp, s);
    case 64: return launch_fa_f32<64>(Q, K, V, O, (int)bh, Sq, Skv, scale, ws, w, split, *dp, s);
    case 96: return launch_fa_f32<96>(Q, K, V, O, (int)bh, Sq, Skv, scale, ws, w, split, *dp, s);
    default: return launch_fa_f32<128>(Q, K, V, O, (int)bh, Sq, Skv, scale, ws, w, split, *dp, s);
  }
}
