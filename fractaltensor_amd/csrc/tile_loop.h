// The main loop of the kernels that form a 256 x 256 tile of an fp16 product with one wave per SIMD, each with a
// 128 x 128 piece of the tile in its accumulators (the plain product, gemm_f16.hip; the streamed LSTM cell, lstm_cell.hip).
//
// 32 MFMAs per 16 KB of fragments, a third less LDS traffic per product than with 128 x 64 outputs to a wave, and the
// whole register file (256 accumulator registers + fragments of two k steps).  With one wave per SIMD nothing fills a
// gap, so the loop leaves none it can avoid: the fragments of a k step are read while the MFMAs of the step before run,
// across the chunk boundary as well -- the barrier sits in the MIDDLE of a chunk, between its two k steps, where the
// second step's fragments are already in registers (what the chunk occupied in LDS is then free for copies) and
// the first step's fragments of the next chunk can be read behind it.
#pragma once

#include "ftk_common.h"

namespace ftk {

template <int V> using GIC = std::integral_constant<int, V>;

constexpr int GT = 256;               // rows and columns of a workgroup's tile
constexpr int GK = 32;                // k chunk: what a Bm stage holds; an A buffer holds a pair of chunks
constexpr int GS = 4;                 // Bm stages
constexpr int GP = 3;                 // A buffers
constexpr int G_ROWB = GT * 2;           // a Bm row of a chunk in LDS
constexpr int G_ABUF = GT * 128;         // A rows of a pair of chunks: 128 bytes, a whole cache line, each (32 KB)
constexpr int G_BST = GK * G_ROWB;       // 16 KB
constexpr int G_B0 = GP * G_ABUF;        // where the Bm stages start
constexpr int G_LDS = G_B0 + GS * G_BST; // 160 KB
constexpr int tile_vmcnt(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }   // s_waitcnt: vmcnt <= n, nothing else

typedef short g4s __attribute__((ext_vector_type(4)));
typedef short g8s __attribute__((ext_vector_type(8)));

// stage and buffer numbers: integral constants in the loop that is unrolled over them, ints elsewhere
template <int M, int V> __device__ __forceinline__ constexpr GIC<(V + 1) % M> next_of(GIC<V>) { return {}; }
template <int M> __device__ __forceinline__ int next_of(int v) { return v + 1 == M ? 0 : v + 1; }
template <int M, int V> __device__ __forceinline__ constexpr GIC<(V + M - 1) % M> prev_of(GIC<V>) { return {}; }
template <int M> __device__ __forceinline__ int prev_of(int v) { return v == 0 ? M - 1 : v - 1; }

// 16 bytes per lane from global memory (wave-uniform base + per-lane byte offset) into LDS at lds_addr + 16 * lane.
// The compiler does not count it: the loop waits with s_waitcnt vmcnt itself.
__device__ __forceinline__ void tile_dma16(const void* gbase, unsigned byte_off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds_addr), "v"(byte_off), "s"(gbase) : "memory", "m0");
}

// LDS: three A buffers, then four Bm stages.  An A buffer holds the tile's 256 rows of a pair of chunks, 128 bytes
// = 8 slots of 16 each: row r keeps k slot c in slot c ^ ((r >> 1) & 7) (16 rows in a row of one k slot fall on 16
// different 16-byte bank groups).  A copy brings 8 rows' whole 128-byte lines; with 64-byte rows, a chunk at a time,
// every line of A went from L2 to the compute unit twice.  Bm row k of a chunk (512 bytes, 32 slots = columns
// 8c .. 8c+7 of the tile) keeps slot c in c ^ ((k & 3) << 2).  The MFMA takes the Bm fragment as its first operand and
// the A fragment as its second: lane (j, hh) then holds, of output tile (rt, nt), row 32 rt + j and columns
// 32 nt + 8 q + 4 hh .. + 3 (q = 0..3) of its wave's piece (rows 128 (wave >> 1), columns 128 (wave & 1) of the tile).
//
// src says where the operands come from.  A pair's copy i (of 8, wave w: rows 64 w + 8 i + lane / 8 of the tile) fetches
// a_next + a_voff[i], or a_back[i & 1] bytes in front of that where the contraction ends in the middle of the pair
// (a_is_half(); what such a lane brings is never read); a chunk's copy i (of 4: k rows 8 w + 2 i + lane / 32) fetches
// b_next + b_voff[i].  a_advance / b_advance move the bases on by a pair / a chunk: (true_type) inside the unrolled loop,
// where the next one exists, (false_type) outside, where the bases have to stop at the last pair and chunk: what is
// requested beyond the end is the last once more, into a buffer nothing reads any more, so that every wait below
// counts the same number of copies whatever the length.  left_main_loop(ch): the unrolled loop ended in front of chunk ch.
// kOnce: what is fetched of Bm is not fetched again soon, and its copies (nt) leave no lines in the caches -- but for those
// outside the unrolled loop, where the last chunk is requested three times more and, without lines, came from memory each time
// (48 KB beside the tile's 1 MB at L 32 T 64 B 256 H 1024: 10.11 -> 9.81 ms).
template <typename Src>
__device__ __forceinline__ void tile_product(Src& src, int nch, v16f (&acc)[4][4]) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char tile_smem[];
  using lds_g4s = __attribute__((address_space(3))) g4s;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int j = lane & 31, hh = lane >> 5;
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)tile_smem);
  const unsigned lds_wave_a = lds0 + (unsigned)(wave * 8192);
  const unsigned lds_wave_b = lds0 + (unsigned)(G_B0 + wave * 4096);
  // Copy i (of 8) of the pair at src.a_next into A buffer ab / copy i (of 4) of the chunk at src.b_next into Bm stage bs: ints,
  // or GICs for numbers known to the compiler (the LDS address is then one scalar addition of a constant away).
  auto copy_a = [&](auto ab, auto i_c, bool half_pair) __attribute__((always_inline)) {
    constexpr int i = decltype(i_c)::value;
    if constexpr (std::is_integral_v<decltype(ab)>) {
      tile_dma16(src.a_next, src.a_voff[i] - (half_pair ? src.a_back[i & 1] : 0u), lds_wave_a + (unsigned)(ab * G_ABUF + i * 1024));
    } else {
      constexpr int AB = decltype(ab)::value;
      asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                   :: "s"(lds_wave_a), "n"(AB * G_ABUF + i * 1024), "v"(src.a_voff[i]), "s"(src.a_next) : "memory", "m0", "scc");
    }
  };
  auto copy_b = [&](auto bs, auto i_c) __attribute__((always_inline)) {
    constexpr int i = decltype(i_c)::value;
    if constexpr (std::is_integral_v<decltype(bs)>) {
      tile_dma16(src.b_next, src.b_voff[i], lds_wave_b + (unsigned)(bs * G_BST + i * 1024));
    } else {
      constexpr int BS = decltype(bs)::value;
      if constexpr (Src::kOnce)
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3 nt"
                     :: "s"(lds_wave_b), "n"(BS * G_BST + i * 1024), "v"(src.b_voff[i]), "s"(src.b_next) : "memory", "m0", "scc");
      else
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                     :: "s"(lds_wave_b), "n"(BS * G_BST + i * 1024), "v"(src.b_voff[i]), "s"(src.b_next) : "memory", "m0", "scc");
    }
  };
  // fragment addresses: A within buffers 0 and 1 (a read's immediate offset reaches 64 KB) and within buffer 2, per k
  // step of the pair; Bm within the four stages
  unsigned a_reg[2][4], b_reg[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    a_reg[0][ks] = (unsigned)((128 * wr + j) * 128 + (((2 * ks + hh) ^ ((j >> 1) & 7)) * 16));
    a_reg[1][ks] = a_reg[0][ks] + 2u * G_ABUF;
    asm volatile("" : "+v"(a_reg[0][ks]), "+v"(a_reg[1][ks]));
  }
  {
    const int ta = (lane & 15) >> 2, tb = lane & 3, th = (lane >> 4) & 1;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      b_reg[nt] = (unsigned)(G_B0 + (8 * hh + ta) * G_ROWB + (((4 * (4 * wc + nt) + 2 * th + (tb >> 1)) ^ (ta << 2)) * 16) +
                             8 * (tb & 1));
      asm volatile("" : "+v"(b_reg[nt]));
    }
  }

#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[rt][nt][r] = 0.0f;

  // the two sets of fragments: one k step of 16 each (4 row tiles of A, 4 column tiles of Bm)
  v8h af0[4], bf0[4], af1[4], bf1[4];
  g4s blo[4];
  // read number n (0..11) of a k step's fragments, in the order in which the MFMAs want them: Bm tile 0 (two
  // halves), A tile 0, Bm tiles 1..3, A tiles 1..3.  The k step is KS4 (0..3) of the pair in A buffer ab, KS4 & 1
  // of the chunk in Bm stage bs.
  auto frag_read = [&](auto ab, auto bs, auto ks4_c, auto n_c, v8h (&af)[4], v8h (&bf)[4]) __attribute__((always_inline)) {
    constexpr int n = decltype(n_c)::value, KS4 = decltype(ks4_c)::value;
    constexpr int kind = n < 2 ? 0 : n == 2 ? 1 : n < 9 ? 0 : 1;            // 0: Bm half, 1: A
    constexpr int nt = (n < 2 || n >= 9) ? 0 : 1 + ((n - 3) >> 1), half = n < 2 ? n : (n - 3) & 1;   // for kind 0
    constexpr int rt = n == 2 ? 0 : n - 8;                                  // for kind 1
    if constexpr (kind == 1) {
      const unsigned char* pa;
      if constexpr (std::is_integral_v<decltype(ab)>) {
        pa = tile_smem + ab * G_ABUF + a_reg[0][KS4];
      } else {
        constexpr int AB = decltype(ab)::value;
        pa = tile_smem + a_reg[AB >> 1][KS4] + (AB & 1) * G_ABUF;
      }
      af[rt] = *reinterpret_cast<const v8h*>(pa + 4096 * rt);
    } else {
      const unsigned char* pb;
      if constexpr (std::is_integral_v<decltype(bs)>) pb = tile_smem + bs * G_BST + b_reg[nt];
      else pb = tile_smem + b_reg[nt] + decltype(bs)::value * G_BST;
      const g4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_g4s*)(pb + 16 * G_ROWB * (KS4 & 1) + 4 * G_ROWB * half));
      if constexpr (half == 0) {
        blo[nt] = v;
      } else {
        const g8s both = {blo[nt][0], blo[nt][1], blo[nt][2], blo[nt][3], v[0], v[1], v[2], v[3]};
        bf[nt] = __builtin_bit_cast(v8h, both);
      }
    }
  };

  // One k step: 16 MFMAs on (af, bf); under them the 12 fragment reads of the step after (A buffer nab, Bm stage
  // nbs, k step nks4) into (naf, nbf) and four of the wave's copies: SET 1 copies 0..3, SET 2 copies 4..7 of the pair
  // at a_next into A buffer cdst; SET 3 the chunk at b_next into Bm stage cdst (0: none).  MAIN: inside the unrolled
  // loop, where every pair and chunk asked for exists.
  auto k_step = [&](v8h (&af)[4], v8h (&bf)[4], auto nab, auto nbs, auto nks4, v8h (&naf)[4], v8h (&nbf)[4], auto set_c,
                    auto cdst, auto main_c) __attribute__((always_inline)) {
    constexpr int SET = decltype(set_c)::value;
    constexpr bool MAIN = decltype(main_c)::value;
    bool half_pair = false;
    if constexpr (!MAIN && (SET == 1 || SET == 2)) half_pair = src.a_is_half();
    static_for<16>([&](auto s_c) __attribute__((always_inline)) {
      constexpr int s = decltype(s_c)::value;
      constexpr int rt = s >> 2, nt = s & 3;
      if constexpr (s < 12) frag_read(nab, nbs, nks4, s_c, naf, nbf);
      acc[rt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[nt], af[rt], acc[rt][nt], 0, 0, 0);
      if constexpr (SET != 0 && s < 12 && s % 3 == 1) {   // steps 1 4 7 10
        if constexpr (SET == 3) copy_b(cdst, GIC<(s / 3)>{});
        else copy_a(cdst, GIC<(4 * (SET - 1) + s / 3)>{}, half_pair);
      }
      if constexpr (s < 12) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    });
    if constexpr (SET == 2) src.a_advance(main_c);
    if constexpr (SET == 3) src.b_advance(main_c);
    __builtin_amdgcn_sched_barrier(0);   // the step's last MFMAs stay in front of what follows
  };

  constexpr std::false_type bounded{};
  // ---- prologue.  The loop below requests, beside chunk c, the Bm rows of chunk c + 3 and then half of an A pair:
  // the second half of pair c/2 + 2 when c is even, the first half of pair (c + 5)/2 when it is odd.  The prologue
  // requests what chunks -3, -2, -1 would have, behind pair 0: Bm 0, pair 1's first half, Bm 1, its second half,
  // Bm 2, pair 2's first half.
  static_assert(GS == 4 && GP == 3, "the order of the copies and the wait counts");
  {
    bool hp = src.a_is_half();
    static_for<8>([&](auto i_c) __attribute__((always_inline)) { copy_a(0, i_c, hp); });
    src.a_advance(bounded);
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_b(0, i_c); });
    src.b_advance(bounded);
    hp = src.a_is_half();
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_a(1, i_c, hp); });
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_b(1, i_c); });
    src.b_advance(bounded);
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_a(1, GIC<4 + decltype(i_c)::value>{}, hp); });
    src.a_advance(bounded);
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_b(2, i_c); });
    src.b_advance(bounded);
    hp = src.a_is_half();
    static_for<4>([&](auto i_c) __attribute__((always_inline)) { copy_a(2, i_c, hp); });
  }
  __builtin_amdgcn_s_waitcnt(tile_vmcnt(20));   // pair 0 and Bm 0 landed: 20 copies were requested behind them
  __builtin_amdgcn_s_barrier();
  static_for<12>([&](auto n_c) __attribute__((always_inline)) { frag_read(0, 0, GIC<0>{}, n_c, af0, bf0); });

  // Chunk ch = the HALF-th of the pair in A buffer ab, in Bm stage bs.
  auto chunk = [&](auto half_c, auto ab, auto bs, auto main_c) __attribute__((always_inline)) {
    constexpr int HALF = decltype(half_c)::value;
    k_step(af0, bf0, ab, bs, GIC<(2 * HALF + 1)>{}, af1, bf1, GIC<3>{}, prev_of<GS>(bs), main_c);
    // Chunk ch + 1 landed: copies complete in the order of their issue, and behind its Bm rows (its A rows are older)
    // 16 copies were requested: half a pair, the Bm rows of chunk ch + 2, half a pair, those of chunk ch + 3.  And
    // this wave's reads of chunk ch are complete.
    __builtin_amdgcn_s_waitcnt(tile_vmcnt(16) & 0xC07F);   // and lgkmcnt(0)
    __builtin_amdgcn_s_barrier();   // every wave has chunk ch in registers
    if constexpr (HALF == 0) {   // the second half of the pair after next, into the buffer in front of this one
      k_step(af1, bf1, ab, next_of<GS>(bs), GIC<2>{}, af0, bf0, GIC<2>{}, prev_of<GP>(ab), main_c);
    } else {                     // this buffer is free: the first half of the pair three on
      k_step(af1, bf1, next_of<GP>(ab), next_of<GS>(bs), GIC<0>{}, af0, bf0, GIC<1>{}, ab, main_c);
    }
  };
  int ch = 0;
  for (; ch + 18 < nch; ch += 12) {   // every copy these twelve chunks request lies inside K
    static_for<12>([&](auto c_c) __attribute__((always_inline)) {
      constexpr int c = decltype(c_c)::value;
      chunk(GIC<(c & 1)>{}, GIC<((c >> 1) % GP)>{}, GIC<(c % GS)>{}, std::true_type{});
    });
  }
  src.left_main_loop(ch);
  int ab = 0, bs = 0;   // ch is a multiple of 12
  for (; ch < nch; ch += 2) {
    chunk(GIC<0>{}, ab, bs, std::false_type{});
    bs = next_of<GS>(bs);
    if (ch + 1 < nch) chunk(GIC<1>{}, ab, bs, std::false_type{});
    bs = next_of<GS>(bs);
    ab = next_of<GP>(ab);
  }
  __builtin_amdgcn_s_waitcnt(tile_vmcnt(0));   // no copy into LDS outlives the workgroup
}

}  // namespace ftk
