// Plain fp16 product C = A @ Bm for shapes made of whole 256 x 256 tiles: one wave per SIMD, each with a
// 128 x 128 piece of the workgroup's tile in its accumulators (the loop is tile_loop.h).
#include <algorithm>

#include "ftk_common.h"
#include "tile_loop.h"

namespace ftk {

// Where the loop finds the operands of a tile of A [M, K] @ Bm [K, N].
struct GemmSource {
  static constexpr bool kOnce = false;
  unsigned a_voff[8], b_voff[4], a_back[2];
  const char *a_next, *b_next;
  size_t b_chunk;
  int nch, npairs, a_idx, b_idx;   // a_idx, b_idx: used outside the unrolled loop only
  template <typename Main>
  __device__ __forceinline__ void a_advance(Main) {
    if constexpr (Main::value) a_next += 128;
    else if (a_idx + 1 < npairs) { a_next += 128; ++a_idx; }
  }
  template <typename Main>
  __device__ __forceinline__ void b_advance(Main) {
    if constexpr (Main::value) b_next += b_chunk;
    else if (b_idx + 1 < nch) { b_next += b_chunk; ++b_idx; }
  }
  __device__ __forceinline__ void left_main_loop(int ch) {
    a_idx = min(ch / 2 + 2, npairs - 1);
    b_idx = min(ch + 3, nch - 1);
  }
  __device__ __forceinline__ bool a_is_half() const { return (nch & 1) != 0 && a_idx == npairs - 1; }
};

__global__ __launch_bounds__(256, 1) void gemm_f16_tile_kernel(const _Float16* __restrict__ A, const _Float16* __restrict__ Bm,
                                                                _Float16* __restrict__ C, int M, int N, int K) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int j = lane & 31, hh = lane >> 5;
  // Which tile: workgroups go to the 8 XCDs round-robin by their linear index, and the 32 that an XCD runs together
  // should share operands in its L2.  XCD x takes the x-th eighth of the tiles in walking order, and the walk goes
  // down a band of 8 (4, 2, 1) row blocks before it moves one column block on: 32 tiles in a row of the walk are 8 row
  // blocks x 4 column blocks, 12 operand panels for 32 tiles.
  const int tiles_m = (M + GT - 1) / GT, tiles_n = N / GT, per = tiles_m * tiles_n;
  int v = (int)blockIdx.x;
  if ((gridDim.x & 7) == 0) v = (v & 7) * (int)(gridDim.x >> 3) + (v >> 3);
  const int prob = v / per, t = v % per;
  const int bh = (tiles_m & 7) == 0 ? 8 : (tiles_m & 3) == 0 ? 4 : (tiles_m & 1) == 0 ? 2 : 1;
  const int band = t / (bh * tiles_n), r = t % (bh * tiles_n);
  const int m0 = (band * bh + r % bh) * GT, n0 = (r / bh) * GT;
  A += (size_t)prob * M * K;
  Bm += (size_t)prob * K * N;
  C += (size_t)prob * M * N;
  GemmSource src;
  src.nch = K / GK;
  src.npairs = (src.nch + 1) >> 1;

  // copies: wave w brings A rows 64 w .. + 64 of a pair of chunks (copy i of 8: 8 rows, row lane / 8) and Bm rows
  // 8 w .. + 8 of a chunk (copy i of 4: 2 rows, row lane / 32)
  unsigned b_lane[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const unsigned kr = (unsigned)(2 * p + (lane >> 5));   // k row & 3
    b_lane[p] = ((unsigned)lane >> 5) * (unsigned)(2 * N) + ((((unsigned)lane & 31) ^ (kr << 2)) * 16);
  }
  // a copy's lane offsets from its operand's base; the bases move on by a pair and by a chunk.  (Rows past the end
  // of A repeat its last row; they are never stored.)
  const int a_row0 = min(m0 + 64 * wave, M - 1);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = min(m0 + 64 * wave + 8 * i + (lane >> 3), M - 1);
    src.a_voff[i] = (unsigned)(row - a_row0) * (unsigned)(2 * K) + (unsigned)(((lane & 7) ^ (4 * (i & 1) + (lane >> 4))) * 16);
    asm volatile("" : "+v"(src.a_voff[i]));   // kept in registers, not formed again at every copy
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    src.b_voff[i] = b_lane[i & 1] + (unsigned)i * (unsigned)(2 * 2 * N);
    asm volatile("" : "+v"(src.b_voff[i]));
  }
  // K an odd number of chunks: the last pair is half a pair, and the lanes of its copies whose k slot lies beyond K
  // take the slot 64 bytes in front of it (what they bring is never read)
  src.a_back[0] = (unsigned)(((lane >> 2) & 1) * 64);
  src.a_back[1] = (unsigned)((((lane >> 2) & 1) ^ 1) * 64);
  src.a_next = reinterpret_cast<const char*>(A + (size_t)a_row0 * K);   // of the pair that is copied next
  src.b_next = reinterpret_cast<const char*>(Bm + (size_t)(8 * wave) * N + n0);   // of the chunk ...
  src.a_idx = src.b_idx = 0;
  src.b_chunk = (size_t)GK * N * 2;
  v16f acc[4][4];
  tile_product(src, src.nch, acc);

  // ---- epilogue.  Of a tile's row, lane (j, 0) holds columns 8 q .. + 3 and lane (j, 1) columns 8 q + 4 .. + 7 for
  // q = 0..3: the two lanes exchange the halves of an even and an odd q, so that lane (j, 0) stores the 8 columns of
  // the even q and lane (j, 1) those of the odd one, 16 bytes each.
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int row = m0 + 128 * wr + 32 * rt + j;
    _Float16* crow = C + (size_t)row * N + n0 + 128 * wc + 8 * hh;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int qp = 0; qp < 2; ++qp) {
        v2u ev, od;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const v2h e = {(_Float16)acc[rt][nt][8 * qp + 2 * w], (_Float16)acc[rt][nt][8 * qp + 2 * w + 1]};
          const v2h o = {(_Float16)acc[rt][nt][8 * qp + 4 + 2 * w], (_Float16)acc[rt][nt][8 * qp + 4 + 2 * w + 1]};
          ev[w] = __builtin_bit_cast(unsigned, e);
          od[w] = __builtin_bit_cast(unsigned, o);
          // upper lanes' ev <-> lower lanes' od
          asm volatile("s_nop 1\n\tv_permlane32_swap_b32_e32 %0, %1\n\ts_nop 1" : "+v"(ev[w]), "+v"(od[w]));
        }
        const v4u o = {ev[0], ev[1], od[0], od[1]};
        if (row < M) *reinterpret_cast<v4u*>(crow + 32 * nt + 16 * qp) = o;
      }
  }
}

// true when the tile kernel takes the shape
bool gemm_f16_tiles_fit(int M, int N, int K) { return M > 0 && N % GT == 0 && K % GK == 0; }

int launch_gemm_f16_tiles(const void* A, const void* Bm, void* C, int G, int M, int N, int K, hipStream_t s) {
  static DeviceOnce attr_once;
  constexpr int lds = G_LDS;
  unsigned attr_bit;
  if (attr_once.pending(&attr_bit)) {
    FTK_HIP(hipFuncSetAttribute((const void*)gemm_f16_tile_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    attr_once.done(attr_bit);
  }
  const long long tiles = (long long)G * ((M + GT - 1) / GT) * (N / GT);
  if (tiles >= (1ll << 31)) return fail(FTK_ERR_UNSUPPORTED_SHAPE, "gemm: too many tiles");
  hipLaunchKernelGGL(gemm_f16_tile_kernel, dim3((unsigned)tiles), dim3(256), lds, s, (const _Float16*)A, (const _Float16*)Bm,
                     (_Float16*)C, M, N, K);
  return check_launch("gemm_f16_tile_kernel");
}

}  // namespace ftk
