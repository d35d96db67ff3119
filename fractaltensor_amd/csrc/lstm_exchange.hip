// Stacked / dilated LSTM for stacks that wait: one launch for the whole (layer, time) grid, made for the time a
// hidden state takes from the compute units that produce it to the compute units that need it next.
//
// What bounds such a stack is not its products but its chain of L + T - 1 dependent steps, so everything here is
// about the length of one step.  A layer is spread over H / 16 workgroups of 4 waves (a team; with several row
// slices a layer has several teams, each with batch rows of its own).  A workgroup owns 16 hidden units = 64 gate
// columns and keeps its slice of [W;U] in registers for the whole launch.  An item is a block of 16 batch rows of one time
// step (32 rows where a workgroup has several blocks to walk; exchange_layers chooses):
//
//   * Its four waves cut the CONTRACTION, not the columns: wave w multiplies quarter w of x_t and quarter w of h_{t-d}
//     with all 64 columns.  A wave therefore loads exactly the activations it needs, from memory straight into the
//     registers the matrix instruction reads (v_mfma_f32_16x16x32_f16, weights as the A operand, activations as B):
//     no tile in LDS and nothing read twice by a compute unit.  The four partial sums of a column meet in LDS, one
//     barrier per item.
//   * The 16 columns of a matrix instruction are 4 units x {i, f, o, c~}, so a lane gets the four gates of one
//     (row, unit) and the state update is one of its own values.
//   * h is handed over as data, without flags.  The words of the exchange buffers hold a value no h can have (all
//     ones: a NaN) until h is there, and whoever needs h loads the words until none of them is that value.  One trip of
//     the data instead of data, acknowledgement, flag, look at the flag, data.
//   * A team sits on one XCD (workgroups are dealt to the XCDs in turn, and the kernel compares the XCC ids it finds),
//     so its members hand h over through the L2 they share: plain stores, agent-scope loads.  Measured between 8 / 16 /
//     32 workgroups that exchange a whole tile: 0.49 / 0.76 / 0.98 us a step, against 0.81 / 1.24 / 1.71 us with
//     write-through stores, which is what a team that does not sit together uses.
//
// A step of a single layer takes 0.85 us at H = 64, 0.9 at 128, 1.2 at 256 and 1.9 at 512 (fp32), where a hand-over of the
// persistent kernel's serial schedule took 5 to 6 and a launch per step 20 and more: L 20 T 30 B 32 H 128 1004 -> 76 us,
// L 8 T 100 B 64 H 512 7.3 -> 0.72 ms, L 1 T 16 B 64 H 256 100 -> 29 us.
//
// The exchange buffers.  ring: the own layer's h for d = 1, four steps deep.  A workgroup that has all of h(t-1) knows
// that every member of its team has read h(t-2) (it published h(t-1) behind a barrier that all its waves reached after
// they had h(t-2)), so it sets its words of slot t-2 back to all ones, which are used again at t+2.  hand: every h of
// every layer, for the layer above and for dilated recurrences; the producer itself sets the words of step t+2 to
// all ones before it publishes step t+1, and a consumer looks at step t+2 only after it has seen step t+1.  The first
// two steps, the ring and the input rows (in the same form) are written at the start of the launch itself
// (exchange_lay_out), or by a small kernel in front where that does not serve (run_exchange).
//
// Products.  fp32 data: an operand is an fp16 value and the fp16 of what that leaves, under a power-of-two scale of its
// weight column or input row (h: 2^14); three fp16 matrix instructions per product, fp32 accumulation (see
// lstm_persistent.hip).  A word of the exchange buffers is the pair.  fp16 data: one instruction per product, the
// exchange buffers hold the fp16 h.
//
// Everything waits with a bound (spin_limit looks); when one runs out the status word is set and the launch drains.
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <random>

#include "ftk_common.h"

namespace ftk {

constexpr int kXLayers = 64;       // layers of one launch
constexpr int kXBlocks = 128;      // row blocks a ragged batch may have
constexpr int kXRing = 4;          // steps the own layer's ring holds
constexpr int kXPlaces = 2047;     // workgroups of one launch
constexpr int kXGaveUp = kXPlaces; // behind their places: the launch that a workgroup gave up in before all it waits for had come
constexpr int kXRowPlaces = 256;   // workgroups that lay out the input rows of a slice: what the layer that reads them looks at
constexpr int kXHandTop = 14;      // the scale of h: 2^14 (|h| < 1)
constexpr unsigned kXSmallBits = (127u - 12u - kXHandTop) << 23;   // h * 2^14 below 2^-12: see ftk_stacked_lstm_small_states

struct ExchangeArgs {
  const void* WU;
  const float* bias;
  void* hsss;
  void* csss;
  int* status;          // [0] error word, [1] small states
  unsigned long long* place;   // [groups]: launch << 8 | 1 + the XCC id, of every workgroup that is there and has laid out what it has to; [kXGaveUp]
  unsigned long long launch;   // what tells this launch's words from any that were there before
  const void* xs;       // not null: this launch lays out its own buffers (exchange_lay_out)
  unsigned char* ring;  // [L][nrb][kXRing] tiles
  unsigned char* hand;  // [L + 1][T][nrb] tiles: the input rows, then every layer's h
  float* xratio;        // [row block][T, rounded up to even][row of it] what the products of an input row are multiplied by to match h's (fp32 data)
  int L, T, B, nrb;
  int slices;           // row slices = teams per layer; slice s walks row blocks s, s + slices, ...
  int units;            // L * slices teams
  int per_xcd;          // > 0: teams per XCD, unit u on XCD u / per_xcd; 0: workgroups in order
  int spin_limit;
  int ragged;
  int row_layers;       // xs: layers whose workgroups lay out the input rows of their slice
  int clear_status;     // xs: this launch clears the status words
  int early;            // no h goes to another XCD: fp32 teams with one row block look for theirs at once (walk_lean)
  int dil[kXLayers];
  int steps_of[kXBlocks];   // ragged: steps row block rb takes part in (T reaches 262143 at H = 64)
};

typedef unsigned long long u64;
typedef float v2f __attribute__((ext_vector_type(2)));

// How words leave a workgroup that is not in a hurry: to `hand` as plain stores (the layer above, if any, on this XCD) or
// write-through, to the ring as plain ones; or (teams over several XCDs) as either, by two stores of which one is out of bounds.
enum { kAnyWay, kPlain, kThrough };
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
// four weights at any place a caller's array may begin
typedef float weights4f __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 weights4h __attribute__((ext_vector_type(4), aligned(2)));
constexpr int kAgentScope = 16;      // sc1 in the cache-policy operand of a buffer load

// A tile of the exchange buffers: the h of a row block.  fp32 data: [H / 4][rows][4 units] words (value, remainder); fp16
// data: [H / 8][rows][8 units] halves.  What a wave stores is contiguous, what a lane loads is 16 bytes.
constexpr int exchange_tile_bytes(int H, bool half, int rows) { return H * rows * (half ? 2 : 4); }

// Hidden units of a workgroup.  Where the batch is large enough to keep workgroups busy (many) a workgroup takes as many
// columns as its registers hold at one workgroup per compute unit: every column more is a use more of an activation that
// has to come through L2 anyway.
constexpr int exchange_units(int H, bool half, bool many) { return many && H * (half ? 1 : 2) == 512 ? 32 : 16; }
// Workgroups a compute unit is to hold: the weights of 16 units take H / 2 registers of a lane (fp16 data: H / 4).
constexpr int exchange_per_cu(int H, bool half, bool many) {
  const int weights = H * exchange_units(H, half, many) / (half ? 64 : 32);
  return weights >= 256 ? 1 : weights >= 128 || many ? 2 : 3;
}

// x times a power of two as an fp16 value and the fp16 of what that leaves: two instructions.
__device__ __forceinline__ v2h value_and_rest(float x, float scale) {
  const _Float16 top = (_Float16)__builtin_fmaf(x, scale, 0.0f);
  return v2h{top, (_Float16)__builtin_fmaf(x, scale, -(float)top)};
}

// An input row in the form of the exchange buffers, by eight lanes, piece i of a lane's N being k group 8 i + lane / 8: put(i, w)
// takes its 16 bytes, ratio(r) what the row's products are multiplied by.  fp32 rows are cut under a power-of-two scale of their own.
template <bool HALF, int N, typename Put, typename Ratio>
__device__ __forceinline__ void exchange_input_row(const v4u (&raw)[N], Put put, Ratio ratio) {
  if constexpr (HALF) {
#pragma unroll
    for (int i = 0; i < N; ++i) put(i, raw[i]);
  } else {
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(__uint_as_float(raw[i][e])));
#pragma unroll
    for (int o = 32; o >= 8; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    const int eb = min(max((int)((__float_as_uint(mx) >> 23) & 0xff), 15), 254);
    const float scale = __uint_as_float((unsigned)(127 + 14 + 127 - eb) << 23);   // the row's largest -> [2^14, 2^15)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v4u w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = __builtin_bit_cast(unsigned, value_and_rest(__uint_as_float(raw[i][e]), scale));
      put(i, w);
    }
    ratio(__uint_as_float((unsigned)eb << 23));   // the products carry 2^(141 - eb), h's 2^14
  }
}

// Before the first step of a launch that lays out its own buffers.  What others of this launch look at (see the top of the file) is written
// here, in front of the weights; then the workgroup's place says that it is done.  Whoever reads waits for the places it depends on, and a
// place is known as this launch's by the number in it, so nothing has to be cleared before the launch.  Words are written through, and no line of
// them is written by two workgroups (they begin on a line of their own: exchange_places_at): no cache holds a part of one.
//
// Bound by latency: input rows that come from memory, stores that go there, places that come from there.  It takes 2 to 3 us where the kernel in
// front took 3.4 to 12 and a launch (us a call with other inputs and weights each time, that kernel and this: L 2 T 36 B 155 H 64 48.6, 46.6; L 1 T 64
// B 100 H 512 145.2, 141.6; L 8 T 100 B 64 H 512 716, 714; fp16 L 10 T 30 B 99 H 256 125.2, 120.3).  With the places
// behind the weights, and the rows between the loads of them, single layers began as early, but the places of a workgroup whose weights came late
// held up the others (fp16 L 10 T 30 B 99 H 256 144.5), and all waves looking at them held up the weights.
template <int H, bool HALF, bool MANY, typename Args>
__device__ __forceinline__ void exchange_lay_out(const Args& a, int unit, int s, int l, int pc) {
  constexpr int W = H / exchange_units(H, HALF, MANY), ROWS = MANY ? 32 : 16, TILE = exchange_tile_bytes(H, HALF, ROWS);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T = a.T, B = a.B, nrb = a.nrb;
  // The input rows, 32 to a workgroup and 8 to a wave at a time: lane (row, k group) so that a store covers whole lines.
  constexpr int PIECES = H / (HALF ? 64 : 32);
  v4u raw[PIECES];
  const int steps = (T + 1) & ~1, per_block = steps * ROWS / 32;
  int group = l * W + pc;
  const int groups = l < a.row_layers ? (MANY ? (nrb - s + a.slices - 1) / a.slices * per_block : per_block) : 0;
  int t, rb, m;   // this lane's row: time step (the last may be past the end), row block, row of it
  auto ask = [&]() __attribute__((always_inline)) {
    const int block = MANY ? group / per_block : 0, r = (group - block * per_block) * 32 + wave * 8 + (lane & 7);
    rb = s + block * a.slices;
    t = r / ROWS;
    m = r % ROWS;
    const char* const from = reinterpret_cast<const char*>(a.xs) + ((size_t)min(t, T - 1) * B + min(rb * ROWS + m, B - 1)) * (H * (HALF ? 2 : 4));
#pragma unroll
    for (int i = 0; i < PIECES; ++i) raw[i] = reinterpret_cast<const v4u*>(from)[8 * i + (lane >> 3)];
  };
  if (group < groups) ask();
  asm volatile("" ::: "memory");

  // the words of this workgroup's units that stand for "not there yet": the ring, and the first two steps of `hand`
  {
    const auto ring = __builtin_amdgcn_make_buffer_rsrc(a.ring + (size_t)l * nrb * kXRing * TILE, 0, (unsigned)(nrb * kXRing * TILE), 0x00020000);
    const auto hand = __builtin_amdgcn_make_buffer_rsrc(a.hand + (size_t)(l + 1) * T * nrb * TILE, 0, (unsigned)((size_t)T * nrb * TILE), 0x00020000);
    constexpr int PART = TILE / W, STORES = PART / 16, AT_ONCE = 256 / STORES;   // bytes of a tile; tiles at a time
    static_assert(256 % STORES == 0, "whole tiles at a time");
    const v4u ones = {~0u, ~0u, ~0u, ~0u};
    const int first = tid / STORES, at = pc * PART + tid % STORES * 16;
    for (int rb = s; rb < (MANY ? nrb : s + 1); rb += a.slices) {
#pragma unroll
      for (int i = 0; i < kXRing; i += AT_ONCE)
        if (i + first < kXRing) __builtin_amdgcn_raw_buffer_store_b128(ones, ring, (rb * kXRing + i + first) * TILE + at, 0, kAgentScope);
#pragma unroll
      for (int i = 0; i < 2; i += AT_ONCE)   // (a step past the last is out of the buffer)
        if (i + first < 2) __builtin_amdgcn_raw_buffer_store_b128(ones, hand, ((i + first) * nrb + rb) * TILE + at, 0, kAgentScope);
    }
  }
  if (a.clear_status && unit == 0 && pc == 0 && tid < (int)(kStatusBytes / sizeof(int)))
    __hip_atomic_store(a.status + tid, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  const auto rows = __builtin_amdgcn_make_buffer_rsrc(a.hand, 0, (unsigned)((size_t)T * nrb * TILE), 0x00020000);
  const auto ratios = __builtin_amdgcn_make_buffer_rsrc(a.xratio, 0, (unsigned)((size_t)nrb * steps * ROWS * 4), 0x00020000);
  while (group < groups) {
    const unsigned live = rb * ROWS + m < B ? ~0u : 0u;   // rows past the batch are zeros
#pragma unroll
    for (int i = 0; i < PIECES; ++i) raw[i] &= live;
    const unsigned at = t < T ? (unsigned)((t * nrb + rb) * TILE + m * 16 + (lane >> 3) * (ROWS * 16)) : 0x80000000u;
    exchange_input_row<HALF>(raw, [&](int i, v4u w) __attribute__((always_inline)) {
      __builtin_amdgcn_raw_buffer_store_b128(w, rows, at, i * (8 * ROWS * 16), kAgentScope);
    }, [&](float ratio) __attribute__((always_inline)) {
      if (lane < 8) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ratio), ratios, ((rb * steps + t) * ROWS + m) * 4, 0, kAgentScope);
    });
    group += a.row_layers * W;
    if (group < groups) ask();
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): what this wave wrote is in memory
  __syncthreads();
}

// MANY == false: one row block of 16 rows per workgroup, where an item waits for the one before it and the wait is what is
// being shortened.  MANY: row blocks of 32 rows (v_mfma_f32_32x32x16_f16: a fifth less time per product, half the
// overhead per row), usually several per workgroup, so that the next item's h is there before this one is done.
template <int H, bool HALF, bool MANY>
__global__ __launch_bounds__(256, exchange_per_cu(H, HALF, MANY))
void lstm_exchange_kernel(ExchangeArgs a) {
  constexpr int UNITS = exchange_units(H, HALF, MANY);
  constexpr int CT = UNITS / 16;
  constexpr int W = H / UNITS;               // workgroups of a team
  constexpr int RT = MANY ? 2 : 1;
  constexpr int ROWS = 16 * RT;              // rows of a block
  constexpr int KW = 32 / RT;                // k of a k step
  constexpr int NT = 4 * CT / RT;            // tiles of 16 RT gate columns
  constexpr int U = RT * CT;                 // units a lane updates
  constexpr bool ROLES = H / 4 < KW;         // a quarter of H is half a k step: waves 0, 1 take x, waves 2, 3 take h
  constexpr int XS = ROLES ? 1 : H / 4 / KW; // k steps per wave in the x half, and in the h half
  constexpr int KS = ROLES ? 1 : 2 * XS;     // resident k steps
  constexpr int NL = HALF ? XS : 2 * XS;     // 16-byte loads of a lane's share of a tile
  constexpr int TILE = exchange_tile_bytes(H, HALF, ROWS);
  constexpr int AR = 4 * RT * RT;            // accumulator registers of a tile
  typedef float accum __attribute__((ext_vector_type(AR)));
  typedef float sums __attribute__((ext_vector_type(4 * U)));   // the gates of a lane's units
  __shared__ sums red[2][4][4][64];          // [parity][wave that takes them][wave that gives them][lane]
  // h and c of an item, for the wave that stores them; a row's 16 units and some more: all lanes on different banks
  using Value = typename std::conditional<HALF, _Float16, float>::type;
  constexpr int OUT_ROW = HALF ? 24 : 20;
  __shared__ __attribute__((aligned(16))) Value outs[MANY ? 1 : 2][MANY ? 1 : 2][MANY ? 1 : 16 * OUT_ROW];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane % ROWS;   // gate column of a weight fragment; batch row of everything else
  const int kg = lane / ROWS;  // k group of a fragment; which of its wave's units a lane updates

  int unit, pc;
  if (a.per_xcd > 0) {
    const int slot = blockIdx.x >> 3, n = slot / W;
    unit = (int)(blockIdx.x & 7) * a.per_xcd + n;
    pc = slot % W;
    if (n >= a.per_xcd) return;
  } else {
    const int q = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    unit = q / W;
    pc = q % W;
  }
  if (unit >= a.units) return;
  const int s = unit / a.L, l = unit % a.L;
  const int d = a.dil[l];
  const int T = a.T, B = a.B, nrb = a.nrb;

  int xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  xcc = (xcc & 0x7f) + 1;

  // (the arguments are read again for it: what the loops need of them would be kept in registers otherwise, from here on)
  auto* again = (const __attribute__((address_space(4))) ExchangeArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(again));
  if (again->xs) exchange_lay_out<H, HALF, MANY>(*again, unit, s, l, pc);
  if (tid == 0) __hip_atomic_store(a.place + unit * W + pc, a.launch << 8 | (unsigned)xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // ---- resident weights: lane (m, kg) holds rows KW i + 8 kg .. +7 of column m of tile tt, for k step i.
  // A column is a gate of a unit, ordered so that a lane gets the four gates of a unit next to each other in its
  // accumulators (lane (m, kg) has rows 4 kg .. +3 of a 16-row result, and rows 8 q + 4 kg .. +3, q = 0 .. 3, of a
  // 32-row one) and, with 32-row results, neighbouring units: two of the half tile its wave finishes, or four of a tile.
  // With 16-row results the four tiles hold a lane four neighbouring units of a gate, which is what one load brings: with
  // a load for each weight H 512 took 16 us to begin.
  auto unit_of = [](int tt, int col) {
    if (RT == 1) return 4 * (col >> 2) + tt;
    if (CT == 1) return 8 * tt + 4 * (col >> 4) + 2 * ((col >> 2) & 1) + ((col >> 3) & 1);
    return 8 * tt + 4 * ((col >> 2) & 1) + (col >> 3);
  };
  v8h wt[KS][NT], wo[HALF ? 1 : KS][HALF ? 1 : NT];
  constexpr float kLog2e = 1.4426950408889634f;
  auto w_row = [&](int i) {      // first row of WU of resident k step i
    if (ROLES) return 32 * wave;
    return i < XS ? wave * (H / 4) + KW * i : H + wave * (H / 4) + KW * (i - XS);
  };
  const int my_unit = UNITS * pc + 4 * CT * wave + U * kg;   // the first of the units whose state this lane updates
  float esc[HALF ? 1 : 4 * U], ebias[4 * U];                  // pre-activations: esc * sum + ebias, with -log2 e for the gates i, f, o
  {
    const size_t base = (size_t)l * 2 * H * 4 * H + (size_t)(m & 3) * H + UNITS * pc;
    int uo[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) uo[tt] = unit_of(tt, m);
    if constexpr (HALF) {
      const _Float16* wl = reinterpret_cast<const _Float16*>(a.WU) + base;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const _Float16* row = wl + (size_t)(w_row(i) + 8 * kg + e) * 4 * H;
          if constexpr (RT == 1) {
            const v4h w = *reinterpret_cast<const weights4h*>(row + uo[0]);
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) wt[i][tt][e] = w[tt];
          } else {
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) wt[i][tt][e] = row[uo[tt]];
          }
        }
        if (i % (2 * RT) == 2 * RT - 1) asm volatile("" ::: "memory");   // 16-bit loads take a register each until they are packed
      }
    } else {
      const float* wl = reinterpret_cast<const float*>(a.WU) + base;
      float raw[KS][NT][8];
#pragma unroll
      for (int i = 0; i < KS; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float* row = wl + (size_t)(w_row(i) + 8 * kg + e) * 4 * H;
          if constexpr (RT == 1) {
            const v4f w = *reinterpret_cast<const weights4f*>(row + uo[0]);
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) raw[i][tt][e] = w[tt];
          } else {
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) raw[i][tt][e] = row[uo[tt]];
          }
        }
      }
      // the largest magnitude of each of the workgroup's columns, over the four waves
      float* const cmaxs = reinterpret_cast<float*>(red);   // [4 waves][tile, column], then what undoes the scales
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        float cmax = 0.0f;
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) cmax = fmaxf(cmax, fabsf(raw[i][tt][e]));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
        if (RT == 1) cmax = fmaxf(cmax, __shfl_xor(cmax, 16));
        cmaxs[wave * (64 * CT) + tt * ROWS + m] = cmax;
      }
      __syncthreads();
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        float cmax = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) cmax = fmaxf(cmax, cmaxs[w * (64 * CT) + tt * ROWS + m]);
        const int eb = min(max((int)((__float_as_uint(cmax) >> 23) & 0xff), 40), 230);
        const float scale = __uint_as_float((unsigned)(127 + 14 + 127 - eb) << 23);   // column max -> [2^14, 2^15)
        cmaxs[256 * CT + tt * ROWS + m] = __uint_as_float((unsigned)(eb - 14 - kXHandTop) << 23);
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {   // six instructions for two
            const v2f w = {raw[i][tt][e] * scale, raw[i][tt][e + 1] * scale};
            const v2h top = __builtin_convertvector(w, v2h);
            const v2f left = {__builtin_fmaf(raw[i][tt][e], scale, -(float)top[0]), __builtin_fmaf(raw[i][tt][e + 1], scale, -(float)top[1])};
            const v2h rest = __builtin_convertvector(left, v2h);
            wt[i][tt][e] = top[0];
            wt[i][tt][e + 1] = top[1];
            wo[i][tt][e] = rest[0];
            wo[i][tt][e + 1] = rest[1];
          }
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          // tile and column of gate g of unit my_unit + u
          const int tt = RT == 1 ? kg : CT == 2 ? wave : wave >> 1;
          const int col = RT == 1 ? 4 * wave + g : CT == 2 ? 8 * u + 4 * kg + g : 16 * (wave & 1) + 8 * u + 4 * kg + g;
          esc[4 * u + g] = cmaxs[256 * CT + tt * ROWS + col] * (g == 3 ? 1.0f : -kLog2e);
        }
      __syncthreads();
    }
  }
  // Where the weights take more than half of the register file, the matrix instructions read some of them from the
  // accumulation registers, which nothing else can: left to itself the compiler keeps them there as spills and moves
  // every one back in front of the instruction that uses it.
  auto to_acc = [](v8h v) __attribute__((always_inline)) -> v8h {
    const v4u u = __builtin_bit_cast(v4u, v);
    unsigned a0, a1, a2, a3;
    asm("v_accvgpr_write_b32 %0, %1" : "=a"(a0) : "v"(u[0]));
    asm("v_accvgpr_write_b32 %0, %1" : "=a"(a1) : "v"(u[1]));
    asm("v_accvgpr_write_b32 %0, %1" : "=a"(a2) : "v"(u[2]));
    asm("v_accvgpr_write_b32 %0, %1" : "=a"(a3) : "v"(u[3]));
    const v4u r = {a0, a1, a2, a3};
    return __builtin_bit_cast(v8h, r);
  };
  if constexpr (H * CT * (HALF ? 1 : 2) >= 1024) {
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        if constexpr (HALF) {
          if (i % 8 != 7 || !MANY) wt[i][tt] = to_acc(wt[i][tt]);
        } else {
          wo[i][tt] = to_acc(wo[i][tt]);
          if (i % 4 < (MANY ? 3 : 2)) wt[i][tt] = to_acc(wt[i][tt]);
        }
      }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      ebias[4 * u + g] = a.bias ? a.bias[(size_t)l * 4 * H + g * H + my_unit + u] * (g == 3 ? 1.0f : -kLog2e) : 0.0f;

  // ---- do the team, and the team above that reads from it, sit on this XCD?
  const bool has_upper = l + 1 < a.L;
  // (looked at by one wave: all looking at all of them at once hold up the weights that other workgroups wait for)
  __shared__ int places_seen;
  if (wave == 0) {
    static_assert(W <= 64, "a lane for each workgroup of a team");
    const int i = min(lane, W - 1);
    // xs: what is read of others' is there: the status words, and the layer below, or the input rows
    const auto& b = *again;
    const bool own_buffers = b.xs != nullptr;
    const int from = l == 0 ? (unit - l) * W : (unit - 1) * W, count = !own_buffers ? 0 : l == 0 ? b.row_layers * W : W;
    auto place = [&](int at) __attribute__((always_inline)) { return __hip_atomic_load(b.place + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto missing_place = [&](u64 p) __attribute__((always_inline)) { return p >> 8 != b.launch; };
    // The workgroup that clears the status words may be the one that others have waited for in vain, and clear what they said.  So they note
    // it behind the places first, and that workgroup looks there after it has cleared: of the two one is seen, whichever came first.
    const bool clears = own_buffers && b.clear_status && unit == 0 && pc == 0;
    const int first_at = !own_buffers ? unit * W : clears ? kXGaveUp : 0, looks = min(b.spin_limit, 1 << 20);
    u64 own, up;
    bool there = true;
    for (int n = 1;; ++n) {
      own = place(unit * W + i);
      up = place((has_upper ? unit + 1 : unit) * W + i);
      const u64 first = place(first_at);
      bool waits = missing_place(own) || missing_place(up) || (!clears && missing_place(first));
      for (int k = 0; k < count; k += 64) waits = missing_place(place(from + min(k + lane, count - 1))) || waits;
      waits = __builtin_amdgcn_ballot_w64(waits) != 0;
      if ((waits && n >= looks) || (clears && !missing_place(first))) {
        __hip_atomic_store(b.place + kXGaveUp, b.launch << 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __hip_atomic_store(b.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        there = false;
        break;
      }
      if (!waits) break;
      __builtin_amdgcn_s_sleep(4);
    }
    int seen = 0;   // (a workgroup that has given up publishes and stores nothing: it takes the loop that asks whether it may)
    if (there) {
      seen = 4;
      if (__builtin_amdgcn_ballot_w64((int)(own & 0xff) != xcc) == 0) seen |= 1;
      if (!has_upper || __builtin_amdgcn_ballot_w64((int)(up & 0xff) != xcc) == 0) seen |= 2;
    }
    places_seen = seen;
  }
  __syncthreads();
  const int seen = __builtin_amdgcn_readfirstlane(places_seen);
  bool alive = (seen & 4) != 0;
  const bool team_here = (seen & 1) != 0, upper_here = (seen & 2) != 0;
  const bool keep_c = d == 1 && s + a.slices >= nrb && !a.ragged;   // one row block: its c stays here
  // Teams that wait for one row block each have a loop with as few stores as their place allows (`lean`): every store
  // instruction of a wave is time on its way round.
  const bool lean = !MANY && keep_c && team_here;
  // a dilated recurrence reads its own h from `hand` too
  const bool own_by_ring = d == 1;
  const bool uses_hand = has_upper || !own_by_ring;
  const bool hand_plain = __builtin_amdgcn_readfirstlane(upper_here && (own_by_ring || team_here)) != 0;
  constexpr int ES = HALF ? 2 : 4;
  constexpr int BLOCK = ROWS * H * ES;         // bytes of a row block of xs, hsss, csss
  const int tiles_t = nrb * TILE;              // bytes of a time step of `hand`
  const int rows_t = B * H * ES;               // bytes of a time step of xs, hsss, csss

  // byte offsets of this lane within a tile
  const unsigned put = HALF ? (my_unit / 8) * (ROWS * 16) + m * 16 + (my_unit % 8) * 2 : (my_unit / 4) * (ROWS * 16) + m * 16 + (my_unit % 4) * 4;
  const int kq = ROLES ? 32 * (wave & 1) : wave * (H / 4);   // first k of this wave's share
  const unsigned get = HALF ? (kq / 8 + kg) * (ROWS * 16) + m * 16 : (kq / 4 + 2 * kg) * (ROWS * 16) + m * 16;
  const bool do_x = !ROLES || wave < 2, do_h = !ROLES || wave >= 2;

  // All memory operations of the loop go through the buffer descriptors of this layer's arrays with a scalar offset that
  // says where in the layer: no 64-bit addresses, and what must not happen (rows past the batch, nothing to store) is
  // out of a descriptor's bounds instead of behind a branch.  Loads and stores complete in order on one
  // counter; with the same number of operations on every path the compiler waits for exactly what it needs.
  auto buffer = [](const void* p, size_t bytes) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (unsigned)bytes, 0x00020000);
  };
  const size_t hand_bytes = (size_t)T * tiles_t, out_bytes = (size_t)T * rows_t, ring_bytes = (size_t)nrb * kXRing * TILE;
  const auto hand_l = buffer(a.hand + (l + 1) * hand_bytes, hand_bytes);
  const auto below_l = buffer(a.hand + l * hand_bytes, hand_bytes);   // the layer below, or the input rows
  const int ratio_steps = (T + 1) & ~1;
  const auto ratios = buffer(a.xratio, (size_t)ratio_steps * nrb * ROWS * sizeof(float));
  const auto own_l = own_by_ring ? buffer(a.ring + l * ring_bytes, ring_bytes) : hand_l;
  const auto h_out = buffer(reinterpret_cast<unsigned char*>(a.hsss) + l * out_bytes, out_bytes);
  const auto c_out = buffer(reinterpret_cast<unsigned char*>(a.csss) + l * out_bytes, out_bytes);
  typedef decltype(buffer(nullptr, 0)) desc;

  typedef v4u share[NL];
  constexpr std::integral_constant<int, kAgentScope> fresh{};
  constexpr std::integral_constant<int, 0> cached{};
  // what k step i needs of a share; at: the tile's scalar offset, lane_at: this lane's offset in it (or out of bounds)
  auto load_piece = [&](auto ic, desc rs, unsigned lane_at, int at, share& v, auto policy_c) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value, policy = decltype(policy_c)::value;
    constexpr int step = KW / (HALF ? 8 : 4) * (ROWS * 16);   // bytes of a k step: 1024 or 2048
    if constexpr (HALF) {
      v[i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_at, at + i * step, policy));
    } else {
      v[2 * i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_at, at + i * step, policy));
      v[2 * i + 1] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rs, lane_at + ROWS * 16, at + i * step, policy));
    }
  };
  auto load_share = [&](desc rs, unsigned lane_at, int at, share& v, auto policy_c) __attribute__((always_inline)) {
    static_for<XS>([&](auto ic) __attribute__((always_inline)) { load_piece(ic, rs, lane_at, at, v, policy_c); });
  };
  auto missing = [&](const share& v) __attribute__((always_inline)) -> bool {
    if constexpr (HALF) {
      v2us mx = {0, 0};
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const unsigned w = v[i][c];
          mx = __builtin_elementwise_max(mx, __builtin_bit_cast(v2us, w));
        }
      return __builtin_amdgcn_ballot_w64(mx[0] == 0xffff || mx[1] == 0xffff) != 0;
    } else {
      unsigned mx = 0;
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) mx = max(mx, v[i][c]);
      return __builtin_amdgcn_ballot_w64(mx == ~0u) != 0;
    }
  };
  auto wait_share = [&](desc rs, int at, share& v) __attribute__((always_inline)) {
    if (!missing(v) || !alive) return;
    int n = 0;
    do {
      if (++n >= a.spin_limit) {
        __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        alive = false;
        return;
      }
      if ((n & 1023) == 0 && __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
        alive = false;
        return;
      }
      asm volatile("" ::: "memory");   // the words change under us
      load_share(rs, get, at, v, fresh);
    } while (missing(v));
  };

  // The sums.  fp32 data, blocks of 16 rows: the products with a remainder have sums of their own (cross), added at the end;
  // every addition rounds, and two thirds of them are of terms 2^-11 the size.  It also makes eight chains of the matrix
  // instructions, which with four wait for each other (19.9 instead of 16 cycles each).
  // Blocks of 32 rows have no registers for that.  Up to H 256 all of a share's products with a remainder go in front of the others,
  // while the sum is small (the x half) or half of what it will be (the h half): the error of h and c against float64 is 4 to 8 % less
  // than in the order of the k steps (H 256 L 32 T 64 B 250 rms of c 1.66e-7, 1.77e-7; L 6 T 64 B 100 dilated 1.89e-7, 2.04e-7) and no
  // larger than with the two chains of the persistent kernel's serial schedule; the time is the same (2259 us at L 32 T 64 B 250).  At H 512 it
  // takes a tenth more (L 8 T 100 B 64 725 -> 796 us): there the products stay in the order of the k steps.
  constexpr bool TWO = !HALF && !MANY;
  constexpr bool RESTS_FIRST = !HALF && MANY && H <= 256;
  accum acc[NT], cross[TWO ? NT : 1];
  auto multiply = [](v8h w, v8h x, accum c) __attribute__((always_inline)) -> accum {
    if constexpr (RT == 1) return __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, c, 0, 0, 0);
  };
  // products of resident k step w with the fragment (top, rest); first: the sums start here
  auto products = [&](auto wc, v8h top, v8h rest, auto first_c) __attribute__((always_inline)) {
    constexpr int w = decltype(wc)::value;
    constexpr bool first = decltype(first_c)::value;
    accum zero;
#pragma unroll
    for (int r = 0; r < AR; ++r) zero[r] = 0.0f;
    if constexpr (TWO) {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
        acc[tt] = multiply(wt[w][tt], top, first ? zero : acc[tt]);
        cross[tt] = multiply(wt[w][tt], rest, first ? zero : cross[tt]);
      }
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) cross[tt] = multiply(wo[w][tt], top, cross[tt]);
    } else {
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[tt] = multiply(wt[w][tt], top, first ? zero : acc[tt]);
      if constexpr (!HALF && !RESTS_FIRST) {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt] = multiply(wt[w][tt], rest, acc[tt]);
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) acc[tt] = multiply(wo[w][tt], top, acc[tt]);
      }
    }
  };
  // the two products with a remainder alone (RESTS_FIRST)
  auto rest_products = [&](auto wc, v8h top, v8h rest, auto first_c) __attribute__((always_inline)) {
    constexpr int w = decltype(wc)::value;
    accum zero;
#pragma unroll
    for (int r = 0; r < AR; ++r) zero[r] = 0.0f;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) acc[tt] = multiply(wt[w][tt], rest, decltype(first_c)::value ? zero : acc[tt]);
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) acc[tt] = multiply(wo[w][tt], top, acc[tt]);
  };
  // all of a share of an exchange tile; base: the first resident k step.  each(i): called when v's part for k step i has
  // been used, for memory operations that are due then
  auto share_products = [&](share& v, auto base_c, auto first_c, auto each) __attribute__((always_inline)) {
    constexpr int base = decltype(base_c)::value;
    constexpr bool first = decltype(first_c)::value;
    auto top_of = [&](int i) __attribute__((always_inline)) {
      const v4u p = v[2 * i], q = v[2 * i + 1];
      const v4u top = {__builtin_amdgcn_perm(p[1], p[0], 0x05040100), __builtin_amdgcn_perm(p[3], p[2], 0x05040100),
                       __builtin_amdgcn_perm(q[1], q[0], 0x05040100), __builtin_amdgcn_perm(q[3], q[2], 0x05040100)};
      return __builtin_bit_cast(v8h, top);
    };
    auto rest_of = [&](int i) __attribute__((always_inline)) {
      const v4u p = v[2 * i], q = v[2 * i + 1];
      const v4u rest = {__builtin_amdgcn_perm(p[1], p[0], 0x07060302), __builtin_amdgcn_perm(p[3], p[2], 0x07060302),
                        __builtin_amdgcn_perm(q[1], q[0], 0x07060302), __builtin_amdgcn_perm(q[3], q[2], 0x07060302)};
      return __builtin_bit_cast(v8h, rest);
    };
    if constexpr (RESTS_FIRST) {
      static_for<XS>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        rest_products(std::integral_constant<int, base + i>{}, top_of(i), rest_of(i), std::integral_constant<bool, first && i == 0>{});
        __builtin_amdgcn_sched_barrier(0x6);
      });
    }
    static_for<XS>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      constexpr std::integral_constant<bool, first && i == 0 && !RESTS_FIRST> start{};
      if constexpr (HALF) {
        products(std::integral_constant<int, base + i>{}, __builtin_bit_cast(v8h, v[i]), v8h{}, start);
        each(ic);
        __builtin_amdgcn_sched_barrier(0x6);   // vector and scalar instructions may pass, the loads stay between the products
      } else {
        const v8h top = top_of(i), rest = rest_of(i);
        each(ic);
        __builtin_amdgcn_sched_barrier(0x6);   // vector and scalar instructions may pass, the loads stay between the products
        products(std::integral_constant<int, base + i>{}, top, rest, start);
      }
    });
  };

  // U words (fp16 data: halves) to a tile of the exchange buffers, as a plain or a write-through store: both are issued,
  // one of them out of bounds (on == false: both)
  constexpr int WORD_BYTES = U * (HALF ? 2 : 4);
  auto store_bytes = [](auto policy_c, auto w, desc rs, unsigned off, int at) __attribute__((always_inline)) {
    constexpr int policy = decltype(policy_c)::value;
    if constexpr (sizeof(w) == 2) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, w), rs, off, at, policy);
    else if constexpr (sizeof(w) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w), rs, off, at, policy);
    else if constexpr (sizeof(w) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, w), rs, off, at, policy);
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, w), rs, off, at, policy);
  };
  struct words {
    typename std::conditional<HALF, unsigned short, unsigned>::type v[U];
  };
  static_assert(sizeof(words) == WORD_BYTES, "a lane's words are stored at once");
  words all_ones;
#pragma unroll
  for (int u = 0; u < U; ++u) all_ones.v[u] = (decltype(all_ones.v[0] + 0))~0u;
  auto put_words = [&](auto way_c, desc rs, int at, words w, bool plain, bool on) __attribute__((always_inline)) {
    constexpr int WAY = decltype(way_c)::value;
    if constexpr (WAY != kThrough) store_bytes(cached, w, rs, on && (WAY == kPlain || plain) ? put : ~0u, at);
    if constexpr (WAY != kPlain) store_bytes(fresh, w, rs, on && (WAY == kThrough || !plain) ? put : ~0u, at);
  };
  // the lane's values of a row of hsss or csss
  struct values {
    Value v[U];
  };
  auto put_row = [&](desc rs, unsigned off, int at, const float (&x)[U]) __attribute__((always_inline)) {
    values w;
#pragma unroll
    for (int u = 0; u < U; ++u) w.v[u] = x[u];
    store_bytes(cached, w, rs, off, at);
  };
  // h and c of an item, and the words of later steps it sets back: stored when the next item has asked for its h, so
  // that nothing the chain waits for is behind them
  struct Later {
    int row = 0, hand = 0, ring = 0;   // scalar offsets
    unsigned row_off = ~0u;
    float hv[U] = {}, cv[U] = {};
    bool on_hand = false, on_ring = false;
  } later;
  auto store_later = [&](auto way_c) __attribute__((always_inline)) {
    put_row(h_out, later.row_off, later.row, later.hv);
    put_row(c_out, later.row_off, later.row, later.cv);
    put_words(way_c, hand_l, later.hand, all_ones, hand_plain, later.on_hand);
    put_words(std::integral_constant<int, decltype(way_c)::value == kAnyWay ? kAnyWay : kPlain>{}, own_l, later.ring, all_ones, team_here, later.on_ring);
  };

  // ---- items.  An item's place: time step, row block, and the byte offsets of its time step
  struct Item {
    int t, rb;
    int tile, row;   // of time step t: in a layer of `hand`, in a layer of xs / hsss / csss
  };
  auto after = [&](Item it) __attribute__((always_inline)) -> Item {   // it.t == T: no further item
    do {
      it.rb += a.slices;
      if (!MANY || it.rb >= nrb) {
        it.rb = s;
        ++it.t;
        it.tile += tiles_t;
        it.row += rows_t;
      }
    } while (a.ragged && it.t < T && it.t >= a.steps_of[it.rb]);
    return it;
  };
  auto h_at = [&](const Item& it) __attribute__((always_inline)) -> int {
    return own_by_ring ? (it.rb * kXRing + ((it.t - 1) & (kXRing - 1))) * TILE : it.tile - d * tiles_t + it.rb * TILE;
  };
  auto row_off_of = [&](int rb) { return rb * ROWS + m < B ? (unsigned)((m * H + my_unit) * ES) : ~0u; };
  float cp[U] = {};   // c of d steps before
  values raw_cp = {};  // the same as it was loaded: converted at once it would have to be there at once
  float xr = 1.0f;
  share v;
  auto ask_c = [&](unsigned off, int at) __attribute__((always_inline)) {
    values v;
    if constexpr (sizeof(values) == 2) v = __builtin_bit_cast(values, __builtin_amdgcn_raw_buffer_load_b16(c_out, off, at, 0));
    else if constexpr (sizeof(values) == 4) v = __builtin_bit_cast(values, __builtin_amdgcn_raw_buffer_load_b32(c_out, off, at, 0));
    else if constexpr (sizeof(values) == 8) v = __builtin_bit_cast(values, __builtin_amdgcn_raw_buffer_load_b64(c_out, off, at, 0));
    else v = __builtin_bit_cast(values, __builtin_amdgcn_raw_buffer_load_b128(c_out, off, at, 0));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (HALF) raw_cp.v[u] = v.v[u];
      else cp[u] = v.v[u];
    }
  };

  bool small_reported = false;
  // four neighbouring units of a row that are all small and not all zero: those of lanes m, m + ROWS, ...
  auto look_for_small = [&](const float (&h)[U]) __attribute__((always_inline)) {
    if constexpr (!HALF) {
      unsigned largest = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) largest = max(largest, __float_as_uint(h[u]) & 0x7fffffffu);
      const u64 sm = __builtin_amdgcn_ballot_w64(largest < kXSmallBits);
      if (__builtin_expect(sm != 0 && !small_reported && alive, 0)) {
        u64 all = sm, any = __builtin_amdgcn_ballot_w64(largest != 0);
        if (U < 4) {
          all &= all >> 32;
          any |= any >> 32;
        }
        if (U < 2) {
          all &= all >> 16;
          any |= any >> 16;
        }
        if (U < 4) all &= U == 1 ? 0xffffull : 0xffffffffull;
        if ((all & any) != 0) {
          small_reported = true;
          if (lane == 0) __hip_atomic_store(a.status + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
  };
  // this wave's sums, to LDS; all four waves' sums of the units it updates, from LDS
  auto give_sums = [&](int parity) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      constexpr int per = 4 * U;   // of a tile's registers: all, or (CT == 1 and 32 rows) the half of a wave
      sums v;
#pragma unroll
      for (int r = 0; r < per; ++r) v[r] = TWO ? acc[w % NT][r % AR] + cross[w % (TWO ? NT : 1)][r % AR] : per == AR ? acc[w % NT][r] : acc[w / 2 % NT][(w % 2) * per % AR + r];
      red[parity][w][wave][lane] = v;
    }
  };
  auto take_sums = [&](int parity) __attribute__((always_inline)) -> sums {
    // (16-row results: unit 4 wave + kg is in tile kg, at the lanes of k group `wave`)
    const int tile = RT == 1 ? kg : wave, at = RT == 1 ? 16 * wave + m : lane;
    sums pre = red[parity][tile][0][at] + red[parity][tile][1][at];
    pre += red[parity][tile][2][at] + red[parity][tile][3][at];
    return pre;
  };
  // the state update of this lane's units and their words of the exchange buffers
  auto update = [&](sums pre, const float (&c_prev)[U], float (&c)[U], float (&h)[U]) __attribute__((always_inline)) -> words {
    auto gate = [](float e) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(e)); };
    words w;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float p[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if constexpr (HALF) p[g] = pre[4 * u + g] * (g == 3 ? 1.0f : -kLog2e) + ebias[4 * u + g];
        else p[g] = pre[4 * u + g] * esc[4 * u + g] + ebias[4 * u + g];
      }
      c[u] = __builtin_fmaf(gate(p[1]), c_prev[u], gate(p[0]) * tanh_f(p[3]));
      h[u] = gate(p[2]) * tanh_f(c[u]);
      // rounded to 32 bits before 16 in every loop: one instruction may do both, with another last bit now and then, and
      // a ragged batch, which takes another loop than a dense one, gives the same bits (with row blocks of either kind: the sums
      // of the two matrix instructions are the same)
      if constexpr (HALF) asm("" : "+v"(c[u]), "+v"(h[u]));
      unsigned word;
      if constexpr (HALF) {
        c[u] = (float)(_Float16)c[u];
        word = __builtin_bit_cast(unsigned short, (_Float16)h[u]);
        if (word == 0xffffu) word = 0x7e00u;   // a NaN, but not the one that stands for "not there yet"
      } else {
        const float v = h[u] * (float)(1 << kXHandTop);
        const _Float16 top = (_Float16)v;
        const v2h pair = {top, (_Float16)(v - (float)top)};
        word = __builtin_bit_cast(unsigned, pair);
        if (word == ~0u) word = 0x7e007e00u;
      }
      w.v[u] = word;
    }
    return w;
  };
  auto ring_at = [&](int rb, int t) { return (rb * kXRing + (t & (kXRing - 1))) * TILE; };
  auto later_of = [&](const Item& it, const float (&h)[U], const float (&c)[U]) __attribute__((always_inline)) {
    later.row = it.row + it.rb * BLOCK;
    later.row_off = alive ? row_off_of(it.rb) : ~0u;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      later.hv[u] = h[u];
      later.cv[u] = c[u];
    }
    later.hand = it.tile + it.rb * TILE + 2 * tiles_t;
    later.on_hand = alive && uses_hand && it.t + 2 < T;
    later.ring = ring_at(it.rb, it.t - 2);
    later.on_ring = alive && own_by_ring && it.t >= 2;
  };
  // x of an item: through the caches, because the team's other workgroups fetch the same tile into this XCD's L2.  (A
  // line that was fetched too early holds all-ones words still; wait_share asks for it again past the caches.)
  auto x_at = [&](const Item& it) { return it.tile + it.rb * TILE; };
  auto ask_ratio = [&](const Item& it) __attribute__((always_inline)) {
    xr = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ratios, m * 4, (it.rb * ratio_steps + it.t) * (ROWS * 4), 0));
  };
  auto scale_input = [&](float ratio) __attribute__((always_inline)) {
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int r = 0; r < AR; ++r) {
        acc[tt][r] *= ratio;
        if constexpr (TWO) cross[tt][r] *= ratio;
      }
  };
  constexpr std::integral_constant<int, 0> x_steps{};
  constexpr std::integral_constant<int, ROLES ? 0 : XS> h_steps{};

  // The loop.  FIRST: the layer reads the input rows.  One set of registers takes turns: while the products of an item's h
  // are formed, the pieces of the next item's x are asked for one by one into the registers that have been used (a burst
  // of loads would hold up the wave: 64 bytes a cycle is what a compute unit gets), and while those of x are formed
  // (which is after this item's h has been published) the pieces of the next h.
  // STORES_FIRST: a team too large for an XCD waits longest for its h, and what is asked for too early costs the whole way once
  // more: its stores go in front (fp16 H 1024 L 4 T 64 B 16 238 -> 184 us).  With several row blocks h is there, and with a
  // dilated recurrence sooner than the stores take (L 3 T 88 B 42 H 64 137 us with the stores in front, 121 behind).
  constexpr bool STORES_FIRST = !MANY && W > 32 * exchange_per_cu(H, HALF, MANY);
  auto walk = [&](auto first_c, auto way_c) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value;
    constexpr std::integral_constant<int, decltype(way_c)::value == kAnyWay ? kAnyWay : kPlain> own_way{};
    constexpr unsigned kOut = 0x80000000u;   // a lane offset beyond every descriptor: the load returns zeros
    // products of the x in v; the pieces of h (and c) of the same item take its place.  Where there is nothing (no step
    // that far back, or the half of the contraction another wave has) v is zeros and the products are those of zeros.
    auto take_x = [&](const Item& it) __attribute__((always_inline)) {
      const bool has_prev = it.t >= d;
      if constexpr (!FIRST) wait_share(below_l, x_at(it), v);
      ask_c(has_prev && !keep_c ? row_off_of(it.rb) : ~0u, has_prev && !keep_c ? it.row - d * rows_t + it.rb * BLOCK : 0);
      const unsigned lane_at = has_prev && do_h ? get : kOut;
      const int at = has_prev ? h_at(it) : 0;
      const float ratio = xr;
      share_products(v, x_steps, std::true_type{}, [&](auto ic) __attribute__((always_inline)) {
        load_piece(ic, own_l, lane_at, at, v, fresh);
      });
      if constexpr (FIRST && !HALF) scale_input(ratio);
    };
    int parity = 0;
    bool follows = false;   // the item before is what this one takes its c from
    Item it{0, s, 0, 0};
    if (a.ragged && a.steps_of[s] == 0) it = after(it);
    if (it.t >= T) return;
    load_share(below_l, do_x ? get : kOut, x_at(it), v, cached);
    if constexpr (FIRST && !HALF) ask_ratio(it);
    take_x(it);
    // nothing yet, but as many stores behind the loads of h as on the way round the loop: the compiler waits for the loads
    // by their number, and on the way round would wait for the stores of the item before with them
    if constexpr (!STORES_FIRST) store_later(way_c);
    while (true) {   // (a wave that has given up walks on without waiting, to every barrier the others wait at)
      const bool has_prev = it.t >= d;
      const Item next = after(it);
      const bool more = next.t < T;
      const int next_x = x_at(more ? next : it);   // there is always something to ask for: the same operations on every path
      wait_share(own_l, has_prev ? h_at(it) : 0, v);
      share_products(v, h_steps, std::false_type{}, [&](auto ic) __attribute__((always_inline)) {
        load_piece(ic, below_l, do_x ? get : kOut, next_x, v, cached);
      });
      if constexpr (FIRST && !HALF) ask_ratio(more ? next : it);
      float c_prev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) c_prev[u] = !has_prev ? 0.0f : keep_c || follows ? later.cv[u] : (HALF ? (float)raw_cp.v[u] : cp[u]);
      follows = next.rb == it.rb && next.t == it.t + d;
      give_sums(parity);
      // what the item before stored is complete before anything of this one is published: only what was asked for since
      // may be outstanding
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL + (FIRST && !HALF ? 1 : 0)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const sums pre = take_sums(parity);
      parity ^= 1;
      float c[U], h[U];
      const words word = update(pre, c_prev, c, h);
      put_words(own_way, own_l, ring_at(it.rb, it.t), word, team_here, alive && own_by_ring);
      put_words(way_c, hand_l, x_at(it), word, hand_plain, alive && uses_hand);
      asm volatile("" ::: "memory");
      later_of(it, h, c);
      look_for_small(h);
      if (!more) break;
      if constexpr (STORES_FIRST) store_later(way_c);
      asm volatile("" ::: "memory");
      take_x(next);
      asm volatile("" ::: "memory");
      if constexpr (!STORES_FIRST) store_later(way_c);
      asm volatile("" ::: "memory");
      it = next;
    }
    store_later(way_c);
  };
  // The loop of a team that has one row block, whose h every step waits for: a wave issues an instruction in four or five
  // cycles at best, so what is not needed is left out of it (the loop above has ten stores an item and forty instructions
  // more for the places of items).  The words go to the ring and to `hand`, and instead of store_later's every wave makes
  // one store of 16 bytes a lane: wave 0 the h of the item before, wave 1 its c (both from LDS, where they are since the
  // last barrier), wave 2 sets back the words of this workgroup's units in the ring, wave 3 those in `hand`.  (With `hand`
  // for the own layer too, and no ring, a step took 0.1 us more: its lines are new to L2.)
  // T 64 B 16 in us, the loop above -> this one, one layer / eight: fp32 H 64 79 -> 62 / 107 -> 94, 128 83 -> 65 / 113 -> 99,
  // 256 103 -> 87 / 135 -> 116, 512 160 -> 142 / 196 -> 175; fp16 H 256 79 -> 58 / 105 -> 100, 512 106 -> 78 / 141 -> 118.
  // PLAIN: the layer above is on this XCD, or there is none.
  auto walk_lean = [&](auto first_c, auto plain_c, auto early_c) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value, PLAIN = decltype(plain_c)::value, EARLY = decltype(early_c)::value;
    constexpr std::integral_constant<int, PLAIN ? 0 : kAgentScope> up_policy{};
    constexpr int step = TILE, wrap = kXRing * TILE - 1;
    const int words_at = s * kXRing * TILE;
    int words = 0;           // of this item in the ring: words_at + words
    int x_at = s * TILE;     // this item's place in `hand` and in the layer below
    // this wave's store: the next one goes to share_base + share_at, which moves on by share_step within share_wrap
    const desc share_l = wave == 0 ? h_out : wave == 1 ? c_out : wave == 2 ? own_l : hand_l;
    const int share_base = wave == 2 ? words_at : 0;
    const int share_step = wave < 2 ? rows_t : wave == 2 ? step : tiles_t, share_wrap = wave == 2 ? wrap : ~0;
    int share_at = wave < 2 ? s * BLOCK - rows_t : wave == 2 ? 2 * step : 2 * tiles_t + s * TILE;
    const int share_row = HALF ? lane >> 1 : lane >> 2, share_part = HALF ? lane & 1 : lane & 3;   // 16 bytes of a row of 16 units
    unsigned share_put = ~0u;
    if (wave < 2 ? share_row < 16 && s * 16 + share_row < B : (wave == 2 || has_upper) && (!HALF || lane < 32))
      share_put = wave < 2 ? (unsigned)((share_row * H + UNITS * pc) * ES + share_part * 16) : (unsigned)(UNITS * pc * 16 * ES + lane * 16);
    unsigned share_next = ~0u;   // where the next one goes
    unsigned my_put = put, up_put = has_upper ? put : ~0u;
    const Value* const share_from = &outs[0][wave & 1][(share_row & 15) * OUT_ROW + share_part * (HALF ? 8 : 4)];
    Value* const share_to = &outs[0][0][m * OUT_ROW + 4 * wave + kg];
    constexpr int OUT_BUF = 2 * 16 * OUT_ROW;
    auto store_share = [&](int parity) __attribute__((always_inline)) {
      v4u w = {~0u, ~0u, ~0u, ~0u};
      if (wave < 2) w = *reinterpret_cast<const v4u*>(share_from + parity * OUT_BUF);
      store_bytes(cached, w, share_l, PLAIN || wave < 3 ? share_next : ~0u, share_base + share_at);
      if constexpr (!PLAIN) store_bytes(fresh, w, share_l, wave < 3 ? ~0u : share_next, share_base + share_at);
      share_at = (share_at + share_step) & share_wrap;
      share_next = share_put;
    };
    auto wait_for = [&](desc rs, int at, share& v) __attribute__((always_inline)) {
      if (__builtin_expect(missing(v), 0)) {
        wait_share(rs, at, v);
        if (!alive) my_put = up_put = share_put = share_next = ~0u;
      }
    };
    load_share(below_l, do_x ? get : 0x80000000u, x_at, v, cached);
    if constexpr (FIRST && !HALF) xr = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ratios, m * 4, s * ratio_steps * (ROWS * 4), 0));
    // h is asked for in front of the products of x, where registers and its way leave time for it, and behind them: what comes
    // too early is not there yet, and to ask again only then costs the whole way once more.  (L 1 T 64 B 16: H 128
    // 69 us when asked for behind x only, 65 with both; L 20 T 30 B 32 H 128 83 and 81.6; fp16 H 512 88 and 78.)  The first time it is asked
    // for when it is about to be there.  Where no h goes to another XCD (EARLY: a single layer, or fp32 stacks whose row slices have an XCD each or share
    // one) steps are short and every cycle in front of it costs, but for fp16 teams that share an XCD; elsewhere the layer whose h comes from
    // another XCD sets the pace, and it is some 320 cycles into the step (fp16 512), at H 64 with three teams or more to an XCD 192.
    // (us with 0, 2, 4, 5, 6 and 8 times 64 cycles, EARLY: H 128 L 2 T 100 B 233 102.7, 106.5, 113.5, 113.5, 115.7, 120.9; H 64 L 5 T 86 B 108 90.1, 93.2, 97.9, 100.3,
    // 102.2, 107.0; a single fp16 layer with 0, 1, 2: T 64 B 32 H 256 54.9, 55.9, 57.5, B 200 63.3, 63.2, 60.2.  Elsewhere with 2, 4, 5, 6, 8: L 6 T 80 B 16 H 128 106.1, 101.6,
    // 100.5, 101.2, 104.5; L 5 T 60 B 60 H 64 79.7, 78.3, 78.0, 78.2, 79.5; fp16 L 4 T 60 B 32 H 256 81.9, 80.1, 79.1, 77.5, 74.9, with 10 and 15 75.5, 83.4;
    // fp16 L 2 T 60 B 33 H 512 with 6, 8, 10 90.2, 88.9, 91.3; H 64 with 3, 4, 5, 6 L 20 T 60 B 20 96.6, 97.7, 99.4,
    // 101.4, L 9 T 77 B 18 98.6, 99.2, 100.4, 101.2, and with two teams to an XCD L 4 T 82 B 35 99.1, 98.4, 98.1, 98.5.  At H 256 fp32, where it is
    // asked for behind x only, any delay costs: L 4 T 60 B 16 93.2 without, 93.7 with 2, 95.7 with 4.)
    constexpr bool TWICE = HALF ? H <= 512 : H <= 128;
    int xcd_teams = 0;
    if constexpr (TWICE) {
      xcd_teams = __builtin_amdgcn_readfirstlane(a.per_xcd);
      asm volatile("" : "+s"(xcd_teams));   // kept: left to itself the compiler reads the argument again in every step
    }
    const bool crowded = xcd_teams >= (HALF ? 2 : 3);
    share vh;
    float c[U] = {}, h[U];
    const unsigned x_get = do_x ? get : 0x80000000u, h_get = do_h ? get : 0x80000000u;   // out of bounds: zeros
    int parity = 0;
    // Nothing to store yet, but as many stores behind the loads of x as on the way round the loop: the compiler waits for
    // the loads by their number, and on the way round would wait for the stores with them.
    asm volatile("" ::: "memory");
    static_for<PLAIN ? 3 : 4>([&](auto ic) __attribute__((always_inline)) {   // (two that are the same would become one)
      store_bytes(cached, all_ones, own_l, ~0u, 64 * decltype(ic)::value);
    });
    if (wave >= 2) share_next = share_put;   // waves 0 and 1 have nothing at their first turn: there is no item before
    for (int t = 0;; ++t) {
      const bool more = t + 1 < T;
      const int next_x = more ? x_at + tiles_t : x_at, before = words_at + ((words - step) & wrap);
      const unsigned h_get_t = t > 0 ? h_get : 0x80000000u;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (TWICE) {
        if constexpr (!EARLY) {
          if (HALF && FIRST && !has_upper) {
            if (crowded) __builtin_amdgcn_s_sleep(2);   // 64 cycles each
          } else if (H == 64 && crowded) {
            __builtin_amdgcn_s_sleep(3);
          } else {
            __builtin_amdgcn_s_sleep(HALF ? 8 : 5);
          }
        }
        load_share(own_l, h_get_t, before, vh, fresh);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!FIRST) wait_for(below_l, x_at, v);
      share_products(v, x_steps, std::true_type{}, [](auto) __attribute__((always_inline)) {});
      if constexpr (FIRST && !HALF) scale_input(xr);
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {   // (left to itself the compiler moves the scaling behind the wait for h)
        asm volatile("" : "+v"(acc[tt]));
        if constexpr (TWO) asm volatile("" : "+v"(cross[tt]));
      }
      __builtin_amdgcn_sched_barrier(0);
      load_share(own_l, h_get_t, before, v, fresh);
      __builtin_amdgcn_sched_barrier(0);
      share& h_words = TWICE ? vh : v;
      if constexpr (TWICE) {
        if (__builtin_expect(missing(vh), 0)) {
          wait_for(own_l, before, v);
#pragma unroll
          for (int i = 0; i < NL; ++i) vh[i] = v[i];
        }
      } else {
        wait_for(own_l, before, v);
      }
      share_products(h_words, h_steps, std::false_type{}, [&](auto ic) __attribute__((always_inline)) {
        load_piece(ic, below_l, x_get, next_x, v, cached);
      });
      if constexpr (FIRST && !HALF)
        xr = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ratios, m * 4, (s * ratio_steps + (more ? t + 1 : t)) * (ROWS * 4), 0));
      give_sums(parity);
      // what was set back after the item before is complete before anything of this one is published
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NL + (FIRST && !HALF ? 1 : 0)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const sums pre = take_sums(parity);
      float c_prev[U];
#pragma unroll
      for (int u = 0; u < U; ++u) c_prev[u] = c[u];
      const struct words word = update(pre, c_prev, c, h);
      store_bytes(cached, word, own_l, my_put, words_at + words);
      store_bytes(up_policy, word, hand_l, up_put, x_at);
      share_to[parity * OUT_BUF] = (Value)h[0];
      share_to[parity * OUT_BUF + 16 * OUT_ROW] = (Value)c[0];
      asm volatile("" ::: "memory");
      look_for_small(h);
      parity ^= 1;
      if (t + 2 >= T && wave == 3) share_put = share_next = ~0u;
      store_share(parity);
      if (!more) break;
      asm volatile("" ::: "memory");
      x_at = next_x;
      words = (words + step) & wrap;
    }
    __syncthreads();   // h and c of the last item
    if (wave < 2) store_share(parity ^ 1);
  };
  if constexpr (!MANY) {
    if (lean) {
      constexpr std::true_type yes{};
      constexpr std::false_type no{};
      if constexpr (!HALF && H <= 128) {
        if (hand_plain && again->early) {
          if (l == 0) walk_lean(yes, yes, yes);
          else walk_lean(no, yes, yes);
          return;
        }
      }
      if (l == 0 && hand_plain) walk_lean(yes, yes, no);
      else if (l == 0) walk_lean(yes, no, no);
      else if (hand_plain) walk_lean(no, yes, no);
      else walk_lean(no, no, no);
      return;
    }
  }
  auto walk_layer = [&](auto way_c) __attribute__((always_inline)) {
    if (l == 0) walk(std::true_type{}, way_c);
    else walk(std::false_type{}, way_c);
  };
  // One store instead of two wherever a team sits on one XCD (L 8 T 100 B 64 H 512 747 -> 732 us; fp32 at H 256 has no
  // register left: with three copies of the loop it spills in the loop, 1070 -> 1190 us at L 16 T 114 B 104).
  if constexpr (MANY && (HALF || CT == 1)) {
    if (team_here && hand_plain) return walk_layer(std::integral_constant<int, kPlain>{});
    if (team_here && own_by_ring) return walk_layer(std::integral_constant<int, kThrough>{});
  }
  walk_layer(std::integral_constant<int, kAnyWay>{});
}

// In front of the kernel above where it does not lay out its buffers itself (run_exchange), by workgroup: the input rows as tiles (the first row_groups of them; one wave per row, rows past
// the batch are zeros; fp32 rows are cut under a power-of-two scale of their own), then the ring and the first two steps of
// `hand`, kPrepareFill words of 16 bytes of a layer to a workgroup; the first of these has the status block and the places too.
// (A grid of rows x (layers + 1), most of whose workgroups had nothing to do, took longer with many of them only: us under the tracer, that
// grid and this, L 8 T 100 B 64 H 512, 9216 workgroups, 14.8, 12.3; L 20 T 30 B 32 H 128, 5040, 5.1, 5.1, the whole call 79.8, 78.7.)
constexpr int kPrepareFill = 1024;
template <bool HALF>
__global__ __launch_bounds__(256) void lstm_exchange_prepare_kernel(int* status, int first_word, unsigned long long* place, int nplaces, v4u* ring,
                                                                    unsigned ring_per_layer, v4u* hand, size_t hand_per_layer,
                                                                    unsigned hand_first, const void* xs, float* xratio, int row_groups,
                                                                    int T, int B, int nrb, int block, int H) {
  if ((int)blockIdx.x >= row_groups) {
    const int g = (int)blockIdx.x - row_groups;
    const unsigned of_layer = ring_per_layer + hand_first, groups = (of_layer + kPrepareFill - 1) / kPrepareFill;
    const unsigned l = (unsigned)g / groups, first = ((unsigned)g - l * groups) * kPrepareFill + threadIdx.x;
    const v4u ones = {~0u, ~0u, ~0u, ~0u};
    v4u* const ring_l = ring + (size_t)l * ring_per_layer;
    v4u* const hand_l = hand + (size_t)(l + 1) * hand_per_layer;
#pragma unroll
    for (int n = 0; n < kPrepareFill / 256; ++n) {
      const unsigned i = first + 256 * n;
      if (i < of_layer) *(i < ring_per_layer ? ring_l + i : hand_l + (i - ring_per_layer)) = ones;
    }
    if (g == 0) {
      for (int i = threadIdx.x; i < nplaces; i += 256) place[i] = 0;
      if (threadIdx.x < kStatusBytes / sizeof(int) && (int)threadIdx.x >= first_word) status[threadIdx.x] = 0;
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const int per_step = nrb * block, rows = T * per_step;   // block: rows of a row block
  for (int r = blockIdx.x * 4 + (threadIdx.x >> 6); r < rows; r += row_groups * 4) {
    const int t = r / per_step, b = r - t * per_step;
    unsigned char* dst = reinterpret_cast<unsigned char*>(hand) + (size_t)(r / block) * exchange_tile_bytes(H, HALF, block) + (r % block) * 16;
    const size_t src = ((size_t)t * B + b) * H;
    if constexpr (HALF) {
      for (int k = 8 * lane; k < H; k += 512) {
        v4u v = {0, 0, 0, 0};
        if (b < B) v = *reinterpret_cast<const v4u*>(reinterpret_cast<const _Float16*>(xs) + src + k);
        *reinterpret_cast<v4u*>(dst + (k >> 3) * (block * 16)) = v;
      }
    } else {
      v4f x[4];   // H <= 1024
      float mx = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 4 * lane + 256 * i;
        x[i] = v4f{0.f, 0.f, 0.f, 0.f};
        if (k < H && b < B) x[i] = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(xs) + src + k);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(x[i][0]), fabsf(x[i][1])), fmaxf(fabsf(x[i][2]), fabsf(x[i][3]))));
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
      const int eb = min(max((int)((__float_as_uint(mx) >> 23) & 0xff), 15), 254);
      const float scale = __uint_as_float((unsigned)(127 + 14 + 127 - eb) << 23);   // the row's largest -> [2^14, 2^15)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 4 * lane + 256 * i;
        v4u w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = x[i][e] * scale;
          const _Float16 top = (_Float16)v;
          const v2h pair = {top, (_Float16)(v - (float)top)};
          w[e] = __builtin_bit_cast(unsigned, pair);
        }
        if (k < H) *reinterpret_cast<v4u*>(dst + (k >> 2) * (block * 16)) = w;
      }
      // the products carry 2^(141 - eb), h's 2^14
      if (lane == 0) xratio[((size_t)(b / block) * ((T + 1) & ~1) + t) * block + b % block] = __uint_as_float((unsigned)eb << 23);
    }
  }
}

namespace {

struct ExchangeFlavour {
  const void* one;    // row blocks of 16 rows, one per workgroup
  const void* many;   // row blocks of 32 rows
};

template <int H, bool HALF>
ExchangeFlavour exchange_flavour() {
  return {(const void*)lstm_exchange_kernel<H, HALF, false>, (const void*)lstm_exchange_kernel<H, HALF, true>};
}

// The kernel for a hidden size and element type, or nulls.
ExchangeFlavour exchange_flavour_of(int H, bool half) {
  if (half) {
    switch (H) {
      case 256: return exchange_flavour<256, true>();
      case 512: return exchange_flavour<512, true>();
      case 1024: return exchange_flavour<1024, true>();
      default: return {nullptr, nullptr};
    }
  }
  switch (H) {
    case 64: return exchange_flavour<64, false>();
    case 128: return exchange_flavour<128, false>();
    case 256: return exchange_flavour<256, false>();
    case 512: return exchange_flavour<512, false>();
    default: return {nullptr, nullptr};
  }
}

// Workgroups the device holds at once (0 on any error).
int exchange_slots(const void* fn) {
  constexpr int kKept = 16, kDev = 16;
  static std::atomic<const void*> fns[kKept];
  static std::atomic<int> kept[kKept][kDev];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDev) return 0;
  int at = 0;
  for (; at < kKept; ++at) {
    const void* f = fns[at].load(std::memory_order_acquire);
    if (f == fn) break;
    if (!f) {
      const void* none = nullptr;
      if (fns[at].compare_exchange_strong(none, fn) || none == fn) break;
    }
  }
  if (at < kKept)
    if (const int v = kept[at][dev].load(std::memory_order_acquire)) return v;
  const DeviceProps* dp = nullptr;
  int per_cu = 0;
  if (device_props(&dp) != FTK_OK || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, 0) != hipSuccess) return 0;
  const int slots = per_cu * dp->cus;
  if (at < kKept) kept[at][dev].store(slots, std::memory_order_release);
  return slots;
}

// How a stack of L layers (as many as one launch holds) is laid out on the chip.
struct ExchangePlan {
  int layers = 0;    // layers per launch, 0: the device cannot hold one
  int slices = 0;    // row slices of a layer
  int per_xcd = 0;   // teams per XCD, 0: workgroups in order
};

// Teams of W workgroups that are on the chip at once.
int exchange_teams(int W, int slots) {
  const int here = std::min(slots, kXPlaces);
  const int room = here / 8 / W;   // teams an XCD holds
  return room ? 8 * room : here / W;   // (a team may be larger than an XCD)
}

ExchangePlan exchange_plan(int L, int W, int nrb, int slots) {   // W: workgroups of a team
  ExchangePlan p;
  const int teams = exchange_teams(W, slots);
  const bool room = teams >= 8;
  if (teams == 0) return p;
  p.layers = std::min({L, teams, kXLayers});
  p.slices = std::max(1, std::min(nrb, teams / p.layers));
  const int blocks = (nrb + p.slices - 1) / p.slices;   // the fewest slices that walk no more blocks each
  p.slices = (nrb + blocks - 1) / blocks;
  if (room) p.per_xcd = (p.layers * p.slices + 7) / 8;
  return p;
}

constexpr size_t align256(size_t v) { return (v + 255) / 256 * 256; }
constexpr size_t exchange_xratio_at = align256((kXPlaces + 1) * sizeof(unsigned long long));   // behind the places

// What the workgroups write for each other begins on a line of its own, wherever a caller's workspace begins (the status block stays at its
// start): no line is shared by workgroups that lay out different parts (exchange_lay_out), and a place is one access.
size_t exchange_places_at(const void* ws) { return align256((size_t)ws + kStatusBytes) - (size_t)ws; }

// ring and hand begin at multiples of 16 KB: tiles are 4 to 128 KB, powers of two, and steps take longer where they lie across such bounds (us
// with `hand` at 0, 256, 1024 bytes beyond one: H 64 L 5 T 94 B 31 117.8, 121.1, 118.6; H 128 L 7 T 80 B 14 108.3, 111.4, 108.7; H 256 L 4 T 105 B 44 148.2, 151.3,
// 150.8, and 150.4 with `ring` at 256; fp16 L 3 T 77 B 78 H 256 90.5, 93.4, 91.8).  Right behind the words in front of them they began at
// 256 bytes times what T and B make of it.
constexpr size_t kXTilesAt = 16384;
struct ExchangeTiles {
  size_t ring, hand, end;   // bytes from the start of the workspace
};
ExchangeTiles exchange_tiles_at(const void* ws, size_t to, size_t ring_from, size_t ring_bytes, size_t hand_bytes) {
  auto up = [&](size_t at) { return ((size_t)ws + at + to - 1) / to * to - (size_t)ws; };
  ExchangeTiles t;
  t.ring = up(ring_from);
  t.hand = up(t.ring + ring_bytes);
  t.end = t.hand + hand_bytes;
  return t;
}

}  // namespace

// Whether lstm_exchange runs this hidden size and type at all.
bool exchange_takes(int H, bool half) { return exchange_flavour_of(H, half).one != nullptr; }

namespace {
// Bytes of [places][xratio][ring][hand] for L layers, with either kind of row block and nothing between them.
size_t exchange_buffer_bytes(int L, int T, int B, int H, bool half) {
  const size_t rows = (size_t)(B + 31) / 32 * 32;   // never less than with blocks of 16
  return exchange_xratio_at + align256((size_t)(T + 1) * rows * sizeof(float)) +
         rows * H * (half ? 2 : 4) * ((size_t)L * kXRing + (size_t)(L + 1) * T);
}
}  // namespace

// Bytes of workspace for L layers: the status block, up to 255 bytes to a line, these, and up to kXTilesAt in front of ring and hand each.
size_t exchange_workspace_bytes(int L, int T, int B, int H, bool half) {
  return kStatusBytes + 256 + 2 * kXTilesAt + exchange_buffer_bytes(L, T, B, H, half);
}

// Whether a layer of a buffer stays below what a buffer descriptor and its offsets reach.
bool exchange_fits(int T, int B, int H, bool half) { return (size_t)T * ((size_t)(B + 31) / 32 * 32) * H * (half ? 2 : 4) < (1ull << 31) - (1 << 20); }

namespace {

// Layers of one launch with one block of 16 rows per workgroup (0: the device holds none).
int exchange_one_block_layers(int L, int B, int H, bool half) {
  const ExchangeFlavour f = exchange_flavour_of(H, half);
  if (!f.one) return 0;
  return std::min({L, kXLayers, exchange_teams(H / exchange_units(H, half, false), exchange_slots(f.one)) / ((B + 15) / 16)});
}

// What the launches of a stack take, in microseconds: `first` and, for each further one, `next` before the steps (weights, places, what they lay
// out, and what a deep stack's launches find less of in the caches), `layer` for every further layer of a launch until the
// pipeline of layers is full, and for a step of each row block that a workgroup walks `step` and `fill` times the workgroups per compute
// unit.  Fitted, for each hidden size, to the times of both kinds over 420 stacks of L up to 32, T 16 .. 128, B 8 .. 256 that blocks of 16
// rows take more launches for, when a kernel in front laid out their buffers; fp32 up to H 256 again, to 280 stacks of L 3 .. 32, T 16 .. 128, B 33 .. 256
// whose weights and inputs change from call to call, since launches do that themselves (the constants before held a further launch for 37
// to 54 us dearer).  Loss against the better kind, in the mean over stacks that were not fitted to, with ordinary and with cooperative launches: H 64 0 and
// 0.2 % (9 stacks), H 128 0.2 and 1.0 (24), H 256 2.4 and 0.1 (62 near the line; with 8 us more charged for a further launch 6.7 and 0.3); with the
// older constants fp32 H 512 0.1 % (27 stacks), fp16 H 256 0 (22), H 512 0 (29), H 1024 0 (6).
struct ExchangeCost {
  float step, fill, layer, first, next;
};

ExchangeCost exchange_cost(int H, bool half, bool many) {
  if (half) {
    if (H == 256) return many ? ExchangeCost{2.63f, 0.04f, 3.0f, 6.0f, 6.0f} : ExchangeCost{0.82f, 0.32f, 1.55f, 16.0f, 21.5f};
    if (H == 512) return many ? ExchangeCost{3.04f, 0.3f, 4.6f, 29.0f, 33.0f} : ExchangeCost{1.29f, 0.16f, 3.35f, 20.5f, 23.0f};
    return many ? ExchangeCost{2.96f, 0.26f, 6.05f, 41.0f, 47.0f} : ExchangeCost{1.7f, 0.76f, 5.0f, 9.0f, 38.0f};
  }
  if (H == 64) return many ? ExchangeCost{0.0f, 1.89f, 0.58f, 21.0f, 21.0f} : ExchangeCost{0.87f, 0.34f, 1.36f, 7.7f, 7.7f};
  if (H == 128) return many ? ExchangeCost{2.58f, 0.27f, 2.15f, 0.0f, 0.0f} : ExchangeCost{0.77f, 0.39f, 1.76f, 6.8f, 8.4f};
  if (H == 256) return many ? ExchangeCost{3.97f, 0.11f, 4.52f, 20.3f, 20.3f} : ExchangeCost{1.3f, 0.24f, 2.82f, 5.1f, 18.0f};
  return many ? ExchangeCost{2.86f, 0.35f, 4.1f, 35.0f, 36.0f} : ExchangeCost{1.73f, 0.24f, 4.35f, 11.5f, 34.0f};
}

// A launch is an ordinary one or, once a process uses a second stream or records graphs, a cooperative one, which takes 16 to 18 us more
// (launch_resident).  Which it is depends on what the process did before.  With fp16 data both kinds of block give the same bits
// (the sums of the two matrix instructions are the same), and a launch is charged what it is going to take.  With fp32 data they
// do not, and what a call computes must not go by that: a launch more is charged most of the difference always.  Loss against the better
// kind of each, mean over 2940 stacks near the line with ordinary launches and 1900 with cooperative ones: 0.4 and 1.5 % with nothing
// charged, 0.8 and 0.5 % with 12 us, 1.2 and 0.4 % with 17 (with the constants of a kernel in front of every launch).
constexpr float kAnyLaunch = 12.0f, kCooperativeLaunch = 17.0f;

// Layers of one launch (0: the device cannot hold one), and the kind of row block.  16 rows and one block per workgroup, whose
// step is the shorter one, wherever that takes no more launches (L 23 T 67 B 10 fp32 H 512, three launches of either kind: 820 us
// with blocks of 32, 527 with blocks of 16), and where the launches it takes more cost less than the steps save: two 16-row workgroups
// of H 256 on a compute unit do their steps in 1.8 us, one 32-row workgroup in 4.2.  us with blocks of 32 and of 16: fp32 L 6
// T 128 B 256 H 256 1091, 752; L 31 T 40 B 20 H 256 306, 243; L 20 T 50 B 100 H 128 303, 211; L 25 T 19 B 106 H 128 162, 119; fp16 L 12 T 30 B 142 H 256
// 263, 170; the other way round at fp32 L 4 T 30 B 128 H 512 228, 315; L 8 T 42 B 215 H 128 126, 139; fp16 L 15 T 25 B 107
// H 512 422, 487; L 3 T 74 B 41 H 1024 469, 562.  `plain`: neither a ragged batch nor a dilation; those take the general loop,
// and ragged ones are slower with blocks of 16 (L 20 T 50 B 250 H 128 528, 639; L 16 T 64 B 220 H 256 1125, 1490; some dilated ones are
// not: L 12 T 64 B 250 H 128 408, 374).
// The steps weigh against the launches, so T counts: fp32 L 16 B 220 H 256 at T 18 375, 399, at T 64 1103, 1043.  Near the line, with
// ordinary launches and with cooperative ones: L 18 T 18 B 216 H 256 603, 469 and 621, 624; L 6 T 92 B 114 H 512 1217, 1222 and 1236, 1316.
// each_launch: us that every launch is charged beyond its cost.
int exchange_layers(int L, int T, int B, int H, bool half, bool plain, float each_launch, bool* many) {
  const ExchangeFlavour f = exchange_flavour_of(H, half);
  *many = false;
  if (!f.one) return 0;
  const int nrb = (B + 31) / 32, W = H / exchange_units(H, half, true), slots = exchange_slots(f.many);
  const int one = exchange_one_block_layers(L, B, H, half);
  const int more = one == L ? 0 : exchange_plan(L, W, nrb, slots).layers;
  if (more == 0 || (one > 0 && (L + one - 1) / one <= (L + more - 1) / more)) return one;
  *many = true;
  const DeviceProps* dp = nullptr;
  if (!plain || one == 0 || device_props(&dp) != FTK_OK) return more;
  const int launches = (L + one - 1) / one, even = (L + launches - 1) / launches;
  auto launch_us = [&](const ExchangeCost& c, bool first, int layers, int slices, int blocks, int team) {
    return each_launch + (first ? c.first : c.next) + (layers - 1) * c.layer + T * blocks * (c.step + c.fill * layers * slices * team / dp->cus);
  };
  const ExchangeCost c16 = exchange_cost(H, half, false), c32 = exchange_cost(H, half, true);
  float us = 0;   // of 16-row blocks minus of 32-row blocks
  for (int l0 = 0; l0 < L; l0 += even)
    us += launch_us(c16, l0 == 0, std::min(even, L - l0), (B + 15) / 16, 1, H / exchange_units(H, half, false));
  for (int l0 = 0; l0 < L; l0 += more) {
    const ExchangePlan p = exchange_plan(std::min(more, L - l0), W, nrb, slots);
    us -= launch_us(c32, l0 == 0, p.layers, p.slices, (nrb + p.slices - 1) / p.slices, W);
  }
  if (us >= 0) return more;
  *many = false;
  return even;
}
}  // namespace

namespace {

// A number that no launch of this process had, and that what a workspace holds by chance does not have: 56 bits, from a random start.
unsigned long long exchange_launch_number() {
  static std::atomic<unsigned long long> next{[] {
    try {
      std::random_device r;
      return (unsigned long long)r() << 32 | r();
    } catch (...) {   // no source of random numbers: the time, spread over the bits
      return (unsigned long long)std::chrono::system_clock::now().time_since_epoch().count() * 0x9e3779b97f4a7c15ull;
    }
  }()};
  while (true)
    if (const unsigned long long v = next.fetch_add(1, std::memory_order_relaxed) & ((1ull << 56) - 1)) return v;
}

}  // namespace

// Whether the whole batch of every layer fits the chip with one block of 16 rows per workgroup.
bool exchange_one_block(int L, int B, int H, bool half) { return exchange_one_block_layers(L, B, H, half) == L; }

// Row blocks of 32 rows that a workgroup has to walk in a stack's first launch (0: the device holds none).
int exchange_blocks(int L, int B, int H, bool half) {
  const ExchangeFlavour f = exchange_flavour_of(H, half);
  if (!f.many) return 0;
  const int nrb = (B + 31) / 32;
  const ExchangePlan p = exchange_plan(L, H / exchange_units(H, half, true), nrb, exchange_slots(f.many));
  return p.layers ? (nrb + p.slices - 1) / p.slices : 0;
}

// Bytes of workspace that run_exchange uses on the current device, however it launches; without a device, what it could at most.
size_t exchange_need(int L, int T, int B, int H, bool half) {
  bool many;
  int most = exchange_layers(L, T, B, H, half, false, kAnyLaunch, &many);
  for (const float each_launch : {0.0f, kAnyLaunch, kCooperativeLaunch}) most = std::max(most, exchange_layers(L, T, B, H, half, true, each_launch, &many));
  return exchange_workspace_bytes(most ? std::min(L, most) : L, T, B, H, half);
}

// Runs the stack; *handled is false when the device cannot hold a layer, or the workspace has less room than that:
// other kernels may do with it.  Deeper stacks than a launch holds run as
// consecutive launches, each reading the hidden sequence of the layer below it like the first reads xs.
int run_exchange(bool half, const void* xs, const void* WU, const float* bias, const int* dil, const int* active, void* hsss,
                 void* csss, int L, int T, int B, int H, void* ws, size_t ws_bytes, hipStream_t s, bool* handled, int spin_limit) {
  *handled = false;
  const ExchangeFlavour f = exchange_flavour_of(H, half);
  if (!f.one) return FTK_OK;
  bool plain = !active;
  for (int l = 0; dil && l < L; ++l) plain = plain && dil[l] == 1;
  bool many;
  const int most = exchange_layers(L, T, B, H, half, plain, !half ? kAnyLaunch : launch_is_cooperative(s) ? kCooperativeLaunch : 0.0f, &many);
  if (most == 0) return FTK_OK;
  const int slots = exchange_slots(many ? f.many : f.one), block = many ? 32 : 16, nrb = (B + block - 1) / block;
  const int W = H / exchange_units(H, half, many);
  const size_t esize = half ? 2 : 4, slab = (size_t)T * B * H, wlayer = (size_t)8 * H * H, tile = exchange_tile_bytes(H, half, block);
  const size_t places_at = exchange_places_at(ws), xratio_at = places_at + exchange_xratio_at;
  const size_t ring_from = xratio_at + align256((size_t)(T + 1) * nrb * block * sizeof(float));
  if (!ws || ws_bytes < places_at + exchange_buffer_bytes(std::min(L, most), T, B, H, half)) return FTK_OK;
  // (less room than the size query asks for, but enough with nothing between the buffers: so)
  auto tiles_of = [&](int layers, size_t to) {
    return exchange_tiles_at(ws, to, ring_from, (size_t)layers * nrb * kXRing * tile, (size_t)(layers + 1) * T * nrb * tile);
  };
  const size_t tiles_to = ws_bytes >= tiles_of(std::min(L, most), kXTilesAt).end ? kXTilesAt : 256;
  const bool records = stream_records(s);
  for (int l0 = 0; l0 < L; l0 += most) {
    const int lc = std::min(most, L - l0);
    const ExchangePlan p = exchange_plan(lc, W, nrb, slots);
    ExchangeArgs a;
    const void* x = l0 == 0 ? xs : (const char*)hsss + (size_t)(l0 - 1) * slab * esize;
    a.WU = (const char*)WU + (size_t)l0 * wlayer * esize;
    a.bias = bias ? bias + (size_t)l0 * 4 * H : nullptr;
    a.hsss = (char*)hsss + (size_t)l0 * slab * esize;
    a.csss = (char*)csss + (size_t)l0 * slab * esize;
    a.status = (int*)ws;
    a.place = (unsigned long long*)((char*)ws + places_at);
    float* xratio = (float*)((char*)ws + xratio_at);
    a.xratio = xratio;
    const ExchangeTiles tiles = tiles_of(lc, tiles_to);
    a.ring = (unsigned char*)ws + tiles.ring;
    a.hand = (unsigned char*)ws + tiles.hand;
    a.L = lc; a.T = T; a.B = B; a.nrb = nrb;
    a.slices = p.slices;
    a.units = lc * p.slices;
    a.per_xcd = p.per_xcd;
    a.spin_limit = spin_limit > 0 ? spin_limit : 1 << 22;
    a.ragged = active && nrb <= kXBlocks ? 1 : 0;
    for (int l = 0; l < kXLayers; ++l) a.dil[l] = l < lc && dil ? dil[l0 + l] : 1;
    for (int rb = 0; rb < kXBlocks; ++rb) {
      int steps = 0;
      if (a.ragged)
        while (steps < T && active[steps] > block * rb) ++steps;
      a.steps_of[rb] = steps;
    }
    const int groups = a.units * W;
    const unsigned grid = p.per_xcd ? 8u * p.per_xcd * W : (unsigned)((groups + 7) / 8 * 8);
    // The launch lays out its own buffers, unless it is recorded (a replay would find the places of the one before, with its number in them), or a
    // workgroup had too many rows to lay out in front of its first step: a turn of 32 takes it 0.6 us once the first two are on their way
    // beside the weights, the kernel in front takes 1 us for some 4000 rows more (us in a row, that kernel and without: L 1 H 64 T 24 B 8, 3 turns,
    // 28.5, 28.2; T 128 B 8, 16 turns, 117.3, 124.4, B 250 129.5, 126.1; L 2 H 64 T 96 B 8, 6 turns, 111.5, 113.0, B 100 96.5, 94.5; L 1 H 256
    // T 128 B 8, 4 turns, 161.4, 161.8, B 40 164.9, 162.4; 230 stacks in all).
    a.launch = exchange_launch_number();
    a.clear_status = l0 == 0;
    a.early = lc == 1 || (p.per_xcd > 0 && p.per_xcd % lc == 0);
    if (const char* e = getenv("FTK_LSTM_EXCHANGE_EARLY")) a.early = e[0] == '1';   // =1 / =0: where no h of the team goes to another XCD / never
    const int row_groups = (nrb + p.slices - 1) / p.slices * ((T + 1) / 2 * 2) * block / 32;   // 32 rows each, of a slice
    a.row_layers = std::max(1, std::min({lc, (row_groups + W - 1) / W, kXRowPlaces / W}));
    const int turns = (row_groups + a.row_layers * W - 1) / (a.row_layers * W);
    bool own = 0.6f * (turns - 2) <= 0.5f + (float)T * B / 4000;
    if (const char* e = getenv("FTK_LSTM_EXCHANGE_FRONT")) own = e[0] != '1';   // =1 / =0: that kernel / none, where both can be
    own = own && !records;
    a.xs = own ? x : nullptr;
    if (!own) {
      const unsigned ring_per_layer = (unsigned)((size_t)nrb * kXRing * tile / 16), hand_first = (unsigned)((size_t)std::min(T, 2) * nrb * tile / 16);
      const size_t hand_per_layer = (size_t)T * nrb * tile / 16;
      const int prepare_groups = (int)std::min<size_t>(((size_t)T * nrb * block + 3) / 4, 2048);
      const dim3 pgrid(prepare_groups + lc * ((ring_per_layer + hand_first + kPrepareFill - 1) / kPrepareFill));
      auto prepare = half ? lstm_exchange_prepare_kernel<true> : lstm_exchange_prepare_kernel<false>;
      hipLaunchKernelGGL(prepare, pgrid, dim3(256), 0, s, a.status, l0 > 0 ? 2 : 0, a.place, groups, (v4u*)a.ring, ring_per_layer, (v4u*)a.hand,
                         hand_per_layer, hand_first, x, xratio, prepare_groups, T, B, nrb, block, H);
      const int rc = check_launch("lstm_exchange_prepare_kernel");
      if (rc) return rc;
    }
    void* kargs[] = {&a};
    const int rc = launch_resident(many ? f.many : f.one, dim3(grid), dim3(256), kargs, 0, s);
    if (rc) return rc;
  }
  *handled = true;
  return FTK_OK;
}

}  // namespace ftk
