// Row-invariant GEMM of the LM head and the projections: out[m, n] = bf16(sum_k x[rows[m], k] * weight[n, k]) with
// the verifier's argmax pass in its epilogue (replaces ParallelLMHead.forward for the rows the verifier reads,
// nanovllm/layers/embed_head.py:56-68, the first read of the logits by verify_drafts, nanovllm/layers/sampler.py:66,
// and, without the argmax, the linear layers of nanovllm/layers/linear.py).
//
// Every output element is a sum of ranges of k in range order, each range one chain of v_mfma_f32_16x16x32_bf16 over
// its k in fp32, rounded once to bf16 at the end. How many ranges (1 to 8) follows from the weight's shape and the
// element's packed tile (Ranges), never from the kernel, its tile or the call's row count: a row's result depends on
// its input row and the weight alone. Ranges shorten the chains: of 4096 x 12288 outputs 2.9e-4 differ from the rounded
// 64-bit product with eight ranges and 4.7e-4 with one chain (4096 x 4096: 1.7e-4 and 2.7e-4). One workgroup runs
// all ranges of its outputs, the finished ranges' sum beside the running one in registers: as workgroups of their own
// their sums went through memory and a second launch, 33 us of the 149 us that a 5-row call of the four Qwen3-8B
// projections took, and 52 of 246 us at 320 rows.
//
// Packed weight (once per weight, lm_head_pack_weight): wp[t][s][r][c] = weight[256 t + r][32 s + c], rows past the
// vocabulary zero: the 16 rows x 32 columns that one wave's A operand needs are one contiguous 1 KB block. The
// activations are read where they are, the logits_indices gather folded into the row addresses.
//
//   stream_gemm  up to 16 rows: one wave per 16 or 32 weight rows, both operands straight into registers, 16 steps
//                of 32 columns ahead. HBM bound: the weight is the traffic.
//   tile_gemm    more rows (and few rows of a vocabulary-sized weight): a workgroup of WN x WM waves owns
//                (16 TN WN) weight rows x (16 TM WM) token rows.
//                  * A (weight): each wave loads its own rows into registers, DA - 1 steps of 32 columns ahead. The
//                    weight does not pass through LDS: at 256 x 256 the LDS reads and writes of a step would take
//                    as long as its MFMAs (128 B a clock), this way they take about 0.6 of that.
//                  * B (tokens): stages of 64 columns (whole 128-byte lines of a row) in an LDS ring of RX slots,
//                    loaded with global_load_lds; slot rows of 128 B, 16-byte chunk c of row r at
//                    c ^ ((r >> 1) & 7), so that 16 rows at one chunk cover all banks. A step's operand reads are
//                    issued one step ahead, column by column, each behind the MFMAs that used its registers.
//                  * One barrier per two steps. Past the end the loads repeat the last step's addresses (never
//                    used), so every wait is a constant count; what ends a range stands between two steps and
//                    touches registers only.
//                Loads, LDS reads and MFMAs are inline asm: next to LDS DMA in flight the compiler would wait for
//                every load before a use. Their results are tied to the waits, and every register set stays
//                allocated until the last load has landed (tests/test_asm_gemm.py checks the compiled code).
#pragma once
#include <type_traits>

#include "sd_common.h"

namespace sd {
namespace lmhead {

constexpr int kN = 256;                            // rows of a packed weight tile
constexpr int kK = 32;                             // columns of a packed block: one MFMA step
constexpr int kBlockBytes = kN * kK * 2;           // 16 KB: one step of a packed tile
constexpr int kStreamRows = 16;                    // stream_gemm's token rows

struct TileBest {  // first argmax of one token row over some weight rows; idx 0x7fffffff: nothing above -inf
  float val;
  int32_t idx;
};
// A workgroup's candidate in memory: the value, which is a bf16, and its index among the workgroup's weight rows
// (0xffff: none). In four bytes, so that 128-row workgroups need no more of the caller's workspace than 256-row ones
// with a whole TileBest.
__device__ __forceinline__ uint32_t pack_best(float val, int32_t idx, int32_t first) {
  return (__builtin_bit_cast(uint32_t, val) & 0xffff0000u) | (idx == 0x7fffffff ? 0xffffu : (uint32_t)(idx - first));
}
__device__ __forceinline__ TileBest unpack_best(uint32_t c, int32_t first) {
  return {__builtin_bit_cast(float, c & 0xffff0000u), (c & 0xffff) == 0xffff ? 0x7fffffff : first + (int32_t)(c & 0xffff)};
}

struct Args {
  const uint16_t* x;        // [*, K] bf16 rows, stride x_stride
  int64_t x_stride;
  const int64_t* rows;      // null (row m is token row m), or the gather; an index outside [0, x_rows) gives zeros
  int64_t x_rows;
  int32_t M;                // token rows
  const uint16_t* wp;       // packed weight
  int32_t N, K;
  uint16_t* out;            // null, or [M, N] bf16 with row stride out_stride
  int64_t out_stride;
  int32_t out_align;        // what out and its row stride are multiples of: 16, 8 or 2 bytes (8, 4 or 1 entries a store)
  int32_t out_nt;           // non-temporal stores of whole lines (logits: they leave the token rows in L2)
  uint32_t* best;           // [M][tiles_n] candidates (pack_best), or null (no argmax)
  int32_t tiles_n, tiles_m;
  int32_t full, splits;     // packed tiles from `full` on are summed in `splits` ranges of k, the others in one
};

// A weight's ranges: `splits` of them in the packed tiles from `full` on. With one 256-row workgroup a tile and 256
// CUs, the tiles of a last round that fills at most half of them are cut into as many ranges as fit the rest, at most
// 8 and none shorter than two steps (Qwen3-8B: the last 82 tiles of the LM head 3 ranges, gate_up_proj 2, the other
// projections 8). The rule is part of the results: 256 is not the device's CU count but a constant.
struct Ranges {
  int full, splits;
};
inline Ranges sum_ranges(int N, int K) {
  constexpr int kRound = 256;
  const int tiles = (N + kN - 1) / kN;
  const int tail = tiles - (tiles - 1) / kRound * kRound;   // tiles of the last round, 1..kRound
  if (2 * tail > kRound) return {tiles, 1};
  const int by_round = kRound / tail, by_k = K / (2 * kK);
  int splits = by_round < by_k ? by_round : by_k;
  if (splits > 8) splits = 8;
  return splits < 2 ? Ranges{tiles, 1} : Ranges{tiles - tail, splits};
}
// Where the ranges of a packed tile end: range r of n covers the steps r S / n .. (r + 1) S / n - 1. No end is given
// for the last range: its sum is added behind the loop. -0 is the sum of no range: -0 + x is x for every x.
struct RangeEnd {
  int left, n, whole, rest, part, end;   // ranges after this one; S = n whole + rest, (r + 1) rest = n (...) + part
  __device__ __forceinline__ void start(int S, int ranges) {
    left = ranges - 1;
    n = ranges;
    whole = S / ranges;
    rest = S - whole * ranges;
    part = rest;
    end = left ? whole : 0x7fffffff;
  }
  __device__ __forceinline__ void next() {
    part += rest;
    end += whole + (part >= n ? 1 : 0);
    if (part >= n) part -= n;
    if (--left == 0) end = 0x7fffffff;
  }
};
__device__ __forceinline__ f32x4 no_sum() { return f32x4{-0.f, -0.f, -0.f, -0.f}; }

// One thread per 16 bytes of the packed weight.
__global__ __launch_bounds__(256) void lm_head_pack_weight(const uint16_t* __restrict__ w, int32_t V, int32_t H,
                                                           int32_t tiles, uint16_t* __restrict__ wp) {
  const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;   // 16-byte chunk of the output
  const int S = H / 32;
  if (o >= (int64_t)tiles * S * kN * 4) return;
  const int c8 = (int)(o % 4);
  const int r = (int)((o / 4) % kN);
  const int64_t ts = o / (4 * kN);
  const int s = (int)(ts % S);
  const int t = (int)(ts / S);
  const int n = kN * t + r;
  u32x4 v = {0, 0, 0, 0};
  if (n < V) v = *(const u32x4*)(w + (int64_t)n * H + 32 * s + 8 * c8);
  *(u32x4*)(wp + o * 8) = v;
}

// The call's token rows copied to dst [M][K] (gathered; an index outside the table gives a zero row), for calls
// whose output overlaps their input. One thread per 16 bytes.
__global__ __launch_bounds__(256) void copy_rows(const uint16_t* __restrict__ x, int64_t stride, int64_t x_rows,
                                                 const int64_t* __restrict__ rows, int32_t M, int32_t K,
                                                 uint16_t* __restrict__ dst) {
  const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int chunks = K / 8;
  if (o >= (int64_t)M * chunks) return;
  const int m = (int)(o / chunks), c = (int)(o % chunks);
  const int64_t r = rows ? rows[m] : (int64_t)m;
  u32x4 v = {0, 0, 0, 0};
  if (r >= 0 && r < x_rows) v = *(const u32x4*)(x + r * stride + 8 * c);
  *(u32x4*)(dst + o * 8) = v;
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15) : "memory");
}
// A value that passes through here is not read before, nor its registers reused until, this point; it is in AGPRs (kA)
// or VGPRs. A kernel that needs more than 256 registers a wave keeps in AGPRs what the VALU touches least: the
// weight, then the accumulators.
template <bool kA, class V>
__device__ __forceinline__ void tie(V& f) {
  if constexpr (kA)
    asm volatile("" : "+a"(f));
  else
    asm volatile("" : "+v"(f));
}
template <bool kAccA, bool kWeightA>
__device__ __forceinline__ void mfma(f32x4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (kAccA && kWeightA)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "a"(a), "v"(b));
  else if constexpr (kAccA)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else if constexpr (kWeightA)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "a"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
// c = 0, where it is: given a new value, the compiler moves the accumulators of a large shape to other registers and back.
template <bool kAccA>
__device__ __forceinline__ void mfma_zero(f32x4& c, const bf16x8& zero) {
  if constexpr (kAccA)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "+a"(c) : "v"(zero));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "+v"(c) : "v"(zero));
}
template <int OFF>
__device__ __forceinline__ void lds_read(bf16x8& f, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f) : "v"(addr), "n"(OFF) : "memory");
}
template <bool kNT, bool kA, int OFF>
__device__ __forceinline__ void load_frag(bf16x8& f, uint32_t off, const uint8_t* base) {
  if constexpr (kNT && kA)
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3 nt" : "=a"(f) : "v"(off), "s"(base), "n"(OFF) : "memory");
  else if constexpr (kNT)
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3 nt" : "=v"(f) : "v"(off), "s"(base), "n"(OFF) : "memory");
  else if constexpr (kA)
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=a"(f) : "v"(off), "s"(base), "n"(OFF) : "memory");
  else
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(f) : "v"(off), "s"(base), "n"(OFF) : "memory");
}

// Calls f(integral_constant<I>) for I = I0 .. N - 1: registers and wait counts are indexed at compile time.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

typedef __attribute__((address_space(3))) void lds_void;

// The token row m (clamped to the call's rows) as a row of x; an index outside the table reads row 0 (its result
// is replaced by zeros in the epilogue).
__device__ __forceinline__ int64_t x_row(const Args& a, int m) {
  m = min(m, a.M - 1);
  if (!a.rows) return m;
  const int64_t r = a.rows[m];
  return r >= 0 && r < a.x_rows ? r : 0;
}
__device__ __forceinline__ bool row_valid(const Args& a, int m) {
  if (!a.rows || m >= a.M) return true;
  const int64_t r = a.rows[m];
  return r >= 0 && r < a.x_rows;
}

// Four consecutive entries of a token row, rounded to bf16 (zeros for an invalid row).
__device__ __forceinline__ uint2 round4(const f32x4& acc, bool valid) {
  const uint2 w = make_uint2(cvt_bf16x2(acc[0], acc[1]), cvt_bf16x2(acc[2], acc[3]));
  return valid ? w : make_uint2(0, 0);
}
// The first argmax (a NaN above all, nothing for -inf alone) of a lane's entries of one token row, w[i] those from
// n + 16 i on. The maximum, then the first entry that equals it: about 3 instructions an entry. A running argmax takes
// 9 in a chain, which one wave a SIMD cannot hide (3 us a workgroup of 256 x 160); it is left for waves with a NaN.
template <int TN>
__device__ __forceinline__ TileBest lane_best(const Args& a, const uint2 (&w)[TN], int n) {
  float v[TN][4], top = -INFINITY;
  bool nan = false;
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    v[i][0] = __builtin_bit_cast(float, w[i].x << 16);
    v[i][1] = __builtin_bit_cast(float, w[i].x & 0xffff0000u);
    v[i][2] = __builtin_bit_cast(float, w[i].y << 16);
    v[i][3] = __builtin_bit_cast(float, w[i].y & 0xffff0000u);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + 16 * i + e >= a.N) v[i][e] = -INFINITY;
    nan |= __builtin_isunordered(v[i][0], v[i][1]) | __builtin_isunordered(v[i][2], v[i][3]);
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(top) : "v"(v[i][0]), "v"(v[i][1]));
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(top) : "v"(v[i][2]), "v"(v[i][3]));
  }
  TileBest b = {top, 0x7fffffff};
  if (__builtin_amdgcn_ballot_w64(nan)) {
    b.val = -INFINITY;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool take = (b.val == b.val) & !(v[i][e] <= b.val);
        b.val = take ? v[i][e] : b.val;
        b.idx = take ? n + 16 * i + e : b.idx;
      }
    return b;
  }
#pragma unroll
  for (int i = TN - 1; i >= 0; --i)
#pragma unroll
    for (int e = 3; e >= 0; --e) b.idx = v[i][e] == top ? n + 16 * i + e : b.idx;
  b.idx = top == -INFINITY ? 0x7fffffff : b.idx;
  return b;
}
// The first argmax over the four lanes that hold one token row's entries (l, l ^ 16, l ^ 32, l ^ 48).
__device__ __forceinline__ void lanes_best(float& bv, int& bi) {
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) {
    const float ov = __shfl_xor(bv, off);
    const int oi = __shfl_xor(bi, off);
    if (better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
}

// Up to 16 token rows. Lane l holds row l % 16 of both operands, columns 8 (l / 16) .. + 7 of each step; one wave takes
// 16 TN weight rows, kStreamDepth steps of 32 columns ahead. More rows a wave read the token rows fewer times per byte
// of weight, fewer keep a small matrix spread over the GPU (row_plan): at 5 rows 4096 x 12288 took 21.0 / 24.3 us
// with 16 / 32 rows a wave, 24576 x 4096 44.2 / 35.9 us (5.6 TB/s).
constexpr int kStreamDepth = 16;
template <int TN>
__global__ __launch_bounds__(kWave) void stream_gemm(Args a) {
  constexpr int D = kStreamDepth;
  const int lane = threadIdx.x, r16 = lane % 16, g = lane / 16;
  const int S = a.K / kK;
  const int n0 = blockIdx.x * 16 * TN;
  const uint8_t* wsrc =
      (const uint8_t*)a.wp + (int64_t)(n0 / kN) * S * kBlockBytes + (n0 % kN) * 64 + r16 * 64 + g * 16;
  const uint8_t* xsrc = (const uint8_t*)(a.x + x_row(a, r16) * a.x_stride) + g * 16;
  bf16x8 fa[D][TN], fb[D];
  f32x4 acc[TN], sum[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    acc[i] = f32x4{};
    sum[i] = no_sum();
  }
  RangeEnd range;
  range.start(S, n0 / kN >= a.full ? a.splits : 1);
  auto load = [&](int t, bf16x8 (&fa)[TN], bf16x8& fb) {   // past the end: the last step again, never used
    const int s = min(t, S - 1);
#pragma unroll
    for (int i = 0; i < TN; ++i)
      fa[i] = __builtin_nontemporal_load((const bf16x8*)(wsrc + (int64_t)s * kBlockBytes + i * 1024));
    fb = *(const bf16x8*)(xsrc + (int64_t)s * 64);
  };
  auto step = [&](int d) {
#pragma unroll
    for (int i = 0; i < TN; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[d][i], fb[d], acc[i], 0, 0, 0);
  };
  auto end_range = [&](int t) {   // behind step t
    if (__builtin_expect(t + 1 == range.end, 0)) {
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        sum[i] = sum[i] + acc[i];
        acc[i] = f32x4{};
      }
      range.next();
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, fa[d], fb[d]);
  int t = 0;
  for (; t + D <= S; t += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      step(d);
      end_range(t + d);
      load(t + d + D, fa[d], fb[d]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (t + d < S) {
      step(d);
      end_range(t + d);
    }
  const bool valid = row_valid(a, r16);
  uint2 ws[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int n = n0 + 16 * i + 4 * g;
    const uint2 w = ws[i] = round4(sum[i] + acc[i], valid);
    if (!a.out || r16 >= a.M) continue;
    uint16_t* dst = a.out + (int64_t)r16 * a.out_stride + n;
    if (n + 3 < a.N && a.out_align >= 8) {
      *(uint2*)dst = w;
    } else {
      const uint16_t bits[4] = {(uint16_t)w.x, (uint16_t)(w.x >> 16), (uint16_t)w.y, (uint16_t)(w.y >> 16)};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < a.N) dst[e] = bits[e];
    }
  }
  if (a.best) {
    TileBest b = lane_best(a, ws, n0 + 4 * g);
    lanes_best(b.val, b.idx);
    if (g == 0 && r16 < a.M) a.best[(int64_t)r16 * a.tiles_n + blockIdx.x] = pack_best(b.val, b.idx, n0);
  }
}

// One workgroup shape of tile_gemm. DA: register sets of weight (steps ahead + 1, even); RX: LDS slots of token
// stages; kAccA / kWeightA: accumulators / weight in AGPRs; kNT: the weight non-temporal (shapes that mostly read it
// once); kEnds: a range may end behind every kEnds-th step (1 or DA; 0: the registers do not take a sum of ranges, the
// shape runs tiles of one range only).
template <int TN_, int TM_, int WN_, int WM_, int DA_, int RX_, bool kAccA_, bool kWeightA_, bool kNT_, int kEnds_ = 1>
struct Tile {
  static constexpr int TN = TN_, TM = TM_, WN = WN_, WM = WM_, DA = DA_, RX = RX_;
  static constexpr bool kAccA = kAccA_, kWeightA = kWeightA_, kNT = kNT_, kSums = kEnds_ > 0;
  static constexpr int kEnds = kEnds_ ? kEnds_ : 1;
  static constexpr int kWaves = WN * WM, kThreads = kWaves * kWave;
  static constexpr int kRowsN = 16 * TN * WN, kRowsM = 16 * TM * WM;
  static constexpr int kSlot = kRowsM * 128;                         // one stage of 64 columns
  static constexpr int kPieces = (kRowsM / 8 + kWaves - 1) / kWaves;  // 1 KB loads of a stage per wave
  static_assert(kEnds == 1 || kEnds == DA, "a group of DA steps has one place or all");
  static_assert(DA % 2 == 0 && 2 * (RX - 2) >= DA - 2, "the stages ahead cover the steps ahead");
  static_assert(kN % kRowsN == 0 && TN <= 4, "a workgroup's weight rows lie in one packed tile");
  static_assert(TM <= 16, "lgkmcnt counts the reads ahead");
  static constexpr int kRing = RX * kSlot, kRed = kRowsM * WN * (int)sizeof(TileBest);
  static_assert(kRing + kRed <= 160 * 1024 && kRowsM * kRowsN * 2 <= kRing, "the ring takes the output tile");
};

template <class T>
__global__ __launch_bounds__(T::kThreads, 1) void tile_gemm(Args a) {
  constexpr int TN = T::TN, TM = T::TM, WN = T::WN, DA = T::DA, RX = T::RX, PX = T::kPieces;
  constexpr int XS = T::kSlot, MT = T::kRowsM;
  __shared__ __attribute__((aligned(16))) uint8_t lds[T::kRing + T::kRed];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wn = wave % WN, wm = wave / WN;
  const int S = a.K / kK, nst = (S + 1) / 2;
  // Workgroups go round-robin over the 8 XCDs: XCD k takes the weight tiles k, k + 8, ..., all token tiles of one
  // before the next, so that a weight tile is read from HBM by one XCD's L2 only.
  const int xcd = blockIdx.x % 8, j0 = blockIdx.x / 8;
  const int nt = xcd + 8 * (j0 / a.tiles_m), mt = j0 % a.tiles_m;
  if (nt >= a.tiles_n) return;
  const int m0 = mt * MT;
  const int nw = nt * T::kRowsN + wn * TN * 16;   // this wave's first weight row
  const uint8_t* wbase = (const uint8_t*)a.wp + (int64_t)(nw / kN) * S * kBlockBytes + (nw % kN) * 64;
  const uint32_t wlane = (lane % 16) * 64 + (lane / 16) * 16;

  // Token loads: lane l's 16 bytes land at the instruction's LDS base + 16 l: row l / 8 of the piece's 8 rows,
  // physical chunk l % 8, so the lane fetches the logical chunk that the swizzle puts there.
  uint64_t xsrc[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int r = 8 * min(wave * PX + i, MT / 8 - 1) + lane / 8;
    xsrc[i] = (uint64_t)(a.x + x_row(a, m0 + r) * a.x_stride + 8 * ((lane % 8) ^ ((r >> 1) & 7)));
    asm volatile("" : "+v"(xsrc[i]));
  }
  const int half_stage = S % 2 ? nst - 1 : -1;  // a last stage of 32 columns: its upper chunks repeat the lower ones
  auto load_x = [&](int st, uint32_t slot, int i) __attribute__((always_inline)) {
    const int q = min(wave * PX + i, MT / 8 - 1);
    uint64_t p = xsrc[i] + (uint64_t)(uint32_t)(st * 128);
    if (st == half_stage && ((lane % 8) ^ (((8 * q + lane / 8) >> 1) & 7)) >= 4) p -= 64;
    __builtin_amdgcn_global_load_lds((const void*)p, (lds_void*)(lds + slot + q * 1024), 16, 0, 0);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      acc[i][j] = f32x4{};
      tie<T::kAccA>(acc[i][j]);
    }
  asm volatile("s_nop 7");
  f32x4 sum[T::kSums ? TN : 1][T::kSums ? TM : 1];
  RangeEnd range;
  if constexpr (T::kSums) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) sum[i][j] = no_sum();
    range.start(S, nw / kN >= a.full ? a.splits : 1);
  }
  // Registers only, so that it may stand between any two steps; the waits are the MFMAs' results to the VALU and
  // the zeros to the next MFMAs.
  auto end_range = [&](int t) __attribute__((always_inline)) {   // behind step t
    if constexpr (T::kSums) {
      if ((t + 1) % T::kEnds != 0 || __builtin_expect(t + 1 != range.end, 1)) return;
      bf16x8 zero = {};
      tie<false>(zero);
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          tie<T::kAccA>(acc[i][j]);
          sum[i][j] = sum[i][j] + acc[i][j];
          tie<false>(sum[i][j]);
          mfma_zero<T::kAccA>(acc[i][j], zero);
        }
      asm volatile("s_nop 15");
      range.next();
    }
  };
  const int r16 = lane % 16, g = lane / 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const uint32_t swz = (r16 >> 1) & 7;
  const uint32_t brow = lds0 + (wm * TM * 16 + r16) * 128;
  const uint32_t boff[2] = {brow + ((g ^ swz) << 4), brow + (((4 + g) ^ swz) << 4)};  // even / odd step of a stage

  bf16x8 fa[DA][TN], fb[TM];
  uint32_t xw = (RX - 1) * XS, xr = 0;   // slots of the next stage to load and of the stage being read
  // Step t: the MFMAs of columns 32 t .. + 31. Behind each token block's MFMAs its next operand read goes out, and
  // the step's loads (the weight of step t + DA - 1; in odd steps the token stage RX - 1 ahead) are spread over
  // the blocks. kLoad = false: the last steps of a K that is not a multiple of 32 DA, everything already loaded.
  auto step = [&](int t, auto dc, auto loadc) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value, prev = (d + DA - 1) % DA, odd = d % 2;
    constexpr bool kLoad = decltype(loadc)::value;
    // Loads issued after those this step needs: its own weight (issued at the end of step t - DA + 1) and, in an
    // odd step, the next stage's tokens (issued in step t - 2 (RX - 2)).
    constexpr int kAfterA = (DA - 2) * TN + (DA / 2 - 1) * PX, kAfterX = 2 * (RX - 2) * TN + (RX - 3) * PX;
    if constexpr (kLoad) wait_vm<odd && kAfterX < kAfterA ? kAfterX : kAfterA>();
    static_for<0, TN>([&](auto i) { tie<T::kWeightA>(fa[d][decltype(i)::value]); });
    if constexpr (odd) {
      // every wave's part of the next stage has landed, and every wave is done with the stage before this one
      if constexpr (kLoad) __builtin_amdgcn_s_barrier();
      xr = xr + XS == RX * XS ? 0 : xr + XS;
    }
    const int xst = min((t - 1) / 2 - 1 + RX, nst - 1);
    const uint32_t baddr = boff[1 - odd] + xr;
    const uint8_t* wnext = wbase + (uint64_t)(uint32_t)min(t + DA - 1, S - 1) * kBlockBytes;
    constexpr int kX = odd ? PX : 0, kItems = kX + TN;
    static_for<0, TM>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      wait_lgkm<TM - 1>();
      tie<false>(fb[j]);
      static_for<0, TN>([&](auto i) {
        mfma<T::kAccA, T::kWeightA>(acc[decltype(i)::value][j], fa[d][decltype(i)::value], fb[j]);
      });
      lds_read<j * 2048>(fb[j], baddr);
      if constexpr (kLoad)
        static_for<j * kItems / TM, (j + 1) * kItems / TM>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          if constexpr (k < kX)
            load_x(xst, xw, k);
          else
            load_frag<T::kNT, T::kWeightA, (k - kX) * 1024>(fa[prev][k - kX], wlane, wnext);
        });
    });
    if constexpr (odd) xw = xw + XS == RX * XS ? 0 : xw + XS;
  };

  for (int st = 0; st < RX - 1; ++st)
#pragma unroll
    for (int i = 0; i < PX; ++i) load_x(min(st, nst - 1), st * XS, i);
  static_for<0, DA - 1>([&](auto d) {
    const uint8_t* p = wbase + (uint64_t)(uint32_t)min((int)decltype(d)::value, S - 1) * kBlockBytes;
    static_for<0, TN>([&](auto i) {
      load_frag<T::kNT, T::kWeightA, decltype(i)::value * 1024>(fa[decltype(d)::value][decltype(i)::value], wlane, p);
    });
  });
  wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  static_for<0, TM>([&](auto j) { lds_read<decltype(j)::value * 2048>(fb[decltype(j)::value], boff[0]); });
  int t = 0;
  for (; t + DA <= S; t += DA) {
    static_for<0, DA>([&](auto d) {
      step(t + decltype(d)::value, d, std::true_type{});
      end_range(t + decltype(d)::value);
    });
  }
  // Nothing in flight past here; until here no register set was free for another value.
  wait_vm<0>();
  static_for<0, DA - 1>([&](auto d) {
    static_for<0, TN>([&](auto i) { tie<T::kWeightA>(fa[decltype(d)::value][decltype(i)::value]); });
  });
  if (t < S) {
    __builtin_amdgcn_s_barrier();
    static_for<0, DA - 1>([&](auto d) {
      if (t + decltype(d)::value < S) {
        step(t + decltype(d)::value, d, std::false_type{});
        end_range(t + decltype(d)::value);
      }
    });
  }
  wait_lgkm<0>();
  static_for<0, TM>([&](auto j) { tie<false>(fb[decltype(j)::value]); });
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMAs' results before the VALU reads them
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) tie<T::kAccA>(acc[i][j]);

  // ---- epilogue: a lane holds entries 16 i + 4 g .. + 3 of token row 16 j + r16. The rounded tile goes through the
  // ring's bytes (row mr of 2 NT bytes, 16-byte chunk c at c ^ (mr % 16)), so that the stores cover whole lines: with
  // 8-byte stores from the accumulators the LM head at 320 rows took 20 us longer with its logits than without ----
  constexpr int NT = T::kRowsN, kChunks = NT / 8, kSwz = (kChunks < 16 ? kChunks : 16) - 1;
  TileBest* red = (TileBest*)(lds + T::kRing);  // [MT][WN]
  __syncthreads();                              // every wave's last reads of the ring
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int mr = wm * TM * 16 + 16 * j + r16;
    const bool valid = row_valid(a, m0 + mr);
    uint2 ws[TN];
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int nr = wn * TN * 16 + 16 * i + 4 * g;
      if constexpr (T::kSums) acc[i][j] = sum[i][j] + acc[i][j];   // the last range
      ws[i] = round4(acc[i][j], valid);
      *(uint2*)(lds + mr * (2 * NT) + (((nr / 8) ^ (mr & kSwz)) << 4) + 8 * (g % 2)) = ws[i];
    }
    if (a.best) {
      TileBest b = lane_best(a, ws, nt * NT + wn * TN * 16 + 4 * g);
      lanes_best(b.val, b.idx);
      if (g == 0) red[mr * WN + wn] = b;
    }
  }
  __syncthreads();
  const int rows = min(MT, a.M - m0), cols = min(NT, a.N - nt * NT);
  if (a.out) {
    uint16_t* out = a.out + (int64_t)m0 * a.out_stride + nt * NT;
    if (a.out_align == 16 && cols == NT) {
      auto store_rows = [&](auto ntc) __attribute__((always_inline)) {
        for (int idx = threadIdx.x; idx < rows * kChunks; idx += T::kThreads) {
          const int mr = idx / kChunks, c = idx % kChunks;
          const u32x4 w = *(const u32x4*)(lds + mr * (2 * NT) + ((c ^ (mr & kSwz)) << 4));
          u32x4* dst = (u32x4*)(out + mr * a.out_stride + 8 * c);
          if constexpr (decltype(ntc)::value)
            __builtin_nontemporal_store(w, dst);
          else
            *dst = w;
        }
      };
      if (a.out_nt)
        store_rows(std::true_type{});
      else
        store_rows(std::false_type{});
    } else if (a.out_align >= 8) {   // and the last columns of a ragged weight
      for (int idx = threadIdx.x; idx < rows * (NT / 4); idx += T::kThreads) {
        const int mr = idx / (NT / 4), n = 4 * (idx % (NT / 4));
        const uint2 w = *(const uint2*)(lds + mr * (2 * NT) + (((n / 8) ^ (mr & kSwz)) << 4) + 2 * (n % 8));
        uint16_t* dst = out + mr * a.out_stride + n;
        if (n + 3 < cols) {
          *(uint2*)dst = w;
        } else {
          const uint16_t bits[4] = {(uint16_t)w.x, (uint16_t)(w.x >> 16), (uint16_t)w.y, (uint16_t)(w.y >> 16)};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < cols) dst[e] = bits[e];
        }
      }
    } else {
      for (int idx = threadIdx.x; idx < rows * NT; idx += T::kThreads) {
        const int mr = idx / NT, n = idx % NT;
        if (n < cols)
          out[mr * a.out_stride + n] =
              *(const uint16_t*)(lds + mr * (2 * NT) + (((n / 8) ^ (mr & kSwz)) << 4) + 2 * (n % 8));
      }
    }
  }
  if (!a.best) return;
  for (int mr = threadIdx.x; mr < rows; mr += T::kThreads) {
    TileBest b = red[mr * WN];
#pragma unroll
    for (int w = 1; w < WN; ++w) {
      const TileBest o = red[mr * WN + w];
      if (better(o.val, o.idx, b.val, b.idx)) b = o;
    }
    a.best[(int64_t)(m0 + mr) * a.tiles_n + nt] = pack_best(b.val, b.idx, nt * NT);
  }
}

// The workgroup shapes, smallest first: the larger, the less is loaded per MFMA (row_plan chooses). Tile32x64 has a
// form for ranges that are multiples of its 16 register sets (Qwen3-8B's projections): with the check behind every
// step 4096 x 12288 takes 42.0 us at 80 rows, with one in 16 steps 39.0, without ranges 38.2. Tile256x32 loads 3 steps
// ahead, so that a CU holds three of its workgroups and 594 (the LM head) are one round: 151936 x 1024 at one row 54.9 us
// with 7 steps ahead and two workgroups, 51.9 with 3; 151936 x 4096 194.1 and 191.7.
typedef Tile<1, 4, 2, 1, 16, 9, false, false, true, 16> Tile32x64E16;
typedef Tile<1, 4, 2, 1, 16, 9, false, false, true> Tile32x64;
typedef Tile<1, 5, 2, 1, 16, 9, false, false, true> Tile32x80;
typedef Tile<1, 5, 4, 1, 8, 6, false, false, true> Tile64x80;
typedef Tile<2, 4, 4, 1, 8, 6, false, false, true> Tile128x64;
typedef Tile<2, 5, 4, 1, 8, 6, false, false, true> Tile128x80;
typedef Tile<2, 10, 4, 1, 8, 6, false, true, false> Tile128x160;
typedef Tile<4, 2, 4, 1, 4, 6, false, false, true> Tile256x32;
typedef Tile<4, 8, 4, 1, 4, 6, true, true, false> Tile256x128;
typedef Tile<4, 10, 4, 1, 4, 6, true, true, true> Tile256x160;
typedef Tile<4, 16, 4, 1, 4, 4, true, false, false, 0> Tile256x256;

}  // namespace lmhead
}  // namespace sd
