// Token GEMM for long prompts on the block-scaled FP6 x FP4 MFMA of gfx950
// (reference: kernels/ternary.cu:688-784, entry points gemm_tile_* with
// GEMM_ARGS; the reference uses dp4a).
//
// y[t, r] = s_x[t] * sum_g P[t, r, g] * scale[r, g] (+ bias[r]), where
// P[t, r, g] = sum over the 128 inputs of group g of (code - 1) * q is exact.
//
// Why not int8 MFMA here: its int32 tiles need a conversion and an fmaf per
// output and group, and those VALU instructions, not the matrix cores, bound
// gemm_wide_kernel.  v_mfma_scale_f32_32x32x64_f8f6f4 accumulates in fp32, so
// P arrives as a float and only the fmaf is left, and it takes operands that
// hold both factors exactly:
//   * an int8 value q = s * (16 h + l), s its sign, h in 0..8, l in 0..15: the
//     FP6 (E2M3) numbers s*h/8 and s*l/8 (their codes are the integers
//     themselves), weighted by the block scales 2^6 and 2^2;
//   * a ternary weight as the FP4 (E2M1) number -2, 0 or +2: bit 3 (sign) is
//     the inverse of the code's high bit, bit 2 (magnitude) that of its low
//     bit, so a packed word gives two FP4 words in three VALU instructions
//     (a zero weight may come out as -0, which adds nothing).
// Every product and partial sum is an integer below 2^15, exact in fp32, so
// P, and with it the fmaf chain in ascending group order, is that of the int8
// kernels bit for bit.  FP6 x FP4 runs at twice the int8 rate, which pays for
// the two halves of q.
//
// lay_out_operands_kernel writes into the caller's workspace, in the order the
// blocks below read them: the two FP6 forms of the token rows (192 bytes per
// token and group), the packed weights as [64-input chunk][row] pieces of 16
// bytes, and the group scales as [group][row].  Read in place, a block takes
// 32 bytes of each of its weight rows per group, so every 128-byte line is
// fetched four times from L2, and each scale costs a line of its own; that
// bounded the kernel (K=4096 -> N=14336 at M=2048: 172 us against 138 on the
// laid-out weights, two stages).
//
// gemm_scaled_kernel: a block of four waves owns 64 tokens x 128 NT rows, a wave
// 64 tokens x 32 NT rows as 2 x NT tiles of 32 x 32 (NT = 1, 2 or 3).  Three
// stages in LDS (two blocks, 154 KB with NT = 3, on a CU), filled by direct buffer-to-LDS loads with two
// groups in flight, one barrier per group.  Per tile and group four MFMAs (two
// halves of the 128 inputs, high and low part) with the previous tile's 16
// fmaf between them.
// Measured (one MI355X, graph replays, the lay-out's 10 us included, the int8
// kernel before): K=4096 -> N=14336 at M=2048 168 -> 137 us (1.75 POPS); K=4096
// -> N=22016 at M=777 123 -> 93; K=11008 -> N=4096 at M=777 72 -> 55.
// What bounds it (counters at K=4096 -> N=14336, M=2048): one MFMA per 69 cycles
// and SIMD over the dispatch, of which it takes 32; an instruction is in issue in
// 68% of the cycles (MFMA and VALU 48%; 6.4 VALU per MFMA, 4 of them the fold,
// 1.5 the expansion), and the two waves of a SIMD, which meet at a barrier per
// group, wait for LDS, memory or it in 19% of theirs.  No bank conflicts.
// Without its loads the kernel still takes 92% of the time; without the copies
// of operands and the per-group addresses of an earlier form it gained 8%.
#include <type_traits>

#include "buffer_ops.hpp"
#include "internal.hpp"
#include "ternary_device.hpp"

namespace ivo {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kSplitGroupBytes = 192;  // FP6 high and low parts of one token's group
constexpr int kScaledTokens = 64;
constexpr int block_rows(int row_tiles) { return 128 * row_tiles; }  // four waves of 32-row tiles

// Rows of the laid-out weights and scales: whole 16-byte pieces of scales.
__host__ __device__ constexpr int row_pitch(int rows) { return (rows + 7) & ~7; }
// Groups of laid-out scales: whole rounds of the kernel's three steps, zeros past the last group.
__host__ __device__ constexpr int padded_groups(int groups) { return (groups + 2) / 3 * 3; }

// Sign-magnitude FP6 codes of four int8 values at six bits each (24 bits):
// the high parts (|q| >> 4) and the low parts (|q| & 15), each with q's sign.
__device__ __forceinline__ unsigned pack6(unsigned bytes) {
  const unsigned pairs = (bytes & 0x003F003Fu) | ((bytes >> 2) & 0x0FC00FC0u);
  return (pairs & 0xFFFu) | ((pairs >> 4) & 0xFFF000u);
}
__device__ __forceinline__ void split6(unsigned q, unsigned& high, unsigned& low) {
  const unsigned sign = (q >> 7) & 0x01010101u;
  const unsigned magnitude = (q ^ ((sign << 8) - sign)) + sign;  // per byte: |q| <= 128
  high = pack6(((magnitude >> 4) & 0x0F0F0F0Fu) | (sign << 5));
  low = pack6((magnitude & 0x0F0F0F0Fu) | (sign << 5));
}

// The three parts of the lay-out, by block index: first the scales, a 64 x 64
// tile through LDS each; then the weights, 64 rows x 16 chunks each; then the
// tokens, one thread per 32 inputs (blk 0..3) of a token's group.  The FP4 form
// of a packed word has its codes in the order: fields 0 and 2 of bytes 0..3,
// then fields 1 and 3; the q8 quad of the same 16 inputs holds field k in word
// k, so interleaving the bytes of words 0 and 2, then of 1 and 3, gives that
// order.  A group's 192 bytes: the first 16 bytes of the eight FP6 runs (blk,
// high/low), then their last 8 bytes, a run pair to a 16-byte piece, its halves
// swapped by token bit 4 and the run's lane half (a wave's reads of one half
// then fall on distinct LDS banks).
struct LayOut {
  const int8_t* q8;
  const uint8_t* packed;
  const uint16_t* scales;
  unsigned char* rows6;
  uint4* weights;      // [2 * groups][pitch]
  uint16_t* scales_t;  // [padded_groups][pitch]
  int m, chunks, groups, rows, pitch, row_bytes, scale_stride, scale_blocks, weight_blocks;
};

__global__ __launch_bounds__(256) void lay_out_operands_kernel(LayOut a) {
  __shared__ __align__(16) uint4 tile[64][17];
  const int tid = threadIdx.x;
  int b = (int)blockIdx.x;
  const int row_tiles = (a.pitch + 63) / 64;
  if (b < a.scale_blocks) {
    uint16_t(*t)[66] = reinterpret_cast<uint16_t(*)[66]>(&tile[0][0]);
    const int r0 = b % row_tiles * 64, g0 = b / row_tiles * 64;
    const int lane = tid & 63, part = tid >> 6;
    uint16_t v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = min(r0 + 4 * i + part, a.rows - 1), g = min(g0 + lane, a.groups - 1);
      v[i] = a.scales[(size_t)row * a.scale_stride + g];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) t[4 * i + part][lane] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int g = g0 + 4 * i + part, row = r0 + lane;
      if (g < padded_groups(a.groups) && row < a.pitch)
        a.scales_t[(size_t)g * a.pitch + row] = g < a.groups ? t[lane][4 * i + part] : (uint16_t)0;
    }
    return;
  }
  b -= a.scale_blocks;
  if (b < a.weight_blocks) {
    const int r0 = b % row_tiles * 64, u0 = b / row_tiles * 16;
    uint4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = i * 256 + tid;
      const int row = min(r0 + (s >> 4), a.rows - 1), u = min(u0 + (s & 15), a.chunks - 1);
      v[i] = *reinterpret_cast<const uint4*>(a.packed + (size_t)row * a.row_bytes + (size_t)u * 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) tile[(i * 256 + tid) >> 4][tid & 15] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = i * 256 + tid;
      const int row = r0 + (s & 63), u = u0 + (s >> 6);
      if (row < a.pitch && u < 2 * a.groups) a.weights[(size_t)u * a.pitch + row] = tile[s & 63][s >> 6];
    }
    return;
  }
  b -= a.weight_blocks;
  const unsigned item = b * 256u + tid;  // the launcher keeps m * groups * 192 below 2^31
  if (item >= (unsigned)a.m * a.groups * 4) return;
  const int blk = (int)(item & 3);
  const unsigned tg = item >> 2;  // token * groups + group
  const int t = (int)(tg / (unsigned)a.groups), g = (int)(tg - (unsigned)t * a.groups);
  const int u = 2 * g + (blk >> 1);
  uint4 quads[2] = {};
  if (u < a.chunks) {
    const uint4* src = reinterpret_cast<const uint4*>(a.q8 + ((size_t)t * a.chunks + u) * kChunk) + 2 * (blk & 1);
    quads[0] = src[0];
    quads[1] = src[1];
  }
  unsigned high[6], low[6];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const unsigned w[4] = {quads[i].x, quads[i].y, quads[i].z, quads[i].w};
    const unsigned ordered[4] = {
        __builtin_amdgcn_perm(w[2], w[0], 0x05010400u), __builtin_amdgcn_perm(w[2], w[0], 0x07030602u),
        __builtin_amdgcn_perm(w[3], w[1], 0x05010400u), __builtin_amdgcn_perm(w[3], w[1], 0x07030602u)};
    unsigned h[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) split6(ordered[k], h[k], l[k]);
    high[3 * i] = h[0] | (h[1] << 24);
    high[3 * i + 1] = (h[1] >> 8) | (h[2] << 16);
    high[3 * i + 2] = (h[2] >> 16) | (h[3] << 8);
    low[3 * i] = l[0] | (l[1] << 24);
    low[3 * i + 1] = (l[1] >> 8) | (l[2] << 16);
    low[3 * i + 2] = (l[2] >> 16) | (l[3] << 8);
  }
  uint4* dst = reinterpret_cast<uint4*>(a.rows6 + (size_t)tg * kSplitGroupBytes);
  dst[2 * blk] = make_uint4(high[0], high[1], high[2], high[3]);
  dst[2 * blk + 1] = make_uint4(low[0], low[1], low[2], low[3]);
  dst[8 + blk] = ((t >> 4) ^ (blk >> 1)) & 1 ? make_uint4(low[4], low[5], high[4], high[5])
                                             : make_uint4(high[4], high[5], low[4], low[5]);
}

// Block -> output tile: each of the 8 XCDs (block b runs on XCD b % 8) takes a
// run of consecutive tiles, and a run walks bands of 8 token tiles with the
// token tile fastest, so the blocks that are on an XCD together (64) read 8
// token tiles and 8 row tiles through its L2.
constexpr int kScaledXcds = 8;
constexpr int kBand = 8;
__device__ __forceinline__ void scaled_tile(int nx, int ny, int& tile_x, int& tile_y) {
  const int nb = nx * ny, b = blockIdx.x;
  const int q = nb / kScaledXcds, r = nb % kScaledXcds;
  const int xcd = b % kScaledXcds, idx = b / kScaledXcds;
  const int t = xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
  const int band = t / (nx * kBand), in_band = t - band * nx * kBand;
  const int height = min(kBand, ny - band * kBand);
  tile_x = in_band / height;
  tile_y = band * kBand + in_band % height;
}

// ~w & mask in one instruction.
__device__ __forceinline__ int inverse_bits(unsigned w, unsigned mask) {
  int d;
  asm("v_bfi_b32 %0, %1, 0, %2" : "=v"(d) : "v"(w), "s"(mask));
  return d;
}

template <int NT>
struct ScaledStage {
  static constexpr int kRows = block_rows(NT);
  static constexpr int kTail = kScaledTokens * 128;            // after 8 head pieces of 16 bytes per token
  static constexpr int kWeights = kTail + kScaledTokens * 64;  // after 4 tail pieces per token
  static constexpr int kScales = kWeights + kRows * 32;        // after 2 pieces of weights per row
  static constexpr int kBytes = kScales + 1024;                // fp16 per row
  static_assert(kRows * 2 <= 1024, "one wave instruction of scales");
};

template <int EPI, int NT>
__global__ __launch_bounds__(256, 2) void gemm_scaled_kernel(const unsigned char* __restrict__ rows6,
                                                             const uint4* __restrict__ weights_t,
                                                             const uint16_t* __restrict__ scales_t,
                                                             const float* __restrict__ scale_in,
                                                             const float* __restrict__ bias,
                                                             float* __restrict__ output, GemmArgs a, int nx, int ny) {
  using S = ScaledStage<NT>;
  constexpr int kScaledRows = S::kRows, kWaveRows = 32 * NT;
  __shared__ __align__(16) unsigned char stages[3][S::kBytes];
  __shared__ __align__(16) float token_scales[kScaledTokens];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, half = lane >> 5;
  const int groups = (a.n + kGroup - 1) / kGroup;
  int tile_x, tile_y;
  scaled_tile(nx, ny, tile_x, tile_y);
  const int token0 = tile_y * kScaledTokens;
  const int row0 = tile_x * kScaledRows;
  const int pitch = row_pitch(a.rows);
  const v4u q_buf = wide_buffer(rows6, (long long)a.m * groups * kSplitGroupBytes);
  const v4u w_buf = wide_buffer(weights_t, (long long)groups * pitch * 32);
  const int step_groups = padded_groups(groups);
  const v4u s_buf = wide_buffer(scales_t, (long long)step_groups * pitch * 2);

  // Direct-to-LDS loads of a thread per group: two head pieces (slot
  // s = j*256 + tid: token s >> 3, piece (s & 7) ^ a_swizzle), one tail piece
  // (token tid >> 2, piece (tid & 3) ^ (token >> 2 & 3)) and NT pieces of
  // weights (slot s = j*256 + tid of [half][rows]); wave 0 also loads the
  // scales.  Tokens past m and rows past the pitch have a vector offset past
  // the buffer and read zeros (the scalar offset only moves by whole groups).
  constexpr int kPast = 0x7FFFFFF0;
  const int token_bytes = groups * kSplitGroupBytes;
  const int head_off = (token0 + (tid >> 3)) * token_bytes + ((tid & 7) ^ a_swizzle(tid >> 3)) * 16;
  const int tail_off = (token0 + (tid >> 2)) * token_bytes + 128 + ((tid & 3) ^ ((tid >> 4) & 3)) * 16;
  int w_off[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int s = j * 256 + tid, h = s >= kScaledRows, row = row0 + s - h * kScaledRows;
    w_off[j] = row < pitch ? (h * pitch + row) * 16 : kPast;
  }
  static_assert(kScaledRows * 2 == NT * 256, "whole pieces of weights per thread");
  const int s_off = row0 + lane * 8 < pitch ? row0 * 2 + lane * 16 : kPast;
  constexpr int kLoads = 3 + NT;  // per group, and one more in wave 0
  const unsigned lds_base = __builtin_amdgcn_readfirstlane(lds_address(&stages[0][0]) + wave * 1024);
  auto load = [&](int g, int stage) {
    const unsigned base = lds_base + stage * S::kBytes;
    const int scale_group = min(g, step_groups - 1);
    g = min(g, groups - 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(q_buf, base + j * 4096, head_off + j * 32 * token_bytes, g * kSplitGroupBytes);
    dma16(q_buf, base + S::kTail, tail_off, g * kSplitGroupBytes);
#pragma unroll
    for (int j = 0; j < NT; ++j) dma16(w_buf, base + S::kWeights + j * 4096, w_off[j], g * pitch * 32);
    if (wave == 0) dma16(s_buf, base + S::kScales, s_off, scale_group * pitch * 2);
  };

  v16f acc[2][NT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = v16f{};
  // The previous tile's P and scale, folded while the next tile's MFMAs run
  // (zero before the first: a fold of zeros leaves acc at +0).
  v16f prev{};
  float prev_sc = 0.0f;

  // LDS read addresses of the lane in stage 0, token c of a 32-token tile, its
  // 32-input blocks 2*half and 2*half + 1: run k = 2 * (block & 1) + (0 high, 1
  // low); weight row c, the 16 packed bytes of the same 64 inputs.  Stage, token
  // tile and row tile are instruction offsets.
  const unsigned char* lds = &stages[0][0];
  const unsigned char *head_read[4], *tail_read[2][4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    head_read[k] = lds + c * 128 + (((4 * half + k) ^ a_swizzle(c)) * 16);
    const int off = S::kTail + c * 64 + (((2 * half + (k >> 1)) ^ ((c >> 2) & 3)) * 16) +
                    ((k & 1) ^ (c >> 4) ^ half) * 8;
    // Opaque: paired with the first tile's read the second would land in
    // registers it has to be copied from.
    int second = off + 32 * 64;
    asm("" : "+v"(second));
    tail_read[0][k] = lds + off;
    tail_read[1][k] = lds + second;
  }
  const unsigned char* w_read = lds + S::kWeights + (half * kScaledRows + wave * kWaveRows + c) * 16;
  const unsigned char* s_read = lds + S::kScales + (wave * kWaveRows + c) * 2;
  constexpr int kHighScale = 0x85, kLowScale = 0x81, kOne = 0x7F;  // 2^6, 2^2, 1

  if (tid < kScaledTokens) token_scales[tid] = scale_in[min(token0 + tid, a.m - 1)];
  load(0, 0);
  load(1, 1);
  auto step = [&](int g, auto stage_c) {
    constexpr int kStage = decltype(stage_c)::value, kOffset = kStage * S::kBytes;
    // The stage of g is filled (the loads of g + 1, issued after its own, stay
    // in flight) and no wave still reads the one that g + 2 goes into: the
    // sequence of direct_load_sync with a count (past the end the last group is
    // loaded again, so the count holds to the end).
    if (wave == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads + 1) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    load(g + 2, (kStage + 2) % 3);
    uint4 raw = *reinterpret_cast<const uint4*>(w_read + kOffset);
    float sc = h2f(*reinterpret_cast<const uint16_t*>(s_read + kOffset));
    v8i q[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint4 a0 = *reinterpret_cast<const uint4*>(head_read[k] + kOffset + mt * 32 * 128);
        const uint2 a1 = *reinterpret_cast<const uint2*>(tail_read[mt][k] + kOffset);
        q[mt][k] = v8i{(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, 0, 0};
      }
    v8i w[2];
    auto expand = [&](int h) {
      const unsigned w0 = h ? raw.z : raw.x, w1 = h ? raw.w : raw.y;
      w[h] = v8i{inverse_bits(w0 << 2, 0xCCCCCCCCu), inverse_bits(w0, 0xCCCCCCCCu),
                 inverse_bits(w1 << 2, 0xCCCCCCCCu), inverse_bits(w1, 0xCCCCCCCCu), 0, 0, 0, 0};
    };
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      expand(0);
      expand(1);
      const float tile_sc = sc;
      if (nt + 1 < NT) {
        raw = *reinterpret_cast<const uint4*>(w_read + kOffset + (nt + 1) * 32 * 16);
        sc = h2f(*reinterpret_cast<const uint16_t*>(s_read + kOffset + (nt + 1) * 64));
      }
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int fold_mt = mt ^ 1, fold_nt = mt ? nt : (nt + NT - 1) % NT;
        v16f p{};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(q[mt][k], w[k >> 1], p, 2, 4, 0,
                                                              (k & 1) ? kLowScale : kHighScale, 0, kOne);
          // The fold starts behind the second MFMA: the previous tile's last
          // one has retired by then.
          constexpr int kFirst[5] = {0, 0, 6, 11, 16};
#pragma unroll
          for (int i = kFirst[k]; i < kFirst[k + 1]; ++i)
            acc[fold_mt][fold_nt][i] = __builtin_fmaf(prev[i], prev_sc, acc[fold_mt][fold_nt][i]);
          __builtin_amdgcn_sched_barrier(0);
        }
        prev = p;
        prev_sc = tile_sc;
      }
    }
    // The step's arithmetic stays in the step: left free, the compiler sinks
    // MFMAs past the next barrier and runs out of registers.
    asm volatile("" : "+v"(prev), "+v"(prev_sc));
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[mt][nt]));
  };
  // Three steps per round, so that every stage is a constant; steps past the
  // last group run it again with the zero scales laid out behind the last
  // group's: fmaf(P, 0, acc) with a finite P returns acc.
  for (int g = 0; g < groups; g += 3) {
    step(g, std::integral_constant<int, 0>{});
    step(g + 1, std::integral_constant<int, 1>{});
    step(g + 2, std::integral_constant<int, 2>{});
  }
  // No direct-to-LDS load may still be in flight when the block's LDS is handed on.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < 16; ++i)
    acc[1][NT - 1][i] = __builtin_fmaf(prev[i], prev_sc, acc[1][NT - 1][i]);

  // Epilogue.  A lane holds row c of a tile for the 16 tokens
  // 8*(i >> 2) + 4*half + (i & 3): 32 lanes write 128 contiguous bytes of an
  // output row.  Buffer accesses over the block's token rows: rows past the
  // matrix get an offset past them, tokens past m are past them, and both are
  // dropped by the range check, so nothing is predicated.
  const int live_tokens = min(a.m - token0, kScaledTokens);
  const int width = EPI == kSiluPair ? a.rows >> 1 : a.rows;
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
      output + (size_t)token0 * a.out_stride, (short)0, ((live_tokens - 1) * a.out_stride + width) * 4, 0x00020000);
  const bool has_bias = bias != nullptr;
  const int stride4 = a.out_stride * 4;
  constexpr int kStream = 2;  // non-temporal: the output is written once
  float bv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    bv[nt] = has_bias ? bias[min(row0 + wave * kWaveRows + nt * 32 + c, a.rows - 1)] : 0.0f;
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    float sx[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f4v v = *reinterpret_cast<const f4v*>(token_scales + mt * 32 + 8 * j + 4 * half);
#pragma unroll
      for (int i = 0; i < 4; ++i) sx[4 * j + i] = v[i];
    }
    const int t_off = (mt * 32 + 4 * half) * stride4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int row = row0 + wave * kWaveRows + nt * 32 + c;
      const bool live = row < a.rows;
      const int off = live ? t_off + (EPI == kSiluPair ? row >> 1 : row) * 4 : kPast;
      if constexpr (EPI == kSiluPair) {
        // A lane pair holds the gate (even lane) and the up row (odd lane) of
        // one output: the even lane finishes token i, the odd lane token i + 1,
        // each sending the other the value it lacks.
        const int odd = c & 1;
        const int pair_off = off + (live ? odd * stride4 : 0);
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          float y0 = acc[mt][nt][i] * sx[i], y1 = acc[mt][nt][i + 1] * sx[i + 1];
          if (has_bias) {
            y0 = y0 + bv[nt];
            y1 = y1 + bv[nt];
          }
          const float got = __int_as_float(pair_swap(__float_as_int(odd ? y0 : y1)));
          const float gate = odd ? got : y0, up = odd ? y1 : got;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ivo_silu(gate) * up), out,
                                                pair_off + (8 * (i >> 2) + (i & 3)) * stride4, 0, kStream);
        }
        continue;
      }
      float base[16];
      if constexpr (EPI == kResidual) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          base[i] = __uint_as_float(
              __builtin_amdgcn_raw_buffer_load_b32(out, off + (8 * (i >> 2) + (i & 3)) * stride4, 0, 0));
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float y = acc[mt][nt][i] * sx[i];
        if (has_bias) y = y + bv[nt];
        if constexpr (EPI == kResidual) y = base[i] + y;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), out, off + (8 * (i >> 2) + (i & 3)) * stride4, 0,
                                              kStream);
      }
    }
  }
}

// The workspace: FP6 rows, laid-out weights, laid-out scales, each 16-byte aligned.
struct ScaledWork {
  size_t weights, scales, bytes;
};
ScaledWork scaled_work(int m, int rows, int n) {
  const size_t groups = ceil_div(n, kGroup), pitch = row_pitch(rows);
  ScaledWork w;
  w.weights = (size_t)m * groups * kSplitGroupBytes;
  w.scales = w.weights + groups * pitch * 32;
  w.bytes = w.scales + padded_groups((int)groups) * pitch * 2;
  return w;
}

template <int EPI, int NT>
hipError_t launch_scaled_shape(hipStream_t stream, const GemmArgs& a, const LayOut& l) {
  const int nx = ceil_div(a.rows, block_rows(NT)), ny = ceil_div(a.m, kScaledTokens);
  hipLaunchKernelGGL((gemm_scaled_kernel<EPI, NT>), dim3(nx * ny), dim3(256), 0, stream, l.rows6, l.weights, l.scales_t,
                     a.scale_in, a.bias, a.output, a, nx, ny);
  return hipGetLastError();
}

template <int EPI>
hipError_t launch_scaled_epi(hipStream_t stream, const GemmArgs& a, const LayOut& l, int row_tiles) {
  switch (row_tiles) {
    case 1: return launch_scaled_shape<EPI, 1>(stream, a, l);
    case 2: return launch_scaled_shape<EPI, 2>(stream, a, l);
    default: return launch_scaled_shape<EPI, 3>(stream, a, l);
  }
}

// Time (us) of one group step of a kernel whose blocks go two to a CU, by the blocks that are left: with one
// block on one CU, one on every CU, two on one CU, two on every CU.
struct StepTimes {
  float one, all, second, both;
};

// Time of a group step over `blocks` blocks: whole rounds of two blocks per CU, then the rest.  A rest past
// one block per CU makes a step: the CUs that hold two blocks take the pair's time, however few they are.
float round_time(long long blocks, int cus, const StepTimes& t) {
  const long long rest = blocks % (2 * cus);
  const float whole = (float)(blocks / (2 * cus)) * t.both;
  if (rest == 0) return whole;
  if (rest <= cus) return whole + t.one + (t.all - t.one) * (float)rest / (float)cus;
  return whole + t.second + (t.both - t.second) * (float)(rest - cus) / (float)cus;
}

}  // namespace

// Row tiles per wave (1, 2 or 3: blocks of 128, 256 or 384 rows), 0 where the
// int8 kernel is expected to finish first: prompts that gemm_wide_kernel would
// take with 2048 inputs and more.  The expected time of either kernel is a
// constant plus a group step's time over its blocks (round_time) times the
// groups; for this kernel the constant is 11.8 us (launch, prologue, epilogue,
// the lay-out's launch) and the lay-out's bytes at 10 TB/s.  Narrow blocks cost
// more per output and win where wide ones leave CUs idle.  Fitted on 257 shapes
// of 128..4096 tokens (graph replays, weights warm, one MI355X) with a mean error
// of 4%.  On those the choice is on average 0.3% slower than the best, at worst
// 14%, and at worst 1% slower than the int8 kernel; on 181 others of random sizes
// 0.6%, 12% and 1.5%.  Some (us; int8, then 1, 2, 3 row tiles, lay-out included):
//   4096 -> 14336, 2048: 168; 150, 137, 141     4096 -> 22016, 777: 123; 101, 101, 93
//   4096 -> 12288, 777: 78; 61, 66, 59          11008 -> 4096, 777: 72; 55, 64, 80
//   8192 -> 8192, 2048: 179; 171, 155, 167      4096 -> 4096, 777: 30; 30, 34, 40
//   4096 -> 4096, 2048: 55; 57, 50, 60          4096 -> 14336, 514: 76; 53, 47, 56
//   2048 -> 6144, 1024: 28; 29, 29, 30          4096 -> 12288, 300: 31; 31, 34, 40
// (Charging a partly filled round the time of a full one, the rule took two row
// tiles for 11008 -> 4096 and for 4096 -> 4096 at 777, 13% behind the int8 kernel
// at worst.)
// Below 2048 inputs the comparison is not made (1024 -> 4096, 2048: int8 17;
// 22, 21, 23).
int gemm_scaled_row_tiles(int m, int rows, int n) {
  const int groups = ceil_div(n, kGroup), cus = device_cus();
  const int int8_tokens = gemm_wide_tokens(m, rows, n);
  const long long limit = 0x7FFFFFF0LL;  // 32-bit buffer offsets, a tile of slack
  if (int8_tokens < 64 || groups < 16 || (m + (long long)kScaledTokens) * groups * kSplitGroupBytes >= limit ||
      (rows + (long long)block_rows(3)) * groups * 32 >= limit)
    return 0;
  const long long int8_blocks = (long long)ceil_div(rows, 256) * ceil_div(m, int8_tokens);
  const float int8_time = int8_tokens == 128
                              ? 7.9f + (float)groups * round_time(int8_blocks, cus, {0.885f, 1.36f, 2.13f, 2.6f})
                              : 4.75f + (float)groups * round_time(int8_blocks, cus, {0.43f, 0.88f, 1.31f, 1.85f});
  float best = 0.97f * int8_time;  // no change for less than the fit's error
  const float lay_out = 11.8f + ((float)m * 320.0f + (float)rows * 68.0f) * (float)groups / 10.0e6f;
  constexpr StepTimes kStep[3] = {
      {0.124f, 0.277f, 0.396f, 0.586f}, {0.416f, 0.599f, 0.769f, 1.05f}, {0.568f, 0.889f, 1.2f, 1.51f}};
  int choice = 0;
  float times[4];
  for (int tiles = 1; tiles <= 3; ++tiles) {
    const long long blocks = (long long)ceil_div(rows, block_rows(tiles)) * ceil_div(m, kScaledTokens);
    times[tiles] = (float)padded_groups(groups) * round_time(blocks, cus, kStep[tiles - 1]) + lay_out;
    if (times[tiles] < best) {
      best = times[tiles];
      choice = tiles;
    }
  }
  // Over more than one round of blocks three tiles gain on two when the call is not repeated on the same
  // buffers (two inputs and weights in turn, quantizer included, us, two and three tiles: 4096 -> 14336 at 4096
  // tokens 278 and 273, 4096 -> 22016 at 2048 223 and 218, 8192 -> 28672 at 2048 520 and 501).
  const long long pairs = (long long)ceil_div(rows, block_rows(2)) * ceil_div(m, kScaledTokens);
  if (choice == 2 && pairs > 2LL * cus && times[3] <= 1.03f * times[2]) choice = 3;
  return choice;
}

size_t gemm_scaled_work(int m, int rows, int n) {
  return gemm_scaled_row_tiles(m, rows, n) == 0 ? 0 : scaled_work(m, rows, n).bytes;
}

hipError_t launch_gemm_scaled(hipStream_t stream, const GemmArgs& a, void* work) {
  // 32-bit buffer offsets into a block's output rows.
  if ((2 * kScaledTokens + 1LL) * a.out_stride * 4 + 4LL * a.rows >= 0x7FFFFFF0LL) return launch_gemm(stream, a);
  const int wave_tiles = gemm_scaled_row_tiles(a.m, a.rows, a.n);
  if (wave_tiles == 0) return launch_gemm(stream, a);
  const ScaledWork w = scaled_work(a.m, a.rows, a.n);
  unsigned char* base = static_cast<unsigned char*>(work);
  LayOut l{};
  l.q8 = a.q8_in;
  l.packed = a.packed;
  l.scales = a.scales;
  l.rows6 = base;
  l.weights = reinterpret_cast<uint4*>(base + w.weights);
  l.scales_t = reinterpret_cast<uint16_t*>(base + w.scales);
  l.m = a.m;
  l.chunks = ceil_div(a.n, kChunk);
  l.groups = ceil_div(a.n, kGroup);
  l.rows = a.rows;
  l.pitch = row_pitch(a.rows);
  l.row_bytes = a.row_bytes;
  l.scale_stride = a.groups;
  const int row_tiles = ceil_div(l.pitch, 64);
  l.scale_blocks = row_tiles * ceil_div(padded_groups(l.groups), 64);
  l.weight_blocks = row_tiles * ceil_div(2 * l.groups, 16);
  const int token_blocks = (int)(((long long)a.m * l.groups * 4 + 255) / 256);
  hipLaunchKernelGGL(lay_out_operands_kernel, dim3(l.scale_blocks + l.weight_blocks + token_blocks), dim3(256), 0,
                     stream, l);
  const hipError_t status = hipGetLastError();
  if (status != hipSuccess) return status;
  switch (a.epi) {
    case kStore: return launch_scaled_epi<kStore>(stream, a, l, wave_tiles);
    case kResidual: return launch_scaled_epi<kResidual>(stream, a, l, wave_tiles);
    case kSiluPair: return launch_scaled_epi<kSiluPair>(stream, a, l, wave_tiles);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ivo
