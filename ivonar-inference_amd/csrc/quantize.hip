// Per-token int8 activation quantizer (reference semantics:
// kernels/ternary.cu:148-197, quantization.py:35-38).
//
// One block owns one token row and reads it once: the row stays in registers
// from the absmax (and the sum of squares or the split-softmax merge before
// it) to the int8 values, so a row costs one memory round trip, whatever its
// mode.  Where rows are few and long, several blocks share a row's conversions
// instead, each reading the row for its absmax (few_long_rows and
// launch_plain_shape say from where on).  What bounds these kernels: for one to a dozen rows the chain of
// latencies (launch, one round trip, one or two block reductions), from some
// hundred rows on the bytes read.
//
//   * PLAIN rows that are 16-byte aligned (quantize_plain_kernel): float4 per
//     thread, up to 32768 inputs;
//   * NORM rows (quantize_norm4_kernel: float4 per thread, up to 8192 inputs;
//     quantize_row_kernel for 1024 inputs and fewer) and rows off a 16-byte
//     boundary (quantize_row_kernel, up to 8192 inputs);
//   * ATTN rows of up to 16384 inputs (quantize_attn_kernel): the softmax
//     weight of every (head, split) is formed once, in LDS, not once per input;
//   * anything longer, and few long rows of the second kind: quantize_rows_kernel,
//     one block per slice of 16 chunks, which first reduces the whole row and
//     then quantizes its slice.
//
// Measured (one MI355X, time per launch in a chain of them, before with the
// slice kernel or clamped duplicate loads -> now): 2048 x 4096 PLAIN 15.6 ->
// 7.5 us (5.6 TB/s), NORM 28.0 -> 9.1, ATTN of 4 splits 326 -> 44.5 (3.2 TB/s);
// one row of 8192 PLAIN 3.4 -> 2.5, NORM 4.3 -> 3.8, ATTN of 4 splits 60 ->
// 5.3; 777 x 11008 PLAIN 20.1 -> 10.2.
#include "internal.hpp"
#include "ternary_device.hpp"

namespace ivo {
namespace {

constexpr int kSliceChunks = kThreads / 16;  // 16 chunks, one q8 word per thread

template <int MODE>
__global__ __launch_bounds__(kThreads) void quantize_rows_kernel(QuantArgs a) {
  __shared__ float slots[64];
  const int t = blockIdx.y;
  const int chunks = (a.n + kChunk - 1) / kChunk;
  const RowSource src{a.input + (size_t)t * a.in_stride, a.aux, a.n, a.eps, a.splits, a.head_dim};
  float inv_rms;
  const float scale = row_scale<MODE>(src, inv_rms, slots);
  const int word = threadIdx.x;
  const int u = blockIdx.x * kSliceChunks + (word >> 4);
  int value = 0;
  if (u < chunks) value = quantize_word<MODE>(src, u, (word >> 2) & 3, word & 3, inv_rms, scale);
  const int total = chunk_lane_sum(word_sum(value));
  const unsigned partner = (unsigned)__builtin_amdgcn_mov_dpp(value, 0x4E, 0xF, 0xF, false);  // lane ^ 2
  if (u < chunks) {
    int32_t* q8 = reinterpret_cast<int32_t*>(a.q8 + (size_t)t * chunks * kChunk);
    q8[u * 16 + (word & 15)] = a.split ? (int)split_quad_word((unsigned)value, partner, word & 3) : value;
    if ((word & 15) == 0) a.xsum[(size_t)t * chunks + u] = total;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) a.scale[t] = scale;
}

// The q8 words, chunk sums and (thread 0) token scale of one row from its q8
// bytes: word f of the row is `word` of the calling thread, 16 consecutive
// lanes hold one chunk, and `bytes_sum` is the sum of four bytes of the same
// chunk.
__device__ __forceinline__ void store_word(const QuantArgs& a, int t, int chunks, int f, unsigned word, int bytes_sum) {
  const int total = chunk_lane_sum(bytes_sum);
  const unsigned partner = (unsigned)__builtin_amdgcn_mov_dpp((int)word, 0x4E, 0xF, 0xF, false);  // lane ^ 2
  if (f >= chunks * 16) return;  // whole chunks of 16 lanes
  reinterpret_cast<unsigned*>(a.q8 + (size_t)t * chunks * kChunk)[f] =
      a.split ? split_quad_word(word, partner, f & 3) : word;
  if ((f & 15) == 0) a.xsum[(size_t)t * chunks + (f >> 4)] = total;
}

// Max over the T threads of the block, for every thread (slots: T/64 floats).
template <int T>
__device__ __forceinline__ float block_absmax(float v, float* slots) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = v;
  __syncthreads();
  v = slots[0];
#pragma unroll
  for (int w = 1; w < T / 64; ++w) v = fmaxf(v, slots[w]);
  return v;
}

// NORM rows of up to 1024 inputs, and NORM or PLAIN rows that are not 16-byte
// aligned, of up to 256 * NB inputs.  The row and its NORM weights are read
// once into registers (quantize_row_to_lds: the reference's order of the sum
// of squares), the q8 bytes are exchanged through LDS, and thread w writes the
// q8 words w + 256 i.
template <int MODE, int NB, typename In>
__global__ __launch_bounds__(kThreads) void quantize_row_kernel(QuantArgs a) {
  __shared__ float slots[64];
  __shared__ __align__(16) unsigned char lds_q[NB * kThreads];
  const int t = blockIdx.y;
  const int chunks = (a.n + kChunk - 1) / kChunk;
  const In* row = reinterpret_cast<const In*>(a.input) + (size_t)t * a.in_stride;
  const RowSource src{reinterpret_cast<const float*>(row), a.aux, a.n, a.eps, a.splits, a.head_dim};
  const float scale = quantize_row_to_lds<MODE, NB, In, true>(src, chunks, lds_q, slots);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (NB + 3) / 4; ++i) {
    const int f = i * kThreads + threadIdx.x;
    const int u = f >> 4, w = (f >> 2) & 3, k = f & 3;
    const int value = u < chunks ? reinterpret_cast<const int*>(lds_q)[(w * chunks + u) * 4 + k] : 0;
    store_word(a, t, chunks, f, (unsigned)value, word_sum(value));
  }
  if (threadIdx.x == 0) a.scale[t] = scale;
}

// NORM rows of up to 4 * T * NC inputs, row and weights 16-byte aligned: thread
// t holds the float4 t + T c of both (four loads per thread at 8192 inputs
// where the layout above needs 64).  The sum of squares keeps the reference's
// order: the raw row goes through LDS and threads 0..255 form the chains over
// inputs t, t + 256, ..; then every thread normalises and quantizes its own.
template <int T, int NC>
__global__ __launch_bounds__(T) void quantize_norm4_kernel(QuantArgs a) {
  static_assert(T >= kThreads, "the chains take 256 threads");
  __shared__ float slots[T / 64 + 8];
  __shared__ __align__(16) float4 raw[NC * T];
  const int t = blockIdx.y, tid = threadIdx.x;
  const int n4 = a.n >> 2;
  const int chunks = (a.n + kChunk - 1) / kChunk;
  const float4* row = reinterpret_cast<const float4*>(a.input + (size_t)t * a.in_stride);
  const float4* weights = reinterpret_cast<const float4*>(a.aux);
  float4 v[NC], w[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] = row[min(c * T + tid, n4 - 1)];
#pragma unroll
  for (int c = 0; c < NC; ++c) w[c] = weights[min(c * T + tid, n4 - 1)];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c * T + tid >= n4) v[c] = float4{0.0f, 0.0f, 0.0f, 0.0f};  // zeros past the row leave the chains unchanged
    raw[c * T + tid] = v[c];
  }
  __syncthreads();
  if (tid < kThreads) {
    float s = 0.0f;
    const float* x = reinterpret_cast<const float*>(raw) + tid;
#pragma unroll
    for (int b = 0; b < 4 * T * NC / kThreads; ++b) s = __builtin_fmaf(x[b * kThreads], x[b * kThreads], s);
    s = half_wave_sum(s);
    if ((tid & 31) == 0) slots[tid >> 5] = s;
  }
  __syncthreads();
  float squares = 0.0f;
#pragma unroll
  for (int i = 0; i < kThreads / 32; ++i) squares = squares + slots[i];
  const float inv_rms = 1.0f / __builtin_sqrtf(squares / (float)a.n + a.eps);
  float amax = 0.0f;
  float e[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float x[4] = {v[c].x, v[c].y, v[c].z, v[c].w}, g[4] = {w[c].x, w[c].y, w[c].z, w[c].w};
    const bool live = c * T + tid < n4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float y = fminf(fmaxf(x[k] * inv_rms, -8.0f), 8.0f) * g[k];
      e[c][k] = live ? y : 0.0f;
      amax = fmaxf(amax, fabsf(e[c][k]));
    }
  }
  amax = block_absmax<T>(amax, slots + 8);
  const float scale = fmaxf(amax / 127.0f, 1e-5f);
  const float inv = 1.0f / scale;
  const QuadTranspose transpose(tid & 3);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const unsigned q4 = quantize4(e[c], inv, scale);
    store_word(a, t, chunks, c * T + tid, transpose.word(q4), word_sum((int)q4));
  }
  if (tid == 0) a.scale[t] = scale;
}

// 16-byte aligned PLAIN rows of up to 4 * T * NC inputs: thread t holds the
// float4 t + T c (of the values, four halves in the half types), whose four int8 values become word j = t & 3 of the quad
// after a byte transpose over its four lanes; word f of the row is then the
// thread's own, so the stores are as contiguous as the loads.  SLICED (few
// long rows): NC blocks per row, each of which takes the absmax of the whole
// row and quantizes one float4 per thread.
template <int T, int NC, bool SLICED, typename In>
__global__ __launch_bounds__(T) void quantize_plain_kernel(QuantArgs a) {
  __shared__ float slots[T / 64];
  const int t = blockIdx.y, tid = threadIdx.x;
  const int chunks = (a.n + kChunk - 1) / kChunk;
  const int n4 = a.n >> 2;
  const In* row = reinterpret_cast<const In*>(a.input) + (size_t)t * a.in_stride;
  float4 v[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] = load4(row, min(c * T + tid, n4 - 1));
  float4 mine;
  if constexpr (SLICED) mine = load4(row, min((int)blockIdx.x * T + tid, n4 - 1));
  float amax = 0.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    amax = fmaxf(fmaxf(amax, fmaxf(fabsf(v[c].x), fabsf(v[c].y))), fmaxf(fabsf(v[c].z), fabsf(v[c].w)));
  amax = block_absmax<T>(amax, slots);
  const float scale = fmaxf(amax / 127.0f, 1e-5f);
  const float inv = 1.0f / scale;
  const QuadTranspose transpose(tid & 3);
  auto quantize = [&](const float4& x, int f) {
    const bool live = f < n4;  // zeros past the row
    const float e[4] = {live ? x.x : 0.0f, live ? x.y : 0.0f, live ? x.z : 0.0f, live ? x.w : 0.0f};
    const unsigned q4 = quantize4(e, inv, scale);
    store_word(a, t, chunks, f, transpose.word(q4), word_sum((int)q4));
  };
  if constexpr (SLICED) {
    quantize(mine, (int)blockIdx.x * T + tid);
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) quantize(v[c], c * T + tid);
  }
  if (blockIdx.x == 0 && tid == 0) a.scale[t] = scale;
}

// ATTN rows of up to 4 * T * NW inputs, heads of a multiple of four inputs:
// first the softmax weight of every (head, split) and each head's weight total
// into LDS, then the merged inputs: thread t merges the inputs 4f .. 4f + 3,
// f = t + T c (one head; two 8-byte loads per split), as source_value does, in
// the same order, and the bytes are transposed as in quantize_plain_kernel.
// (Reading a q8 word's four inputs directly, 4 apart in their 16-input quad,
// needs no transpose but touches four times the cache lines per load: 54.6
// instead of 44.5 us at 2048 rows of 4096 inputs and 4 splits, 132 instead of
// 86 us at 8192 inputs.)
constexpr int kAttnLdsFloats = 12288;  // weights and totals of a row

template <int T, int NW>
__global__ __launch_bounds__(T) void quantize_attn_kernel(QuantArgs a) {
  extern __shared__ __align__(16) float lds_weights[];  // [heads * splits], then [heads] totals
  __shared__ float slots[T / 64];
  const int t = blockIdx.y, tid = threadIdx.x;
  const int splits = a.splits, quads = a.head_dim >> 2;  // float4 per head
  const int n4 = a.n >> 2;
  const int chunks = (a.n + kChunk - 1) / kChunk;
  const int stride = a.head_dim + 2;
  const int heads = n4 / quads;
  const float* row = a.input + (size_t)t * a.in_stride;
  float* totals = lds_weights + heads * splits;
  for (int p = tid; p < heads * splits; p += T) {
    const int head = splits == 1 ? p : p / splits;
    const float* base = row + (size_t)head * splits * stride;
    const float own = base[(p - head * splits) * stride];
    float peak = -__builtin_inff();
#pragma unroll 4
    for (int s = 0; s < splits; ++s) peak = fmaxf(peak, base[s * stride]);
    lds_weights[p] = own == -__builtin_inff() ? 0.0f : ivo_expf(own - peak);
  }
  __syncthreads();
  for (int head = tid; head < heads; head += T) {
    const float* base = row + (size_t)head * splits * stride + 1;
    float total = 0.0f;
#pragma unroll 4
    for (int s = 0; s < splits; ++s) total = __builtin_fmaf(lds_weights[head * splits + s], base[s * stride], total);
    totals[head] = total;
  }
  int head_of[NW];
  const float2* src[NW];
  float v[NW][4];
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    const int f = min(c * T + tid, n4 - 1);
    const int head = f / quads;
    head_of[c] = head;
    src[c] = reinterpret_cast<const float2*>(row + (size_t)head * splits * stride + 2 + 4 * (f - head * quads));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[c][e] = 0.0f;
  }
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
#pragma unroll
    for (int c = 0; c < NW; ++c) {
      const float w = lds_weights[head_of[c] * splits + s];
      const float2 lo = src[c][s * (stride >> 1)], hi = src[c][s * (stride >> 1) + 1];
      v[c][0] = __builtin_fmaf(w, lo.x, v[c][0]);
      v[c][1] = __builtin_fmaf(w, lo.y, v[c][1]);
      v[c][2] = __builtin_fmaf(w, hi.x, v[c][2]);
      v[c][3] = __builtin_fmaf(w, hi.y, v[c][3]);
    }
  }
  __syncthreads();
  float amax = 0.0f;
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    const float total = totals[head_of[c]];
    const bool live = c * T + tid < n4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[c][e] = live ? v[c][e] / total : 0.0f;  // zeros past the row
      amax = fmaxf(amax, fabsf(v[c][e]));
    }
  }
  amax = block_absmax<T>(amax, slots);
  const float scale = fmaxf(amax / 127.0f, 1e-5f);
  const float inv = 1.0f / scale;
  const QuadTranspose transpose(tid & 3);
#pragma unroll
  for (int c = 0; c < NW; ++c) {
    const unsigned q4 = quantize4(v[c], inv, scale);
    store_word(a, t, chunks, c * T + tid, transpose.word(q4), word_sum((int)q4));
  }
  if (tid == 0) a.scale[t] = scale;
}

template <int MODE, typename In = float>
bool launch_row(hipStream_t stream, const QuantArgs& a) {
  const dim3 grid(1, a.m), block(kThreads);
  // One input per thread: one division, not four values of which three are past the row (4096 NORM rows of
  // 256: 7.1 -> 5.5 us).
  if (a.n <= kThreads) hipLaunchKernelGGL((quantize_row_kernel<MODE, 1, In>), grid, block, 0, stream, a);
  else if (a.n <= 4 * kThreads) hipLaunchKernelGGL((quantize_row_kernel<MODE, 4, In>), grid, block, 0, stream, a);
  else if (a.n <= 8 * kThreads) hipLaunchKernelGGL((quantize_row_kernel<MODE, 8, In>), grid, block, 0, stream, a);
  else if (a.n <= 16 * kThreads) hipLaunchKernelGGL((quantize_row_kernel<MODE, 16, In>), grid, block, 0, stream, a);
  else if (a.n <= 32 * kThreads) hipLaunchKernelGGL((quantize_row_kernel<MODE, 32, In>), grid, block, 0, stream, a);
  else return false;
  return true;
}

// Rows from which a layout with fewer threads per row (more inputs per thread,
// fewer idle lanes at the barriers) is used: below it, one block per row leaves
// CUs idle and a row's own chain of latencies counts (500 rows of 4096 PLAIN:
// 3.5 us with 256 threads, 4.6 with 1024; 77 rows fill a third of the CUs
// either way).
constexpr int kManyRows = 256;

// Whether rows of more than `least` and up to `most` inputs go to the slice
// kernel: so few of them that `per_cu` of its blocks per CU hold all slices.
// A row's conversions are then shared by its slices, which saves more than
// their repeated reads of the row cost.  PLAIN rows off a 16-byte boundary,
// slices against one block per row: 12 x 8190 3.0 and 4.3 us, 12 x 2050 2.7 and
// 3.2, 60 x 8190 3.5 and 4.4, 150 x 8190 7.7 and 4.7; between two and four blocks
// per CU slices still finish first (100 x 8190 4.1 and 4.5) but the GEMM behind
// them then takes longer than they save (77 x 8190 -> 4100: 22.5 and 20.6).  NORM
// rows read the row three times in slices: 12 x 8190 4.5 and 5.0 us, 40 x 4096
// 3.6 and 3.9, 64 x 4097 5.6 and 5.0; read as float4 only past 3072 inputs (12 x
// 4096 3.5 and 3.7, 12 x 3072 3.6 both).
bool few_long_rows(const QuantArgs& a, int least, int most, int per_cu) {
  if (a.n <= least || a.n > most || a.m > kManyRows) return false;
  return (long long)a.m * ceil_div(a.n, kSliceChunks * kChunk) <= (long long)per_cu * device_cus();
}

bool launch_norm(hipStream_t stream, const QuantArgs& a, bool aligned) {
  const int n4 = a.n >> 2;
  if (aligned ? few_long_rows(a, 3072, 4096, 1) : few_long_rows(a, 8 * kThreads, 32 * kThreads, 1)) return false;
  if (!aligned || n4 <= 256 || (reinterpret_cast<uintptr_t>(a.aux) & 15) != 0) return launch_row<kNorm>(stream, a);
  const dim3 grid(1, a.m);
  const bool many = a.m >= kManyRows;
  if (n4 <= 512) hipLaunchKernelGGL((quantize_norm4_kernel<512, 1>), grid, dim3(512), 0, stream, a);
  else if (n4 <= 1024 && many) hipLaunchKernelGGL((quantize_norm4_kernel<256, 4>), grid, dim3(256), 0, stream, a);
  else if (n4 <= 1024) hipLaunchKernelGGL((quantize_norm4_kernel<1024, 1>), grid, dim3(1024), 0, stream, a);
  else if (n4 <= 2048 && many) hipLaunchKernelGGL((quantize_norm4_kernel<512, 4>), grid, dim3(512), 0, stream, a);
  else if (n4 <= 2048) hipLaunchKernelGGL((quantize_norm4_kernel<1024, 2>), grid, dim3(1024), 0, stream, a);
  else return false;
  return true;
}

template <int T, int NC, typename In>
void launch_plain_shape(hipStream_t stream, const QuantArgs& a) {
  // Few long rows: one CU would spend more time on a row's conversions than on
  // its absmax (12 rows of 28672: 5.4 us with one block per row, 3.5 with its
  // seven slices).  Slices past one block per CU cost more than they share out
  // (40 rows of 28672: 7.3 us in slices, 5.5 in rows; 80 of 9000: 4.1, 3.3 with
  // three slices instead of four).
  int slices = ceil_div(ceil_div(a.n, kChunk) * 16, T);
  if (NC == 4 && (long long)a.m * NC <= device_cus()) slices = NC;  // one of them empty or not: 2.9 us, 3.0 with three
  if (NC > 1 && (long long)a.m * slices <= device_cus())
    hipLaunchKernelGGL((quantize_plain_kernel<T, NC, (NC > 1), In>), dim3(slices, a.m), dim3(T), 0, stream, a);
  else
    hipLaunchKernelGGL((quantize_plain_kernel<T, NC, false, In>), dim3(1, a.m), dim3(T), 0, stream, a);
}

template <typename In>
bool launch_plain(hipStream_t stream, const QuantArgs& a) {
  const int n4 = a.n >> 2;
  const bool many = a.m >= kManyRows;
  if (n4 <= 256) launch_plain_shape<256, 1, In>(stream, a);
  else if (n4 <= 1024 && many) launch_plain_shape<256, 4, In>(stream, a);
  else if (n4 <= 1024) launch_plain_shape<1024, 1, In>(stream, a);
  else if (n4 <= 2048 && many) launch_plain_shape<512, 4, In>(stream, a);
  else if (n4 <= 2048) launch_plain_shape<1024, 2, In>(stream, a);
  else if (n4 <= 4096) launch_plain_shape<1024, 4, In>(stream, a);
  else if (n4 <= 8192) launch_plain_shape<1024, 8, In>(stream, a);
  else return false;
  return true;
}

template <int T, int NW>
void launch_attn_shape(hipStream_t stream, const QuantArgs& a, size_t lds) {
  hipLaunchKernelGGL((quantize_attn_kernel<T, NW>), dim3(1, a.m), dim3(T), lds, stream, a);
}

bool launch_attn(hipStream_t stream, const QuantArgs& a) {
  // Heads of a multiple of four inputs whose partials are read as float2.
  if ((a.head_dim & 3) != 0 || (a.in_stride & 1) != 0 || (reinterpret_cast<uintptr_t>(a.input) & 7) != 0) return false;
  const long long floats = (long long)(a.n / a.head_dim) * (a.splits + 1);
  if (floats > kAttnLdsFloats) return false;
  const size_t lds = (size_t)floats * sizeof(float);
  const bool many = a.m >= kManyRows;
  if (a.n <= 1024) launch_attn_shape<256, 1>(stream, a, lds);
  else if (a.n <= 4096 && many) launch_attn_shape<256, 4>(stream, a, lds);
  else if (a.n <= 4096) launch_attn_shape<1024, 1>(stream, a, lds);
  else if (a.n <= 8192 && many) launch_attn_shape<512, 4>(stream, a, lds);
  else if (a.n <= 8192) launch_attn_shape<1024, 2>(stream, a, lds);
  else if (a.n <= 16384) launch_attn_shape<1024, 4>(stream, a, lds);
  else return false;
  return true;
}

}  // namespace

bool quantize_half_applies(int n, const void* input) {
  return (n & 3) == 0 && (reinterpret_cast<uintptr_t>(input) & 7) == 0 ? n <= 32768 : n <= 32 * kThreads;
}

hipError_t launch_quantize(hipStream_t stream, const QuantArgs& a) {
  if (a.m <= 0) return hipSuccess;
  if (a.dtype != kFloat32) {
    if (a.mode != kPlain || a.n <= 0 || !quantize_half_applies(a.n, a.input)) return hipErrorInvalidValue;
    const bool aligned = (a.n & 3) == 0 && (a.in_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(a.input) & 7) == 0;
    bool launched = false;
    if (a.dtype == kFloat16) launched = aligned ? launch_plain<Half>(stream, a) : launch_row<kPlain, Half>(stream, a);
    if (a.dtype == kBfloat16)
      launched = aligned ? launch_plain<Bfloat>(stream, a) : launch_row<kPlain, Bfloat>(stream, a);
    return launched ? hipGetLastError() : hipErrorInvalidValue;
  }
  const int chunks = ceil_div(a.n, kChunk);
  const bool aligned = (a.n & 3) == 0 && (a.in_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(a.input) & 15) == 0;
  bool launched = false;
  switch (a.mode) {
    case kPlain:
      if (aligned) launched = launch_plain<float>(stream, a);
      else if (!few_long_rows(a, 8 * kThreads, 32 * kThreads, 2)) launched = launch_row<kPlain>(stream, a);
      break;
    case kNorm: launched = launch_norm(stream, a, aligned); break;
    case kAttn: launched = launch_attn(stream, a); break;
    default: return hipErrorInvalidValue;
  }
  if (launched) return hipGetLastError();
  const dim3 grid(ceil_div(chunks, kSliceChunks), a.m);
  switch (a.mode) {
    case kPlain: hipLaunchKernelGGL(quantize_rows_kernel<kPlain>, grid, dim3(kThreads), 0, stream, a); break;
    case kNorm: hipLaunchKernelGGL(quantize_rows_kernel<kNorm>, grid, dim3(kThreads), 0, stream, a); break;
    case kAttn: hipLaunchKernelGGL(quantize_rows_kernel<kAttn>, grid, dim3(kThreads), 0, stream, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace ivo
