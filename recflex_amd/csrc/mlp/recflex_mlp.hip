// The MLP behind the fused embedding (RecomModel): Linear + ReLU layers and a last Linear to one
// unit with a sigmoid, to fp32's precision on the matrix cores.
//
// Reference counterpart: the nn.Sequential of RecFlex/rec_modules.py:150-179.
//
// A batch of 512 through 4408 -> 1024 -> 256 -> 128 -> 1 is 5 GFLOP, 32 us at the rate a large fp32
// product reaches here (154 TFLOP/s), and most of it the first layer.  Library products with
// activations between them are eight launches and, one after the other in a graph, 77 us; batches
// of 1, 64 and 256 take 55, 54 and 89 us.  Here they are three launches (four where the first
// layer's K is split) and 64 us; 25, 31 and 46 us for the smaller batches:
//   gemm_nt    a layer: X [M, K] times W [N, K] transposed, bias and ReLU on the way out;
//   tail       the last hidden layer, its ReLU, the dot product with the last layer's row and
//              the sigmoid, and ahead of them the sum of the K-splits of the layer before.
// Where a layer has too few tiles for the device its K is split over workgroups; the splits' sums
// go to a buffer and are added in order (tail, or reduce_splits for an earlier layer): the result
// does not depend on which workgroup ends first.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "recflex_mlp.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// x, or 0 where x is not positive; a NaN stays one
__device__ __forceinline__ float relu(const float x) { return x <= 0.f ? 0.f : x; }

// ---------------------------------------------------------------------------------------------
// gemm_nt: a workgroup of eight wavefronts computes a tile of 32 or 64 rows x 64 units of fp32 products on
// the bf16 matrix cores: every operand is the sum of three bf16 numbers (8 + 8 + 8 bits with their signs
// hold the 24 exactly), and of their nine products all but that of the low parts (at most 2^-34) are formed.
// Those of the high parts have a sum of their own, in which the others would be cut off: a matrix instruction
// rounds down what it adds (measured, by up to one unit in the last place).  So one product alone comes out as
// fp32 rounds it, and long sums are rounded less often than fp32 products would be.
// Errors against 64 bits, 2-norm, first hidden layer, as fp32 products and so: 4 408 inputs, 512 rows 5.9e-7 and
// 1.1e-7, one row 2.0e-7 and 1.0e-7; 23 980 inputs, 512 rows 6.9e-7 and 2.3e-7; one active input per row 2.5e-8
// both, at most 6.0e-8 both.  (With six of the products and one sum: 2.6e-7, 1.4e-7, 6.6e-7, and 3.3e-8, at most
// 1.6e-7, for 59 us of the whole MLP at 4 408 inputs and 512 rows where this takes 64.)
// The wavefronts split K among them, each with the whole tile to itself: no operand is taken apart twice
// and they meet once, to add up their sums.  A step's operands (16 of K) go through the wavefront's own LDS (as
// loaded: rows of 64 bytes; as read: a lane's eight of a row) and are taken apart in registers.
// 512 rows, 4 408 -> 1 024 units: 57 us as fp32 products, 46 and 5 for the sum of two splits so.  The whole MLP at 512
// rows, 4 408 and 23 980 inputs: 68 and 240 us, 65 and 235 so.
// Bound by the two kinds of instructions, which hardly overlap: the matrix cores are busy 35 % of the time and the
// vector units 38 %, of a wavefront's time 15 % goes to waiting for memory (4 408 inputs, 512 rows).  Without the
// conversions the MLP takes 61 us instead of 66, without the loads 58, with three products of the eight 54.
// N and K are multiples of 4 (valid): a vector of four units is whole or beyond N.
// ---------------------------------------------------------------------------------------------
constexpr int kTileN = 64, kThreads = 512, kWaves = kThreads / 64, kStep = 16;
constexpr int kRedRow = kTileN + 4;
// Of numbers between these (and zeros) the three parts are exact and no product of parts leaves fp32's range or nears
// its subnormals.  A step with others is left out and taken as fp32 products at the end: at 4 408 inputs and 512
// rows 98 us for the MLP with such a number in every step, 65 without (fp32 products throughout: 68).  The question
// costs a vector instruction per number, and three where there are zeros.
constexpr float kSmallest = 0x1p-60f, kLargest = 0x1p60f;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Eight {
  f32x4 v[2];
  __device__ __forceinline__ float operator[](const int i) const { return v[i / 4][i % 4]; }
};

// eight fp32 numbers as high + middle + low
struct Parts { bf16x8 high, middle, low; };
__device__ __forceinline__ Parts parts_of(const Eight &v) {
  u32x4 part[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x = v[2 * i], y = v[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      // (the builtin and not the instruction by hand: its result goes to a matrix instruction, and the
      // compiler keeps the two wait states between them only where it knows the writer)
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2));
      part[p][i] = w;
      x -= __uint_as_float(w << 16);
      y -= __uint_as_float(w & 0xffff0000u);
    }
  }
  return {__builtin_bit_cast(bf16x8, part[0]), __builtin_bit_cast(bf16x8, part[1]), __builtin_bit_cast(bf16x8, part[2])};
}

// the wavefront's own LDS: what it wrote before what it reads next, and the other way round
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// TM rows
template <int TM>
__global__ void __launch_bounds__(kThreads)
gemm_nt(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
        float *__restrict__ out, const int M, const int N, const int K, const int splits) {
  constexpr int ROWS = TM + kTileN, LANES = kStep / 4, LOADS = ROWS * LANES / 64, WM = TM / 32, WN = kTileN / 32;
  constexpr int ROW = kStep + 4;                 // LDS row, in floats: 16-byte reads of 8 rows spread over all banks
  constexpr int LDS = kWaves * ROWS * ROW > kWaves * TM * kRedRow ? kWaves * ROWS * ROW : kWaves * TM * kRedRow;
  __shared__ float lds[LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_n = (N + kTileN - 1) / kTileN;
  const int tiles = tiles_n * ((M + TM - 1) / TM);
  const int split = blockIdx.x / tiles, tile = blockIdx.x - split * tiles;
  // consecutive workgroups (one XCD each) take the units of the same rows: an XCD keeps to an
  // eighth of the weights, the larger operand
  const int m0 = tile / tiles_n * TM, n0 = tile % tiles_n * kTileN;
  const int steps = (K + kStep - 1) / kStep;
  const int per_split = (steps + splits - 1) / splits;
  const int first = split * per_split, last = min(steps, first + per_split);

  // rows beyond M or N repeat the last one (their sums are not stored); K beyond the end reads 0
  const int col = lane % LANES * 4;
  const float *src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (i * 64 + lane) / LANES;
    src[i] = (i * 64 / LANES < TM ? x + static_cast<int64_t>(min(m0 + row, M - 1)) * K
                          : w + static_cast<int64_t>(min(n0 + row - TM, N - 1)) * K) + col;
  }
  f32x4 next[LOADS];
  auto request = [&](const int step) {
    const int k = min(step * kStep, K - 4 - col);     // stays within the row
#pragma unroll
    for (int i = 0; i < LOADS; ++i) next[i] = *reinterpret_cast<const f32x4 *>(src[i] + k);
  };
  float *mine = lds + wave * (ROWS * ROW);
  // what was requested, to LDS; whether the parts hold all of it, the same in every lane
  auto put = [&](const int step) {
    if (step * kStep + kStep > K) {              // the last step's surplus
      const bool in = step * kStep + col < K;
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) next[i][j] = in ? next[i][j] : 0.f;
    }
    float least = kLargest, most = 0.f;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      *reinterpret_cast<f32x4 *>(mine + (i * 64 + lane) / LANES * ROW + col) = next[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        least = fminf(least, fabsf(next[i][j]));
        most = __builtin_elementwise_maximum(most, fabsf(next[i][j]));        // (a NaN stays)
      }
    }
    bool fits = most < kLargest;
    if (__builtin_amdgcn_ballot_w64(!(least >= kSmallest)) != 0) {            // zeros, or small numbers
      unsigned lowest = ~0u;
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)                                           // (a zero becomes the largest)
          lowest = min(lowest, (__float_as_uint(next[i][j]) << 1) - 1u);
      fits = fits && lowest >= (__float_as_uint(kSmallest) << 1) - 1u;
    }
    return __builtin_amdgcn_ballot_w64(!fits) == 0;
  };

  // the products of the high parts (and fp32 products), and the others
  f32x16 acc[WM][WN], rest[WM][WN];
#pragma unroll
  for (int m = 0; m < WM; ++m)
#pragma unroll
    for (int n = 0; n < WN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[m][n][r] = rest[m][n][r] = 0.f;
  // lane (i, h) of a 32x32x16 product holds row i at eight values of k, one set per h (of eight 32x32x2 products
  // one value each)
  const float *frag = mine + (lane & 31) * ROW + (lane >> 5) * 8;
  auto operand = [&](const int block) {
    const float *at = frag + block * 32 * ROW;
    return Eight{*reinterpret_cast<const f32x4 *>(at), *reinterpret_cast<const f32x4 *>(at + 4)};
  };
  bool left_out = false;
  if (first + wave < last) request(first + wave);
  for (int step = first + wave; step < last; step += kWaves) {
    const bool fits = put(step);
    if (step + kWaves < last) request(step + kWaves);
    wave_lds_fence();
    if (__builtin_expect(fits, 1)) {
      Parts a[WM], b[WN];
#pragma unroll
      for (int n = 0; n < WN; ++n) b[n] = parts_of(operand(WM + n));
#pragma unroll
      for (int m = 0; m < WM; ++m) a[m] = parts_of(operand(m));
      auto add = [](f32x16 &sum, const bf16x8 p, const bf16x8 q) {
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p, q, sum, 0, 0, 0);
      };
#pragma unroll
      for (int m = 0; m < WM; ++m) {             // smallest first, neighbours in the row on different sums
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].middle, b[n].low);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].low, b[n].middle);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].middle, b[n].middle);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].high, b[n].low);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].low, b[n].high);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].high, b[n].middle);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(rest[m][n], a[m].middle, b[n].high);
#pragma unroll
        for (int n = 0; n < WN; ++n) add(acc[m][n], a[m].high, b[n].high);
      }
    } else {
      left_out = true;
    }
    wave_lds_fence();
  }
  // The steps left out: infinities, NaN, numbers beyond kSmallest and kLargest.
  if (__builtin_expect(left_out, 0))
    for (int step = first + wave; step < last; step += kWaves) {
      request(step);
      if (put(step)) continue;
      wave_lds_fence();
#pragma unroll
      for (int m = 0; m < WM; ++m) {
        const Eight a = operand(m);
#pragma unroll
        for (int n = 0; n < WN; ++n) {
          const Eight b = operand(WM + n);
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc[m][n], 0, 0, 0);
        }
      }
      wave_lds_fence();
    }

  // the wavefronts' shares of K, added in order
  __syncthreads();
#pragma unroll
  for (int m = 0; m < WM; ++m)
#pragma unroll
    for (int n = 0; n < WN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m * 32 + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
        lds[(wave * TM + row) * kRedRow + n * 32 + (lane & 31)] = acc[m][n][r] + rest[m][n][r];
      }
  __syncthreads();
  for (int at = tid; at < TM * (kTileN / 4); at += kThreads) {
    const int row = at / (kTileN / 4), unit = at % (kTileN / 4) * 4;
    f32x4 sum = *reinterpret_cast<const f32x4 *>(lds + row * kRedRow + unit);
#pragma unroll
    for (int g = 1; g < kWaves; ++g)
      sum += *reinterpret_cast<const f32x4 *>(lds + (g * TM + row) * kRedRow + unit);
    if (m0 + row >= M || n0 + unit >= N) continue;
    float *dst = out + (static_cast<int64_t>(split) * M + m0 + row) * N + n0 + unit;
    if (bias) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] = relu(sum[j] + bias[n0 + unit + j]);
    }
    *reinterpret_cast<f32x4 *>(dst) = sum;
  }
}

// The splits' sums at p, p + stride, ..., added in order; kAhead loads at a time, because each comes from
// beyond this XCD's L2 (the whole MLP, 1 / 37 rows with 16 and 8 splits: 25.7 / 34.1 us one after the
// other, 22.1 / 29.4 us this way; 512 rows with four splits ahead of the tail 65.7 and 65.0).
constexpr int kAhead = 4;
template <typename V>
__device__ __forceinline__ V sum_splits(const float *__restrict__ p, const int64_t stride, const int splits) {
  V sum = {};
  for (int s = 0; s < splits; s += kAhead) {
    V part[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      part[j] = *reinterpret_cast<const V *>(p + min(s + j, splits - 1) * stride);
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (s + j < splits) sum += part[j];
  }
  return sum;
}

// out = ReLU(bias + the splits' sums, in order)
__global__ void __launch_bounds__(256)
reduce_splits(const float *__restrict__ parts, const float *__restrict__ bias, float *__restrict__ out,
              const int64_t count, const int N, const int splits) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    out[i] = relu(sum_splits<float>(parts + i, count, splits) + bias[i % N]);
  }
}

// ---------------------------------------------------------------------------------------------
// tail: 16 rows a workgroup.  Its input (K <= kTailMaxK) stays in LDS, the last hidden layer's
// weights (N <= kTailMaxN units) come through LDS in chunks, wavefront w computes the units
// 16 w .. 16 w + 15, and what leaves is one number per row.  A matter of latencies -- 32 workgroups
// for a batch of 512 --, worth it because its three steps would be three launches.
// ---------------------------------------------------------------------------------------------
constexpr int kTailRows = 16, kTailMaxN = RECFLEX_MLP_TAIL_MAX_UNITS, kTailMaxK = RECFLEX_MLP_TAIL_MAX_INPUTS;
constexpr int kTailChunk = 128, kTailRow = kTailChunk + 4;
constexpr int kTailLoads = kTailMaxN * (kTailChunk / 4) / kThreads;
static_assert(kTailMaxN == kThreads / 64 * 16, "16 units per wavefront");

__global__ void __launch_bounds__(kThreads)
tail(const float *__restrict__ parts, const int splits, const float *__restrict__ bias0,
     float *__restrict__ hidden0, const float *__restrict__ w, const float *__restrict__ bias,
     float *__restrict__ hidden, const float *__restrict__ w_last, const float *__restrict__ b_last,
     float *__restrict__ out, const int M, const int N, const int K) {
  __shared__ float xs[kTailRows * (kTailMaxK + 4)];
  __shared__ float ws[kTailMaxN * kTailRow];
  __shared__ float dots[kThreads / 64][kTailRows];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.x * kTailRows;
  const int padded = (K + kTailChunk - 1) / kTailChunk * kTailChunk;   // <= kTailMaxK
  const int stride = padded + 4;

  f32x4 next[kTailLoads];
  auto request = [&](const int k0) {
#pragma unroll
    for (int i = 0; i < kTailLoads; ++i) {
      const int at = i * kThreads + tid, row = at / (kTailChunk / 4), k = k0 + at % (kTailChunk / 4) * 4;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (k < K) v = *reinterpret_cast<const f32x4 *>(w + static_cast<int64_t>(min(row, N - 1)) * K + k);
      next[i] = v;
    }
  };
  request(0);

  // the input: the splits of the layer before, its bias and ReLU
  const int64_t count = static_cast<int64_t>(M) * K;
  for (int at = tid; at < kTailRows * (padded / 4); at += kThreads) {
    const int row = at / (padded / 4), k = (at - row * (padded / 4)) * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (m0 + row < M && k < K) {
      const int64_t i = static_cast<int64_t>(m0 + row) * K + k;
      v = sum_splits<f32x4>(parts + i, count, splits);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = relu(v[j] + bias0[k + j]);
      if (hidden0) *reinterpret_cast<f32x4 *>(hidden0 + i) = v;
    }
    *reinterpret_cast<f32x4 *>(xs + row * stride + k) = v;
  }

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < padded; k0 += kTailChunk) {
#pragma unroll
    for (int i = 0; i < kTailLoads; ++i) {
      const int at = i * kThreads + tid;
      *reinterpret_cast<f32x4 *>(ws + at / (kTailChunk / 4) * kTailRow + at % (kTailChunk / 4) * 4) = next[i];
    }
    __syncthreads();
    if (k0 + kTailChunk < padded) request(k0 + kTailChunk);
    const float *xf = xs + (lane & 15) * stride + k0 + (lane >> 4) * 4;
    const float *wf = ws + (wave * 16 + (lane & 15)) * kTailRow + (lane >> 4) * 4;
#pragma unroll
    for (int s = 0; s < kTailChunk / 16; ++s) {
      const f32x4 a = *reinterpret_cast<const f32x4 *>(xf + s * 16);
      const f32x4 b = *reinterpret_cast<const f32x4 *>(wf + s * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc, 0, 0, 0);
    }
    __syncthreads();                            // before the next chunk takes this one's place
  }

  // lane: unit wave * 16 + lane % 16, rows (lane / 16) * 4 + r
  const int unit = wave * 16 + (lane & 15);
  const float b = unit < N ? bias[unit] : 0.f, wl = unit < N ? w_last[unit] : 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = (lane >> 4) * 4 + r;
    const float h = relu(acc[r] + b);
    if (hidden && unit < N && m0 + row < M) hidden[static_cast<int64_t>(m0 + row) * N + unit] = h;
    float d = unit < N ? h * wl : 0.f;
    d += __shfl_xor(d, 8, 64);
    d += __shfl_xor(d, 4, 64);
    d += __shfl_xor(d, 2, 64);
    d += __shfl_xor(d, 1, 64);
    if ((lane & 15) == 0) dots[wave][row] = d;
  }
  __syncthreads();
  if (tid < kTailRows && m0 + tid < M) {
    float z = dots[0][tid];
#pragma unroll
    for (int v = 1; v < kThreads / 64; ++v) z += dots[v][tid];
    out[m0 + tid] = 1.f / (1.f + expf(-(z + b_last[0])));
  }
}

int ceil_div(const int64_t a, const int64_t b) { return static_cast<int>((a + b - 1) / b); }

// How a layer is cut: tiles of 32 or 64 rows, and its K into splits.  A CU takes 1.4 us (32 rows) or 2.4 us (64 rows)
// for a chunk (16 of K for every wavefront) with all CUs at work, and 3 us for the first loads and the last sums.
// Splits cost their traffic and, ahead of any layer but the tail, a kernel that adds them up; that traffic is priced
// high, so the chunks are priced lower than they measure, in their proportion: over 1 to 512 rows and the first
// layers 512, 1 000, 4 408, 12 000, 23 980 x 1 024 to 8 192 the better number of rows is taken to within 3 % of the
// whole MLP (with 1.4 and 2.4 here, 4 408 x 1 024 and 512 rows would go unsplit: 69 us instead of 65).
struct Plan { int rows, splits; };
Plan plan_of(const int M, const int N, const int K, const int cus, const bool feeds_tail) {
  Plan best{32, 1};
  double best_us = 1e30;
  for (int rows = 32; rows <= 64; rows += 32) {
    const int64_t tiles = static_cast<int64_t>(ceil_div(M, rows)) * ceil_div(N, kTileN);
    const int chunks = ceil_div(K, kWaves * kStep);
    for (int s = 1; s <= RECFLEX_MLP_MAX_SPLITS && s <= chunks; ++s) {
      const int per_split = ceil_div(chunks, s);
      if (static_cast<int64_t>(per_split) * (s - 1) >= chunks) continue;            // an empty split
      const double chunk_us = rows == 32 ? 1.2 : 1.9;
      double us = (chunk_us * per_split + 3.) * ceil_div(tiles * s, cus);
      if (s > 1) us += (feeds_tail ? 0. : 3.) + 2. * s * M * N * 4 / 4e6;
      if (us < best_us * 0.98) { best = {rows, s}; best_us = us; }
    }
  }
  return best;
}

struct Device { int id, cus; };
hipError_t current_device(Device *d) {
  static int cus[64];                           // written with the same value by whoever is first
  hipError_t e = hipGetDevice(&d->id);
  if (e != hipSuccess) return e;
  if (d->id < 0 || d->id >= 64) return hipErrorInvalidDevice;
  int n = __atomic_load_n(&cus[d->id], __ATOMIC_RELAXED);
  if (n <= 0) {
    e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, d->id);
    if (e != hipSuccess) return e;
    __atomic_store_n(&cus[d->id], n, __ATOMIC_RELAXED);
  }
  d->cus = n;
  return hipSuccess;
}

bool valid(const recflex_mlp_args *a) {
  if (!a || a->batch < 0 || a->layers < 2 || a->layers > RECFLEX_MLP_MAX_LAYERS || !a->x) return false;
  for (int l = 0; l <= a->layers; ++l) {
    if (a->units[l] <= 0 || !a->weights[l] || !a->biases[l]) return false;
    if (l < a->layers && (a->units[l] % 4 || reinterpret_cast<uintptr_t>(a->weights[l]) % 16)) return false;
  }
  return reinterpret_cast<uintptr_t>(a->x) % 16 == 0 &&
         a->units[a->layers] <= kTailMaxN && a->units[a->layers - 1] <= kTailMaxK;
}

} // namespace

extern "C" int recflex_mlp_workspace_floats(const recflex_mlp_args *a, int64_t *floats) {
  if (!valid(a) || !floats) return static_cast<int>(hipErrorInvalidValue);
  Device d;
  const hipError_t e = current_device(&d);
  if (e != hipSuccess) return static_cast<int>(e);
  int64_t most = 0;
  for (int l = 0; l + 1 < a->layers; ++l) {
    const int s = plan_of(a->batch, a->units[l + 1], a->units[l], d.cus, l + 2 == a->layers).splits;
    const int64_t need = static_cast<int64_t>(s) * a->batch * a->units[l + 1];
    if ((s > 1 || l + 2 == a->layers) && need > most) most = need;
  }
  *floats = most;
  return 0;
}

extern "C" int recflex_mlp_forward(const recflex_mlp_args *a) {
  if (!valid(a) || !a->out || !a->workspace || reinterpret_cast<uintptr_t>(a->workspace) % 16)
    return static_cast<int>(hipErrorInvalidValue);
  for (int l = 0; l + 2 < a->layers; ++l)       // the tail's input needs no buffer of its own
    if (!a->hidden[l] || reinterpret_cast<uintptr_t>(a->hidden[l]) % 16) return static_cast<int>(hipErrorInvalidValue);
  if (reinterpret_cast<uintptr_t>(a->hidden[a->layers - 2]) % 16) return static_cast<int>(hipErrorInvalidValue);
  if (a->batch == 0) return 0;
  Device d;
  hipError_t e = current_device(&d);
  if (e != hipSuccess) return static_cast<int>(e);
  hipStream_t stream = static_cast<hipStream_t>(a->stream);
  auto launch = [&](const void *kernel, int64_t blocks, int threads, void **args) {
    if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    return hipLaunchKernel(kernel, dim3(static_cast<unsigned>(blocks)), dim3(threads), args, 0, stream);
  };
  int M = a->batch;
  const float *x = a->x;
  int splits = 1;
  for (int l = 0; l + 1 < a->layers; ++l) {
    int K = a->units[l], N = a->units[l + 1];
    const bool feeds_tail = l + 2 == a->layers;
    const Plan plan = plan_of(M, N, K, d.cus, feeds_tail);
    splits = plan.splits;
    const bool direct = splits == 1 && !feeds_tail;
    const float *w = a->weights[l], *bias = direct ? a->biases[l] : nullptr;
    float *out = direct ? a->hidden[l] : a->workspace;
    void *args[] = {&x, &w, &bias, &out, &M, &N, &K, &splits};
    const int64_t tiles = static_cast<int64_t>(ceil_div(M, plan.rows)) * ceil_div(N, kTileN);
    const void *kernel = plan.rows == 32 ? reinterpret_cast<const void *>(&gemm_nt<32>)
                                         : reinterpret_cast<const void *>(&gemm_nt<64>);
    e = launch(kernel, tiles * splits, kThreads, args);
    if (e != hipSuccess) return static_cast<int>(e);
    if (!direct && !feeds_tail) {
      int64_t count = static_cast<int64_t>(M) * N;
      const float *parts = a->workspace;
      bias = a->biases[l];
      out = a->hidden[l];
      void *rargs[] = {&parts, &bias, &out, &count, &N, &splits};
      const int64_t blocks = (count + 255) / 256;
      e = launch(reinterpret_cast<const void *>(reduce_splits), blocks > 4096 ? 4096 : blocks, 256, rargs);
      if (e != hipSuccess) return static_cast<int>(e);
    }
    x = feeds_tail ? a->workspace : a->hidden[l];
  }
  const int t = a->layers - 1;                  // the last hidden layer
  int K = a->units[t], N = a->units[t + 1];
  const float *bias0 = a->biases[t - 1], *w = a->weights[t], *bias = a->biases[t];
  const float *w_last = a->weights[t + 1], *b_last = a->biases[t + 1];
  float *hidden0 = a->hidden[t - 1], *hidden = a->hidden[t], *out = a->out;
  void *args[] = {&x, &splits, &bias0, &hidden0, &w, &bias, &hidden, &w_last, &b_last, &out, &M, &N, &K};
  return static_cast<int>(launch(reinterpret_cast<const void *>(tail), ceil_div(M, kTailRows), kThreads, args));
}
