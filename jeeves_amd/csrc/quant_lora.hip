// The per-token quantizer with the LoRA down-projection for prefill batches:
// quant_row (quant_row.h) over two rows per workgroup.
//
// Bound: the reads of A. One row per workgroup reads all 16 x K of A for each
// row: 128 KB of L2 traffic beside 8 KB of x at K = 4096, 1 MB per CU at 2048
// rows. Here each 16-byte piece of A, once in registers, serves two rows
// (graphs of back-to-back launches, us, one row -> two: K = 4096 at 1024 /
// 2048 / 8000 rows 10.6 / 18.7 / 61.6 -> 9.3 / 15.2 / 45.2, K = 12288 at 512 /
// 2048 / 8000 15.8 / 47.0 / 158.6 -> 14.5 / 39.1 / 119.6). Four rows hold too
// many registers: within 10 % either way at K <= 4096 and slower above. On the
// matrix cores (16 rows x 16 ranks, A turned through LDS) 2048 rows of 4096
// took 11.9 us, but t's error against 64 bits grew by half (1.15e-7 from
// 7.9e-8), so the products stay here.
// Codes, scales and the order of each row's sums are quant_row's, so the bits
// do not depend on which of the two a batch takes.
#include "quant_row.h"

namespace jv {

namespace {

constexpr int kThreads = 256, kRank = 16, ROWS = 2;

// NC 8-element chunks per thread and row: K <= NC * 8 * 256.
template <int NC, bool PACKED>
__global__ __launch_bounds__(kThreads) void quant_lora_kernel(const uint16_t* __restrict__ x, int64_t ldx, int K, int M,
                                                              uint8_t* __restrict__ codes, int64_t ldc,
                                                              float* __restrict__ scales,
                                                              const uint16_t* __restrict__ lora_a,
                                                              float* __restrict__ lora_t) {
  constexpr int NW = kThreads / 64;
  __shared__ uint32_t red_max[ROWS][NW];
  __shared__ float red_t[ROWS][NW][kRank];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nchunks = K >> 3;
  const int row0 = packed_tile_row<ROWS>((int)blockIdx.x, (M + 15) >> 4);
  if (row0 < 0 || (!PACKED && row0 >= M)) return;  // the whole workgroup

  uint4 v[ROWS][NC];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int i = 0; i < NC; ++i)
      v[r][i] = *reinterpret_cast<const uint4*>(x + (int64_t)min(row0 + r, M - 1) * ldx +
                                                (int64_t)min(tid + i * kThreads, nchunks - 1) * 8);
  float t[ROWS][kRank];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int q = 0; q < kRank; ++q) t[r][q] = 0.0f;
  // A by 8 ranks of a chunk at a time, the next batch in flight under this
  // one's products (as quant_row).
  constexpr int RB = 8, NB = kRank / RB, G = NC * NB;
  uint4 ab[2][RB];
  auto load_a = [&](int g, uint4(&dst)[RB]) {
    const int c = min(tid + (g / NB) * kThreads, nchunks - 1), r0 = (g % NB) * RB;
#pragma unroll
    for (int b = 0; b < RB; ++b) dst[b] = *reinterpret_cast<const uint4*>(lora_a + (r0 + b) * (int64_t)K + (int64_t)c * 8);
  };
  load_a(0, ab[0]);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (g + 1 < G) load_a(g + 1, ab[(g + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
    const int i = g / NB;
    if (tid + i * kThreads < nchunks) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) lora_accumulate<kRank, RB>(t[r], v[r][i], ab[g & 1], (g % NB) * RB);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    uint32_t am = 0;
    // A repeated last chunk does not change the maximum.
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      am = pk_max_chunk(am, v[r][i]);
    }
    am = wave_max_u32(max(am & 0xFFFFu, am >> 16));
    if (lane == 0) red_max[r][wave] = am;
    const float s = lora_wave_sum<kRank>(t[r], lane);
    if (lane < kRank) red_t[r][wave][lane] = s;
  }
  __syncthreads();
  if (tid < ROWS * kRank) {
    const int r = tid / kRank, q = tid % kRank;
    float sum = red_t[r][0][q];
#pragma unroll
    for (int w = 1; w < NW; ++w) sum += red_t[r][w][q];
    if (row0 + r < M) lora_t[(int64_t)(row0 + r) * kRank + q] = sum;
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int row = row0 + r;
    const bool real = row < M;
    uint32_t amax_bits = red_max[r][0];
#pragma unroll
    for (int w = 1; w < NW; ++w) amax_bits = max(amax_bits, red_max[r][w]);
    amax_bits = __builtin_amdgcn_readfirstlane(amax_bits);
    const float scale = scale_from_amax_bits(amax_bits);
    if (tid == 0 && real) scales[row] = scale;
    const bool fast = amax_bits < 0x7F80u;
    const float rcp = 1.0f / scale;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = tid + i * kThreads;
      if (c >= nchunks || !(PACKED || real)) continue;
      uint8_t* out = codes + (PACKED ? packed_x_offset(row, c * 8, K >> 7) : (int64_t)row * ldc + (int64_t)c * 8);
      *reinterpret_cast<uint2*>(out) = real ? encode8(v[r][i], scale, rcp, fast) : uint2{0u, 0u};
    }
  }
}

template <int NC, bool PACKED>
hipError_t launch(const uint16_t* x, int64_t ldx, int64_t M, int K, uint8_t* codes, int64_t ldc, float* scales,
                  const uint16_t* lora_a, float* lora_t, hipStream_t stream) {
  const int64_t tiles = (M + 15) / 16;
  quant_lora_kernel<NC, PACKED><<<dim3((unsigned)((tiles + 7) / 8 * 8 * (16 / ROWS))), dim3(kThreads), 0, stream>>>(
      x, ldx, K, (int)M, codes, ldc, scales, lora_a, lora_t);
  return hipGetLastError();
}

template <bool PACKED>
hipError_t launch_chunks(const uint16_t* x, int64_t ldx, int64_t M, int K, uint8_t* codes, int64_t ldc, float* scales,
                         const uint16_t* lora_a, float* lora_t, hipStream_t stream) {
  if (K <= 2048) return launch<1, PACKED>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
  if (K <= 4096) return launch<2, PACKED>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
  if (K <= 8192) return launch<4, PACKED>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
  if (K <= 12288) return launch<6, PACKED>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
  return launch<8, PACKED>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
}

}  // namespace

hipError_t quant_lora_bf16(const uint16_t* x, int64_t ldx, int64_t M, int K, uint8_t* codes, int64_t ldc, float* scales,
                           const uint16_t* lora_a, float* lora_t, bool packed, hipStream_t stream) {
  if (M <= kDecodeMaxRows || K <= 0 || (K & 7) || (packed && (K & 127)) || K > 16384) return hipErrorInvalidValue;
  return packed ? launch_chunks<true>(x, ldx, M, K, codes, 0, scales, lora_a, lora_t, stream)
                : launch_chunks<false>(x, ldx, M, K, codes, ldc, scales, lora_a, lora_t, stream);
}

}  // namespace jv
