// Weight intake (FP8Linear.load_weight, inference/fp8.py:164-166): the row
// quantizer of quantize_rows (inference/fp8_weights.py:16-19) over a
// checkpoint's bf16 or fp32 weight, writing the row-major codes, the scales
// and the tiled copy the GEMMs read in one pass.
//
// Bound: HBM. The weight is read once and each layout of the codes written
// once (4 bytes per bf16 element, 6 per fp32 element). As separate passes --
// quantize into a temporary, copy it into the module's buffer, retile that
// copy -- a bf16 element moved 7 bytes, and the retiling pass stored 16-byte
// pieces 256 bytes apart (94 us of the 212 us that a 24576 x 4096 bf16 weight
// took; now 78 us, 5.15 TB/s, where a 2 GiB device copy reaches 4.9).
//
// A workgroup takes 8 rows, WR waves per row, so that each 128-byte line of a
// fragment (8 rows x 16 bytes) is written by one store instruction. A lane
// owns 16-element units (unit = p + 64 WR i for its position p in the row),
// kept in registers between the maximum and the encode where they fit
// (CACHED), else loaded again; a unit's 16 codes go to the row-major row as
// they are and through LDS into fragment order. The LDS slot of (unit, row) is
// unit * 8 + (row ^ unit % 8): the writes of 8 consecutive lanes (one row, 8
// units) and the reads (8 rows of one unit) both cover all banks.
#include "fp8_common.h"
#include "kernels.h"

namespace jv {

namespace {

constexpr int kLoadRows = 8;

// 16 elements of a row: their magnitude maximum (bf16 patterns, or fp32
// patterns) and their codes.
template <typename T>
struct Unit;

template <>
struct Unit<uint16_t> {
  uint4 v[2];
  __device__ __forceinline__ void load(const uint16_t* p) {
    v[0] = *reinterpret_cast<const uint4*>(p);
    v[1] = *reinterpret_cast<const uint4*>(p + 8);
  }
  __device__ __forceinline__ uint32_t magnitude() const {
    uint32_t am = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      am = pk_max_chunk(am, v[i]);
    }
    return max(am & 0xFFFFu, am >> 16);
  }
  static __device__ __forceinline__ float scale(uint32_t bits) { return scale_from_amax_bits(bits); }
  static constexpr uint32_t kInf = 0x7F80u;
  __device__ __forceinline__ uint4 encode(float scale, float r, bool fast) const {
    const uint2 a = encode8(v[0], scale, r, fast), b = encode8(v[1], scale, r, fast);
    return uint4{a.x, a.y, b.x, b.y};
  }
};

template <>
struct Unit<float> {
  float4 v[4];
  __device__ __forceinline__ void load(const float* p) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const float4*>(p + 4 * i);
  }
  __device__ __forceinline__ uint32_t magnitude() const {
    uint32_t am = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) am = max(am, __float_as_uint(f[j]) & 0x7FFFFFFFu);
    }
    return am;
  }
  // NaN patterns sort above infinity; a NaN row's scale is the canonical NaN.
  static __device__ __forceinline__ float scale(uint32_t bits) {
    return scale_from_amax_f32(__uint_as_float(bits > 0x7F800000u ? 0x7FC00000u : bits));
  }
  static constexpr uint32_t kInf = 0x7F800000u;
  // The IEEE quotient: the correction that replaces it for bf16 elements is
  // proven for bf16 pairs only, and the division hides under the loads.
  __device__ __forceinline__ uint4 encode(float scale, float, bool fast) const {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float q[4] = {v[i].x / scale, v[i].y / scale, v[i].z / scale, v[i].w / scale};
      if (fast) {
        int c = cvt_pk_fp8<false>(q[0], q[1], 0);
        w[i] = (uint32_t)cvt_pk_fp8<true>(q[2], q[3], c);
      } else {
        w[i] = e4m3_encode_sw(q[0]) | (e4m3_encode_sw(q[1]) << 8) | (e4m3_encode_sw(q[2]) << 16) |
               (e4m3_encode_sw(q[3]) << 24);
      }
    }
    return uint4{w[0], w[1], w[2], w[3]};
  }
};

// Rows [8 blockIdx.x, +8) of x [N, K] (K % 16 == 0; with `tiled`, K % 128 ==
// 0 and N % 16 == 0). NU units per lane cover the row: NU * WR * 1024 >= K.
template <typename T, int WR, int NU, bool CACHED, bool TILED>
__global__ __launch_bounds__(64 * WR * kLoadRows) void load_rows_kernel(const T* __restrict__ x, int64_t ldx, int N, int K,
                                                                        uint8_t* __restrict__ codes, int64_t ldc,
                                                                        float* __restrict__ scales,
                                                                        uint8_t* __restrict__ tiled) {
  constexpr int LANES = 64 * WR;  // positions in a row
  __shared__ uint32_t red[kLoadRows * WR];
  __shared__ uint4 stage[TILED ? 2 : 1][TILED ? LANES * kLoadRows : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = wave / WR, p = (wave % WR) * 64 + lane;
  const int row0 = blockIdx.x * kLoadRows;
  const int row = min(row0 + r, N - 1);
  const int units = K >> 4;
  const T* xr = x + (int64_t)row * ldx;

  Unit<T> u[CACHED ? NU : 1];
  uint32_t am = 0;
  // A repeated unit past the row's end does not change the maximum, so every
  // load is unconditional and they go out together.
  if constexpr (CACHED) {
#pragma unroll
    for (int i = 0; i < NU; ++i) u[i].load(xr + (int64_t)min(p + i * LANES, units - 1) * 16);
#pragma unroll
    for (int i = 0; i < NU; ++i) am = max(am, u[i].magnitude());
  } else {
#pragma unroll 4
    for (int i = 0; i < NU; ++i) {
      u[0].load(xr + (int64_t)min(p + i * LANES, units - 1) * 16);
      am = max(am, u[0].magnitude());
    }
  }
  am = wave_max_u32(am);
  if constexpr (WR > 1) {
    if (lane == 0) red[wave] = am;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WR; ++w) am = max(am, red[r * WR + w]);
  }
  const float scale = Unit<T>::scale(am);
  const bool fast = am < Unit<T>::kInf;
  const float rcp = 1.0f / scale;
  const bool real = row0 + r < N;
  if (p == 0 && real) scales[row] = scale;

  uint8_t* cr = codes + (int64_t)row * ldc;
  const int ksteps = K >> 7;
  uint8_t* tr = TILED ? tiled + (int64_t)(row0 >> 4) * ksteps * 2048 + (row0 & 8) * 16 : nullptr;
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    if (i * LANES >= units) break;  // uniform over the workgroup
    const int unit = p + i * LANES;
    if constexpr (!CACHED) u[0].load(xr + (int64_t)min(unit, units - 1) * 16);
    const uint4 c = u[CACHED ? i : 0].encode(scale, rcp, fast);
    if (unit < units && real) *reinterpret_cast<uint4*>(cr + (int64_t)unit * 16) = c;
    if constexpr (TILED) {
      stage[i & 1][p * kLoadRows + (r ^ (p & 7))] = c;
      // One barrier per unit: the next unit stages into the other buffer, and
      // the barrier after it orders this unit's reads before the buffer's reuse.
      lds_barrier();
      const int pu = tid >> 3, rr = tid & 7, un = pu + i * LANES;
      if (un < units) {
        // (k % 128) / 16 = un % 8: its bit 0 is the half, the rest the quarter.
        const int64_t off = ((int64_t)(un >> 3) * 2 + (un & 1)) * 1024 + ((un & 7) >> 1) * 256 + rr * 16;
        *reinterpret_cast<uint4*>(tr + off) = stage[i & 1][pu * kLoadRows + (rr ^ (pu & 7))];
      }
    }
  }
}

template <typename T, int WR, int NU, bool CACHED>
hipError_t launch_load(const T* x, int64_t ldx, int64_t N, int K, uint8_t* codes, int64_t ldc, float* scales,
                       uint8_t* tiled, hipStream_t stream) {
  const dim3 grid((unsigned)((N + kLoadRows - 1) / kLoadRows)), block(64 * WR * kLoadRows);
  if (tiled)
    load_rows_kernel<T, WR, NU, CACHED, true><<<grid, block, 0, stream>>>(x, ldx, (int)N, K, codes, ldc, scales, tiled);
  else
    load_rows_kernel<T, WR, NU, CACHED, false><<<grid, block, 0, stream>>>(x, ldx, (int)N, K, codes, ldc, scales, nullptr);
  return hipGetLastError();
}

}  // namespace

// One wave per row up to K = 4096 (four units of 16 elements per lane), two
// above; fp32 rows past 8192 elements do not fit the registers of 16 waves
// and are read twice (the second time mostly from the Infinity Cache).
hipError_t load_rows_bf16(const uint16_t* x, int64_t ldx, int64_t N, int K, uint8_t* codes, int64_t ldc, float* scales,
                          uint8_t* tiled, hipStream_t stream) {
  if (N == 0) return hipSuccess;
  if (K <= 0 || K > kLoadMaxCols || (K & 15) || (tiled && ((K & 127) || (N & 15)))) return hipErrorInvalidValue;
  if (K <= 2048) return launch_load<uint16_t, 1, 2, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  if (K <= 4096) return launch_load<uint16_t, 1, 4, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  if (K <= 8192) return launch_load<uint16_t, 2, 4, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  return launch_load<uint16_t, 2, 8, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
}

hipError_t load_rows_f32(const float* x, int64_t ldx, int64_t N, int K, uint8_t* codes, int64_t ldc, float* scales,
                         uint8_t* tiled, hipStream_t stream) {
  if (N == 0) return hipSuccess;
  if (K <= 0 || K > kLoadMaxCols || (K & 15) || (tiled && ((K & 127) || (N & 15)))) return hipErrorInvalidValue;
  if (K <= 2048) return launch_load<float, 1, 2, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  if (K <= 4096) return launch_load<float, 1, 4, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  if (K <= 8192) return launch_load<float, 2, 4, true>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
  return launch_load<float, 2, 8, false>(x, ldx, N, K, codes, ldc, scales, tiled, stream);
}

}  // namespace jv
