// Pieces shared by the dense-layer kernels (projections on MFMA): the matrix
// instructions, a launch's parameters, the epilogues and four-element packets.
#pragma once

#include "common.cuh"

namespace rlse {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct DenseMma;
template <>
struct DenseMma<bf16> {
  static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
};
template <>
struct DenseMma<f16> {
  static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
};
// f32 (the reference CPU path's dtype): a 16-byte operand load holds four
// floats, so a k step spans 16 elements, lane l holding elements
// 4*(l/16) .. +3 of its row. v_mfma_f32_16x16x4_f32 number m takes each
// lane's element m, for A and B alike: its four k indices are 4g + m over
// the lane groups g, and the four products cover the step. The accumulator
// layout is the 16-bit products' (lane l: D[4*(l/16) + v][l%16]).
template <>
struct DenseMma<float> {
  static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[m]), __uint_as_float(b[m]), c, 0,
                                               0, 0);
    return c;
  }
};
// Elements of one k step (four lanes groups' 16-byte loads) and of one
// lane's load.
template <typename T>
__host__ __device__ constexpr int dense_step_elems() { return 64 / (int)sizeof(T); }

enum : int { kEpiStore = 0, kEpiQkv = 1, kEpiResidual = 2, kEpiSiluMul = 3 };

struct DenseParams {
  const void* x;     // [rows][K]
  const void* w;     // [N][K]
  const void* bias;  // [N] or null (kEpiStore, kEpiQkv)
  void* out0;        // y [rows][N] | q [rows][n1] | x_res [rows][N] | act [rows][n1]
  void* out1;        // k [rows][n2 - n1] (kEpiQkv)
  void* out2;        // v [rows][N - n2] (kEpiQkv)
  // KS > 1: sticky error flags, one launch counter per wave slot
  // (kDenseCtrWords) and (tile groups) x (KS - 1) records of FT*RT*256
  // tagged 64-bit words.
  uint32_t* ws_err;
  uint32_t* ws_ctr;
  uint64_t* ws_rec;
  unsigned long long wait_ticks;
  int rows, K, N, n1, n2;
  int ksplit;        // KS
  int steps;         // 32-wide k steps per wave
  int packed;        // w in the tile order rlse_dense_pack writes
  int xpacked;       // x in the packed row order (RLSE_PACKED_ROWS)
  int opacked;       // kEpiSiluMul: act in the packed row order (RLSE_PACKED_OUT)
  const void* norm_w;  // RMSNorm weight [K]: x is the raw residual (null: x as it is)
  void* norm_h;        // [whole 16-row tiles][K], where the norm is a launch of its own
  float eps, inv_k;
};

template <typename T>
__device__ __forceinline__ void load4(const T* p, float* v) {
  if constexpr (sizeof(T) == 4) {
    const float4 u = *reinterpret_cast<const float4*>(p);
    v[0] = u.x;
    v[1] = u.y;
    v[2] = u.z;
    v[3] = u.w;
  } else {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    const uint4 q = make_uint4(u.x, u.y, 0, 0);
    float t[8];
    Packet<T>::unpack(q, t);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = t[e];
  }
}

template <typename T>
__device__ __forceinline__ void store4(T* p, const float* v) {
  if constexpr (sizeof(T) == 4)
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  else
    *reinterpret_cast<uint2*>(p) = make_uint2(Packet<T>::pack2(v[0], v[1]),
                                              Packet<T>::pack2(v[2], v[3]));
}

// out[r][i] = silu(gate[r][i]) * up[r][i] with gate_up = [rows][2*inter]
// (gate columns, then up columns): silu(v) = v / (1 + exp(-v)) rounded per
// op (exp, the sum, the quotient), then the product rounded.
template <typename T>
__device__ __forceinline__ float silu_mul_rounded(float g, float u) {
#pragma clang fp contract(off)
  const float e = round_cvt<T>(expf(-g));
  const float s = round_cvt<T>(g / round_cvt<T>(1.f + e));
  return s * u;
}

// The tiled kernel of dense_tile.hip: kEpiQkv, kEpiResidual and kEpiSiluMul
// over more rows than a decode batch (bf16/f16, the entry points' checks done).
int launch_dense_tile(int epi, int dtype, const DenseParams& p, hipStream_t s);

}  // namespace rlse
