// Pieces shared by the bf16 GEMM kernels (gemm.hip: verify-size rows, wgemm.hip:
// prefill-size rows), and the launcher of the latter.
#pragma once

#include "vnx_internal.h"

namespace vnx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kVgChunk = 64;  // K per chunk
constexpr int kVgXcds = 8;    // XCDs the dispatcher deals workgroups over
constexpr int kVgRowB = 128;  // bytes of one staged X row (64 bf16)

template <int OT>
__device__ __forceinline__ void vg_store(char* y, int64_t off, float v) {
  if constexpr (OT == 0) {
    reinterpret_cast<float*>(y)[off] = v;
  } else if constexpr (OT == 1) {
    reinterpret_cast<__bf16*>(y)[off] = static_cast<__bf16>(v);
  } else {
    reinterpret_cast<_Float16*>(y)[off] = static_cast<_Float16>(v);
  }
}

// Eight consecutive outputs of type OT from fp32 (16 bytes for bf16 / fp16,
// 32 for fp32); NT: 16-bit ones past the caches.
template <int OT, bool NT = false>
__device__ __forceinline__ void vg_store8(char* y, int64_t off, const float (&v)[8]) {
  if constexpr (OT == 0) {
    float* d = reinterpret_cast<float*>(y) + off;
    *reinterpret_cast<f32x4*>(d) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(d + 4) = f32x4{v[4], v[5], v[6], v[7]};
  } else if constexpr (OT == 1) {
    __bf16 t[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = static_cast<__bf16>(v[e]);
    u32x4* d = reinterpret_cast<u32x4*>(reinterpret_cast<__bf16*>(y) + off);
    if constexpr (NT) __builtin_nontemporal_store(__builtin_bit_cast(u32x4, t), d);
    else *d = __builtin_bit_cast(u32x4, t);
  } else {
    _Float16 t[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = static_cast<_Float16>(v[e]);
    u32x4* d = reinterpret_cast<u32x4*>(reinterpret_cast<_Float16*>(y) + off);
    if constexpr (NT) __builtin_nontemporal_store(__builtin_bit_cast(u32x4, t), d);
    else *d = __builtin_bit_cast(u32x4, t);
  }
}

__device__ __forceinline__ bf16x8 as_b8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// LDS byte offset of 16-byte column c16 (0..7) of staged row r (0..31).
__device__ __forceinline__ int xs_off(int r, int c16) { return r * kVgRowB + ((c16 ^ ((r >> 1) & 7)) << 4); }

// A product of many rows (k_wgemm): for group z < batch, rows j < n_z,
//   acc[j, n] = sum_k X_z[j, k] * W_z[n, k], X_z[j] = x + z*sxb + row(j)*ldx,
// row(j) = rows[z*M + j] (rows NULL: j), n_z = counts[z] (counts NULL: M);
// output row j of group z at y + z*syb + j*ldy.  epi 0: the sums, 1: SwiGLU
// (32-row blocks of 16 gate + 16 up rows) times comb[row(j)*ldc + z] (comb
// NULL: 1), 3: y fp32 += the sums.
struct WgParams {
  const uint16_t* x;
  const uint16_t* w;       // vnx_pack_bf16 order, group z at w + z*swb
  void* y;
  const float* comb;
  const int32_t* rows;
  const int32_t* counts;
  int64_t ldx, sxb, swb, ldy, syb, ldc;
  int M, N, K, batch;
  int64_t total_rows;      // with counts: their expected sum (0: batch * M), for the choice of a tile shape
  int nt, ng;              // 32-column tiles, N groups of a workgroup's (set by wg_run)
  int vec_out;
};

int wg_run(WgParams p, int epi, int y_dtype, hipStream_t s);

// Where vnx_gemm_bf16 / _residual leave the verify-size kernel (32 x 32
// outputs per wave, K split over the waves, every operand re-read per 32 rows)
// for k_wgemm: from 2,048 output tiles of 32 x 32.  Measured (us, k_vgemm /
// k_wgemm): 448 rows x 2,048 x 1,024 6.8 / 7.6, x 1,024 x 2,752 11.0 / 15.8
// (448 tiles); 1,016 rows x 1,024 x 1,024 8.2 / 9.4 (1,024 tiles); 1,016 rows
// x 2,048 x 1,024 10.0 / 8.3 (2,048 tiles); 448 rows x 5,504 x 1,024 13.8 /
// 12.3 (2,408 tiles); 2,048 rows x 5,504 x 1,024 51 / 29.
constexpr int64_t kWgMinTiles = 2048;

}  // namespace vnx
