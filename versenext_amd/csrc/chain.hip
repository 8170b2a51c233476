// Chain attention of long forwards on gfx950 (vnx_chain_attn): the N new rows
// of every sequence (a prompt, or any chain too long for one tree mask word)
// over its cached rows, all TriSparse paths in one launch
// (packages/verse_nex/verse_nex/tri_sparse_attn.py:258-378 window, :469-495
// global rows, :489-530 ALiBi, mixed as :585-608).  The new rows are already
// in the cache, so row j of the cache is the key at position j and node i of
// batch row b sits at tp_b + i and sees j <= tp_b + i.
//
// Work split: a workgroup (4 waves) owns 32 * CW query columns of one (b, kv
// head); column c is node c / n_rep of query head kvh * n_rep + c % n_rep, so
// the heads that share K and V share every staged row and a workgroup's
// columns are consecutive positions (a narrow causal range).  Its waves are
// CW (32 columns each) x KW = 4 / CW (key splits): a step stages KW * 64 keys
// in LDS, wave (cw, kw) takes keys 64 kw .. +64 of it.
//   S^T[key][q] = K Q^T   v_mfma_f32_32x32x16_bf16; K's LDS row order is the
//                         permutation that makes a lane's 16 results the 16
//                         keys it must hold as the next product's B operand
//                         (key = 16 (i / 8) + 8 h + i % 8 of its block), so P
//                         never leaves its registers;
//   online softmax        lane-local but for one exchange with lane ^ 32;
//   O^T[dim][q] += V^T P^T with P as bf16 hi + lo parts (two MFMAs), the
//                         relative accuracy ~2^-17 of vnx_tree_attn.
// V is transposed on its way into LDS (pairs of keys packed to 32 bits).
// Both tiles are XOR-swizzled by 16-byte unit: conflict-free 16-byte reads.
// The next step's rows are loaded to registers under this step's math.
//
// What bounds it: at 4 x 512 rows x 16 heads of 64 the products take ~2 us of
// the matrix cores and the softmax ~4 us of VALU; the rest is the serial walk
// of a late tile's key steps.  One launch replaces eight of vnx_tree_attn
// (64-row chunks, each with its own lens + c kernel and sometimes a merge).
#include <climits>

#include "vnx_internal.h"

namespace vnx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct ChainParams {
  const uint16_t* q;
  const uint16_t* kc;
  const uint16_t* vc;
  void* out;
  int64_t q_sb, q_sh, q_sr;
  int64_t c_sb, c_sh, c_sr;
  int64_t o_sb, o_sh, o_sr;
  const int32_t* tp_batch;
  const uint16_t* k2;
  const uint16_t* v2;
  int64_t s2_sb, s2_sh, s2_sr;
  const float* gates;
  const float* slopes;
  int B, H, Hkv, n_rep, Tp, N, T2;
  int tiles;       // query tiles per (b, kv head)
  int window, alibi_max;
  float c;         // scale * log2(e)
};

__device__ __forceinline__ bf16x8 ca_b8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ u32x4 ca_ldg16(const uint16_t* p) {
  typedef const __attribute__((address_space(1))) u32x4* gptr;
  return *(gptr)(p);
}

__device__ __forceinline__ float ca_ex2(float x) { return __builtin_amdgcn_exp2f(x); }

template <int OT>
__device__ __forceinline__ void ca_store4(void* out, int64_t off, float a, float b, float c, float d) {
  if constexpr (OT == 0) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + off) = f32x4{a, b, c, d};
  } else if constexpr (OT == 1) {
    const __bf16 t[4] = {static_cast<__bf16>(a), static_cast<__bf16>(b), static_cast<__bf16>(c),
                         static_cast<__bf16>(d)};
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + off) = __builtin_bit_cast(uint2, t);
  } else {
    const _Float16 t[4] = {static_cast<_Float16>(a), static_cast<_Float16>(b), static_cast<_Float16>(c),
                           static_cast<_Float16>(d)};
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + off) = __builtin_bit_cast(uint2, t);
  }
}

template <int D, int OT, int CW>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void k_chain_attn(ChainParams p) {
  constexpr int KW = 4 / CW;
  constexpr int KB = KW * 64;          // keys staged per step
  constexpr int UD = D / 8;            // 16-byte units of a K row
  constexpr int UK = KB / 8;           // 16-byte units of a V^T row
  constexpr int DT = D / 32;           // 32-dim tiles of O
  constexpr int KLD = KB * UD / 256;   // K loads per thread and step
  constexpr int VLD = KB / 2 * UD / 256;  // V key-pair loads (two rows each)
  constexpr int TILE_B = KB * D * 2;
  // partial (O, m, l) of the key splits, over the dead tiles
  constexpr int MERGE_B = (KW - 1) * CW * 64 * (DT * 16 + 2) * 4;
  static_assert(MERGE_B <= 2 * TILE_B, "the merge fits the tiles");
  __shared__ __attribute__((aligned(16))) char smem[2 * TILE_B];
  char* s_k = smem;
  char* s_v = smem + TILE_B;

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = w % CW, kw = w / CW;
  const int r = lane & 31, h = lane >> 5;
  // Late tiles see the most keys and start first; a (b, kv head)'s tiles run
  // on one XCD (workgroup t on XCD t % 8) whenever the heads divide by 8.
  const int BH = p.B * p.Hkv;
  int head, tile;
  if (BH % 8 == 0) {
    const int slot = blockIdx.x >> 3;
    head = (blockIdx.x & 7) + 8 * (slot % (BH / 8));
    tile = p.tiles - 1 - slot / (BH / 8);
  } else {
    head = blockIdx.x % BH;
    tile = p.tiles - 1 - blockIdx.x / BH;
  }
  const int kvh = head % p.Hkv, b = head / p.Hkv;
  int tp = p.Tp;
  if (p.tp_batch) tp = min(max(p.tp_batch[b], 0), p.Tp);
  tp = __builtin_amdgcn_readfirstlane(tp);

  const int NQ = p.n_rep * p.N;
  const int c0 = tile * 32 * CW;
  const int cl = min(c0 + 32 * cw + r, NQ - 1);  // this lane's column (clamped past the end: not stored)
  const bool live = c0 + 32 * cw + r < NQ;
  const int node = cl / p.n_rep, qh = kvh * p.n_rep + cl % p.n_rep;
  const int qpos = tp + node;
  // positions of this wave's first and last columns, and of the workgroup's
  const int wlo = tp + min(c0 + 32 * cw, NQ - 1) / p.n_rep;
  const int whi = tp + min(c0 + 32 * cw + 31, NQ - 1) / p.n_rep;
  const int glo = tp + c0 / p.n_rep;
  const int ghi = tp + min(c0 + 32 * CW - 1, NQ - 1) / p.n_rep;

  bf16x8 qf[D / 16];
  {
    const uint16_t* qr = p.q + b * p.q_sb + qh * p.q_sh + (int64_t)node * p.q_sr;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = ca_b8(ca_ldg16(qr + (2 * s + h) * 8));
  }
  const bool alibi = p.slopes && tp + p.N <= p.alibi_max;
  const float slope = alibi ? p.slopes[qh] * 1.4426950408889634f : 0.0f;

  // staging: K row key goes to LDS row lr(key); V pair rows (2 kp, 2 kp + 1)
  const int su = tid % UD;             // 16-byte unit of the row
  const int sr = tid / UD;             // first row (K) / key pair (V)
  constexpr int SR = 256 / UD;         // rows per pass
  u32x4 kreg[KLD], vreg[VLD][2];
  const uint16_t* kbase = nullptr;
  const uint16_t* vbase = nullptr;
  int64_t rs = 0;
  int kend = 0;                        // rows of the segment
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < KLD; ++i)
      kreg[i] = ca_ldg16(kbase + (int64_t)min(k0 + sr + i * SR, kend - 1) * rs + su * 8);
#pragma unroll
    for (int i = 0; i < VLD; ++i) {
      const int kp = 2 * (sr + i * SR);
      vreg[i][0] = ca_ldg16(vbase + (int64_t)min(k0 + kp, kend - 1) * rs + su * 8);
      vreg[i][1] = ca_ldg16(vbase + (int64_t)min(k0 + kp + 1, kend - 1) * rs + su * 8);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < KLD; ++i) {
      const int key = sr + i * SR, k32 = key & 31;
      const int j = k32 & 7;
      const int lr = (key & ~31) + 8 * (2 * (k32 >> 4) + (j >> 2)) + 4 * ((k32 >> 3) & 1) + (j & 3);
      *reinterpret_cast<u32x4*>(s_k + lr * (D * 2) + ((su ^ (lr & 7)) << 4)) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < VLD; ++i) {
      const int kp = sr + i * SR;      // keys 2 kp, 2 kp + 1: unit kp / 4, dword kp % 4
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t a = vreg[i][0][e >> 1], z = vreg[i][1][e >> 1];
        const uint32_t v = (e & 1) ? (a >> 16) | (z & 0xFFFF0000u) : (a & 0xFFFFu) | (z << 16);
        const int dim = su * 8 + e;
        const int u = (kp >> 2) ^ ((dim ^ (dim >> 3)) & 7);
        *reinterpret_cast<uint32_t*>(s_v + dim * (KB * 2) + (u << 4) + ((kp & 3) << 2)) = v;
      }
    }
  };

  float fin[DT][16];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) fin[t][i] = 0.0f;

  const bool has2 = p.T2 > 0;
  // seg 0: window path; 1: global rows; 2: ALiBi
  for (int seg = 0; seg < 3; ++seg) {
    if ((seg == 1 && !has2) || (seg == 2 && !alibi)) continue;  // uniform over the workgroup
    int klo = 0;
    if (seg == 1) {
      const int64_t base = b * p.s2_sb + kvh * p.s2_sh;
      kbase = p.k2 + base;
      vbase = p.v2 + base;
      rs = p.s2_sr;
      kend = p.T2;
    } else {
      const int64_t base = b * p.c_sb + kvh * p.c_sh;
      kbase = p.kc + base;
      vbase = p.vc + base;
      rs = p.c_sr;
      kend = ghi + 1;
      if (seg == 0 && p.window > 0) klo = max(0, glo - p.window + 1);
    }
    const int win = seg == 0 && p.window > 0 ? p.window : INT_MAX;  // qpos - key < win
    float m = kNegInf, l = 0.0f;
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;

    load(klo);
    for (int kb = klo; kb < kend; kb += KB) {
      stage();
      __syncthreads();
      if (kb + KB < kend) load(kb + KB);
      const int k0 = kb + 64 * kw;     // this wave's first key of the step
      const bool any = seg == 1 ? k0 < kend : (k0 <= whi && (win == INT_MAX || k0 + 63 > wlo - win));
      if (any) {                       // uniform per wave
        f32x16 s[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[t][i] = 0.0f;
          const int lr = 64 * kw + 32 * t + r;
#pragma unroll
          for (int ks = 0; ks < D / 16; ++ks) {
            const u32x4 a = *reinterpret_cast<const u32x4*>(s_k + lr * (D * 2) + (((2 * ks + h) ^ (lr & 7)) << 4));
            s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca_b8(a), qf[ks], s[t], 0, 0, 0);
          }
        }
        // scores in the exp2 domain; keys outside the column's range to -inf
        const bool full = seg == 1 ? k0 + 64 <= kend : (k0 + 63 <= wlo && (win == INT_MAX || k0 > whi - win));
        float mx = kNegInf;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * t + 16 * (i >> 3) + 8 * h + (i & 7);
            float x = s[t][i] * p.c;
            if (seg == 2) x = __builtin_fmaf(slope, (float)(key - qpos), x);
            if (!full) {
              const bool vis = seg == 1 ? key < kend : (key <= qpos && (win == INT_MAX || qpos - key < win));
              x = vis ? x : kNegInf;
            }
            s[t][i] = x;
            mx = fmaxf(mx, x);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float mr = mn == kNegInf ? 0.0f : mn;   // no key yet: every term is 0
        const float al = ca_ex2(m - mr);
        m = mn;
        float ls = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            s[t][i] = ca_ex2(s[t][i] - mr);
            ls += s[t][i];
          }
        l = l * al + ls;
        if (__any(al != 1.0f)) {
#pragma unroll
          for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[t][i] *= al;
        }
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {               // 16-key chunks
          bf16x8 hi, lo;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float x = s[cc >> 1][8 * (cc & 1) + j];
            hi[j] = static_cast<__bf16>(x);
            lo[j] = static_cast<__bf16>(x - static_cast<float>(hi[j]));
          }
#pragma unroll
          for (int t = 0; t < DT; ++t) {
            const int dim = 32 * t + r;
            const int u = (8 * kw + 2 * cc + h) ^ ((dim ^ (dim >> 3)) & 7);
            const u32x4 a = *reinterpret_cast<const u32x4*>(s_v + dim * (KB * 2) + (u << 4));
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca_b8(a), hi, o[t], 0, 0, 0);
            o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca_b8(a), lo, o[t], 0, 0, 0);
          }
        }
      }
      __syncthreads();                 // the tiles are read before the next step stages
    }
    l += __shfl_xor(l, 32);
    if constexpr (KW > 1) {
      // key splits 1 .. of a column group -> LDS, merged in split order by split 0
      float* red = reinterpret_cast<float*>(smem);
      constexpr int RW = DT * 16 + 2;
      if (kw > 0) {
        float* d = red + ((kw - 1) * CW + cw) * RW * 64 + lane;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) d[(t * 16 + i) * 64] = o[t][i];
        d[(DT * 16) * 64] = m;
        d[(DT * 16 + 1) * 64] = l;
      }
      __syncthreads();
      if (kw == 0) {
#pragma unroll
        for (int k = 1; k < KW; ++k) {
          const float* d = red + ((k - 1) * CW + cw) * RW * 64 + lane;
          const float m2 = d[(DT * 16) * 64], l2 = d[(DT * 16 + 1) * 64];
          const float mn = fmaxf(m, m2), mr = mn == kNegInf ? 0.0f : mn;
          const float a1 = ca_ex2(m - mr), a2 = ca_ex2(m2 - mr);
          m = mn;
          l = l * a1 + l2 * a2;
#pragma unroll
          for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[t][i] = o[t][i] * a1 + d[(t * 16 + i) * 64] * a2;
        }
      }
      __syncthreads();                 // read before the next segment stages
    }
    const float gate = (has2 || p.slopes) ? p.gates[seg] : 1.0f;
    const float inv = l > 0.0f ? gate / l : 0.0f;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) fin[t][i] = __builtin_fmaf(o[t][i], inv, fin[t][i]);
  }
  if (kw != 0 || !live) return;
  const int64_t ob = b * p.o_sb + qh * p.o_sh + (int64_t)node * p.o_sr;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ca_store4<OT>(p.out, ob + 32 * t + 8 * i + 4 * h, fin[t][4 * i], fin[t][4 * i + 1], fin[t][4 * i + 2],
                    fin[t][4 * i + 3]);
}

bool ca_strides_ok(const int64_t (&s)[3], int unit) {
  return s[0] >= 0 && s[1] >= 0 && s[2] >= 0 && s[0] % unit == 0 && s[1] % unit == 0 && s[2] % unit == 0;
}

// Column waves per workgroup: wide tiles re-stage a key for the fewest
// columns, narrow ones leave more workgroups and split the walk of the keys
// over the waves; the widest that still gives every CU `per` workgroups.
int ca_column_waves(int64_t heads, int64_t columns) {
  const int64_t cus = device_cus();
  if (heads * ((columns + 127) / 128) >= 2 * cus) return 4;
  if (heads * ((columns + 63) / 64) >= cus) return 2;
  return 1;
}

template <int D, int OT>
void ca_launch(const ChainParams& p0, hipStream_t st) {
  ChainParams p = p0;
  const int64_t heads = (int64_t)p.B * p.Hkv, cols = (int64_t)p.n_rep * p.N;
  const int cw = ca_column_waves(heads, cols);
  p.tiles = (int)((cols + 32 * cw - 1) / (32 * cw));
  const dim3 grid((unsigned)(heads * p.tiles));
  if (cw == 4) hipLaunchKernelGGL((k_chain_attn<D, OT, 4>), grid, dim3(256), 0, st, p);
  else if (cw == 2) hipLaunchKernelGGL((k_chain_attn<D, OT, 2>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((k_chain_attn<D, OT, 1>), grid, dim3(256), 0, st, p);
}

}  // namespace
}  // namespace vnx

using namespace vnx;

extern "C" {

int vnx_chain_attn(const vnx_tree_attn_args* a, void* stream) {
  if (!a) return VNX_ERR_INVALID_ARG;
  const int B = a->B, H = a->H, Hkv = a->Hkv, N = a->N, Tp = a->Tp, d = a->d;
  if (B < 0 || H <= 0 || Hkv <= 0 || H % Hkv || N < 1 || Tp < 0 || a->T2 < 0) return VNX_ERR_INVALID_ARG;
  if (a->out_dtype != VNX_F32 && a->out_dtype != VNX_BF16 && a->out_dtype != VNX_F16) return VNX_ERR_UNSUPPORTED;
  if (d != 64 && d != 128) return VNX_ERR_UNSUPPORTED;
  if (a->f32_rows || a->qkv || a->anc || a->k_tree || a->v_tree) return VNX_ERR_UNSUPPORTED;
  if (a->window < 0 || a->alibi_max_keys < 0) return VNX_ERR_INVALID_ARG;
  if (!(a->scale > 0.0f) || !__builtin_isfinite(a->scale)) return VNX_ERR_INVALID_ARG;
  if (B == 0) return VNX_OK;
  if (!a->q || !a->k_cache || !a->v_cache || !a->out) return VNX_ERR_INVALID_ARG;
  const auto mis4 = [](const void* x) { return (reinterpret_cast<uintptr_t>(x) & 3u) != 0; };
  if ((a->T2 > 0 || a->alibi_slopes) && (!a->gates || mis4(a->gates))) return VNX_ERR_INVALID_ARG;
  if (mis4(a->alibi_slopes) || mis4(a->tp_batch)) return VNX_ERR_INVALID_ARG;
  if (a->T2 > 0 && (!a->k_seg2 || !a->v_seg2)) return VNX_ERR_INVALID_ARG;
  // 16-byte loads of bf16 rows; 16-byte (fp32) / 8-byte (16-bit) output stores
  if (!ca_strides_ok(a->q_strides, 8) || !ca_strides_ok(a->cache_strides, 8) || !ca_strides_ok(a->out_strides, 4) ||
      (a->T2 > 0 && !ca_strides_ok(a->seg2_strides, 8)))
    return VNX_ERR_UNSUPPORTED;
  if (!aligned16(a->q) || !aligned16(a->k_cache) || !aligned16(a->v_cache) || !aligned16(a->out) ||
      (a->T2 > 0 && (!aligned16(a->k_seg2) || !aligned16(a->v_seg2))))
    return VNX_ERR_UNSUPPORTED;
  // 32-bit positions, columns and workgroup ids
  if ((int64_t)Tp + N >= INT_MAX || (int64_t)(H / Hkv) * N >= INT_MAX ||
      (int64_t)B * Hkv * (((int64_t)(H / Hkv) * N + 31) / 32) >= INT_MAX)
    return VNX_ERR_UNSUPPORTED;
  ChainParams p{};
  p.q = static_cast<const uint16_t*>(a->q);
  p.kc = static_cast<const uint16_t*>(a->k_cache);
  p.vc = static_cast<const uint16_t*>(a->v_cache);
  p.out = a->out;
  p.q_sb = a->q_strides[0]; p.q_sh = a->q_strides[1]; p.q_sr = a->q_strides[2];
  p.c_sb = a->cache_strides[0]; p.c_sh = a->cache_strides[1]; p.c_sr = a->cache_strides[2];
  p.o_sb = a->out_strides[0]; p.o_sh = a->out_strides[1]; p.o_sr = a->out_strides[2];
  p.tp_batch = a->tp_batch;
  if (a->T2 > 0) {
    p.k2 = static_cast<const uint16_t*>(a->k_seg2);
    p.v2 = static_cast<const uint16_t*>(a->v_seg2);
    p.s2_sb = a->seg2_strides[0]; p.s2_sh = a->seg2_strides[1]; p.s2_sr = a->seg2_strides[2];
    p.T2 = a->T2;
  }
  p.gates = a->gates;
  p.slopes = a->alibi_slopes;
  p.B = B; p.H = H; p.Hkv = Hkv; p.n_rep = H / Hkv; p.Tp = Tp; p.N = N;
  p.window = a->window;
  p.alibi_max = a->alibi_max_keys;
  p.c = (float)((double)a->scale * 1.4426950408889634);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int ot = a->out_dtype == VNX_F32 ? 0 : a->out_dtype == VNX_BF16 ? 1 : 2;
  if (d == 64) {
    if (ot == 0) ca_launch<64, 0>(p, st);
    else if (ot == 1) ca_launch<64, 1>(p, st);
    else ca_launch<64, 2>(p, st);
  } else {
    if (ot == 0) ca_launch<128, 0>(p, st);
    else if (ot == 1) ca_launch<128, 1>(p, st);
    else ca_launch<128, 2>(p, st);
  }
  VNX_LAUNCH_CHECK();
  return VNX_OK;
}

}  // extern "C"
